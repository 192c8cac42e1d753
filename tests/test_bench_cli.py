"""bench.py's command line on the CPU: more than one GPU is refused before anything touches
a device, with a message that says so."""

import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_more_than_one_gpu_is_refused():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 2
    assert "measures one GPU" in r.stderr and "--gpus 2" in r.stderr
    assert r.stdout == ""  # no JSON line


def test_every_expert_product_is_counted():
    """The FLOP table and the MoE layer's share know every expert entry point of the library."""
    sys.path.insert(0, ROOT)
    import bench
    from abacus_amd import _lib

    experts = [n for n in _lib.SIGNATURES if "_experts_" in n and not n.endswith("_bytes")]
    assert len(experts) >= 5 and all(bench.is_moe(n) for n in experts)
    bench.check_known(n for n in _lib.SIGNATURES if not n.endswith("_bytes"))


def test_settle_takes_the_set_up_out_of_the_collector():
    import gc

    import bench

    try:
        bench.settle()
        assert gc.get_freeze_count() > 0 and gc.isenabled()
    finally:
        gc.unfreeze()

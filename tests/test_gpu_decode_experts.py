"""abacus_experts_decode_fwd (small forward batches) against fp64: hidden sizes of any alignment, reductions off
the 32-row step, column tiles that overlap, row groups that are part full, one and several down slices."""

import itertools

import pytest
import torch

from abacus_amd import _lib
from abacus_amd.moe import MoE
from oracle import moe_oracle as oracle

pytestmark = pytest.mark.gpu

call, ptr = _lib.call, _lib.ptr


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("counts,D,M", [
    ([1, 0, 1], 1024, 4096),                   # one row each: sliced down projection
    ([0, 3, 16, 17, 32, 33, 70, 0, 0, 0, 0], 136, 136),  # every row-group remainder, one tile and an overlapping one
    ([58, 1, 0, 5], 264, 263),                 # odd hidden size; an expert of two row tiles
    ([1, 0, 2] * 60, 384, 384),                # enough tiles for blocks of 4 waves
    ([150] + [0] * 127 + [3] * 40, 1032, 520),  # ... and numbered row tiles past the first
    ([6, 9], 128, 2731),                       # odd, several slices with a tail block
    ([2, 1, 0, 4], 320, 130),
], ids=["single_rows", "row_groups", "odd", "four_waves", "one_heavy", "odd_sliced", "two_mod_vector"])
def test_decode_experts_match_fp64(dtype, counts, D, M):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(41)
    E, R = len(counts), sum(counts)
    offs = [0] + list(itertools.accumulate(counts))
    offsets = torch.tensor(offs, dtype=torch.int32, device=dev)
    dt, s = _lib.dtype_code(dtype), _lib.stream_of(dev)
    vec = 16 // torch.empty(0, dtype=dtype).element_size()
    ld_h = -(-M // vec) * vec

    def rn(*shape, scale=1.0):
        return (torch.randn(*shape, device=dev, generator=gen) * scale).to(dtype)

    xp, wg, wu, wd = rn(R, D), rn(E, D, M, scale=0.05), rn(E, D, M, scale=0.05), rn(E, M, D, scale=0.05)
    nbytes = _lib.query("abacus_experts_decode_ws_bytes", R, D, M, E, dt)
    assert nbytes >= 0
    ws = torch.full((nbytes // 4 + 1,), float("nan"), dtype=torch.float32, device=dev)
    h = torch.full((R, ld_h), float("nan"), dtype=dtype, device=dev)
    y = torch.full((R, D), float("nan"), dtype=dtype, device=dev)
    call("abacus_experts_decode_fwd", ptr(xp), ptr(wg), ptr(wu), ptr(wd), ptr(offsets), R, D, M, E, dt, ld_h, ptr(h),
         ptr(y), ptr(ws), nbytes, s)
    torch.cuda.synchronize()
    assert not torch.isnan(h).any() and not torch.isnan(y).any()
    assert torch.count_nonzero(h[:, M:]) == 0
    # at most four bf16 roundings (2^-9 each) meet in a value of h, one in y; fp32 sums of up to 2731 terms
    tol = 1e-2 if dtype == torch.bfloat16 else 1e-5
    for e in range(E):
        a, b = offs[e], offs[e + 1]
        if a == b:
            continue
        x64 = xp[a:b].double()
        g = x64 @ wg[e].double()
        for name, got, want in (("h", h[a:b, :M], g * torch.sigmoid(g) * (x64 @ wu[e].double())),
                                ("y", y[a:b], h[a:b, :M].double() @ wd[e].double())):
            err = float((got.double() - want).norm() / want.norm())
            assert err < tol, f"{name} expert {e}: relative error {err:.3g}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("counts,D,M", [
    ([0, 300, 1, 0] + [0] * 66 + [700, 33, 32] + [0] * 55, 264, 263),  # row tiles past the first of four experts
    ([0] * 127 + [2048], 128, 136),            # all rows on the last expert
    ([1] * 70, 384, 1025),                     # odd hidden size, blocks of 4 waves
    ([2] * 24, 1024, 1031),                    # ... weights past the caches (read nontemporal), 8 waves
    ([2] * 60 + [40, 0, 0, 33], 512, 1031),    # ... 4 waves, and rows past the first tile
], ids=["later_tiles", "one_expert", "odd_four_waves", "odd_streamed", "odd_streamed_four_waves"])
def test_decode_experts_variants(dtype, counts, D, M):
    """The forms of the kernels that a size or the routing selects, as test_decode_experts_match_fp64."""
    test_decode_experts_match_fp64(dtype, counts, D, M)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("T,D,M,E,K", [(1, 256, 301, 8, 2), (37, 132, 160, 16, 4)])
def test_small_forward_matches_oracle(dtype, T, D, M, E, K):
    """The eval layer (decode kernels; D off the vector width pads first) against the oracle in fp64."""
    torch.manual_seed(7)
    moe = MoE(D, E, K, hidden_dim=M).to("cuda", dtype).eval()
    x = torch.randn(1, T, D, device="cuda").to(dtype)
    with torch.no_grad():
        got = moe(x)
    idx = moe.router.last_routing.indices_TK
    p = {n: t.detach().double().cpu() for n, t in moe.named_parameters()}
    want, _ = oracle.moe_forward(x.reshape(T, D).double().cpu(), p["router.w_DE"], torch.zeros(E, dtype=torch.float64),
                                 p["w_gate_EDM"], p["w_up_EDM"], p["w_down_EMD"], K, indices_TK=idx.cpu())
    err = float((got.reshape(T, D).double().cpu() - want).norm() / want.norm())
    assert err < (2e-2 if dtype == torch.bfloat16 else 1e-5), err


@pytest.mark.parametrize("args,msg", [((17, 256, 256, 1, 1, 256), "not taken"), ((8, 256, 257, 4, 1, 257), "ld_h")])
def test_rejected_shapes(args, msg):
    R, D, M, E, dt, ld = args
    with pytest.raises(RuntimeError, match=msg):
        call("abacus_experts_decode_fwd", None, None, None, None, None, R, D, M, E, dt, ld, None, None, None, 0, None)

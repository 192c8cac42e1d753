"""abacus_experts_decode_fwd with 16 to 128 rows per expert (bf16 hidden sizes off the 16-byte vector) against fp64:
remainders of the 16-row groups and 64-row blocks, more experts than lanes, overlapping and single column tiles,
reductions off the 32-row step, one and several down slices; and which shapes it takes."""

import itertools

import pytest
import torch

from abacus_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,D,M", [
    ([0, 1, 16, 32, 33, 63, 64, 65, 0, 129, 200], 136, 263),
    ([40, 30], 128, 2731),                  # a few tiles: sliced down projection with a tail block
    ([33] * 70 + [0] * 59 + [90], 264, 130),  # three lane blocks of experts, the last with one row block
    ([0] * 3 + [500], 520, 1001),           # all rows on one expert
], ids=["row_groups", "sliced", "many_experts", "one_expert"])
def test_unaligned_rows_match_fp64(counts, D, M):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(43)
    E, R, ld_h = len(counts), sum(counts), -(-M // 8) * 8
    offs = [0] + list(itertools.accumulate(counts))
    assert 16 * E < R <= 128 * E

    def rn(*shape, scale=1.0):
        return (torch.randn(*shape, device=dev, generator=gen) * scale).to(torch.bfloat16)

    xp, wg, wu, wd = rn(R, D), rn(E, D, M, scale=0.05), rn(E, D, M, scale=0.05), rn(E, M, D, scale=0.05)
    nbytes = _lib.query("abacus_experts_decode_ws_bytes", R, D, M, E, _lib.BF16)
    assert nbytes >= 0
    ws = torch.full((nbytes // 4 + 1,), float("nan"), dtype=torch.float32, device=dev)
    h, y = (torch.full((R, n), float("nan"), dtype=torch.bfloat16, device=dev) for n in (ld_h, D))
    ptr = _lib.ptr
    _lib.call("abacus_experts_decode_fwd", ptr(xp), ptr(wg), ptr(wu), ptr(wd),
              ptr(torch.tensor(offs, dtype=torch.int32, device=dev)), R, D, M, E, _lib.BF16, ld_h, ptr(h), ptr(y), ptr(ws),
              nbytes, _lib.stream_of(dev))
    torch.cuda.synchronize()
    assert not torch.isnan(h).any() and not torch.isnan(y).any()
    assert torch.count_nonzero(h[:, M:]) == 0
    for e in range(E):
        a, b = offs[e], offs[e + 1]
        if a == b:
            continue
        x64 = xp[a:b].double()
        g = x64 @ wg[e].double()
        for name, got, want in (("h", h[a:b, :M], g * torch.sigmoid(g) * (x64 @ wu[e].double())),
                                ("y", y[a:b], h[a:b, :M].double() @ wd[e].double())):
            err = float((got.double() - want).norm() / want.norm())
            assert err < 1e-2, f"{name} expert {e}: {err:.3g}"  # at most four bf16 roundings (2^-9 each) meet in a value


def test_taken_up_to_128_rows_per_expert():
    taken = lambda R, M, dt: _lib.query("abacus_experts_decode_ws_bytes", R, 256, M, 4, dt) >= 0
    assert taken(512, 257, _lib.BF16) and not taken(513, 257, _lib.BF16)
    assert taken(64, 256, _lib.BF16) and not taken(65, 256, _lib.BF16)
    assert taken(256, 257, _lib.F32) and not taken(257, 257, _lib.F32)

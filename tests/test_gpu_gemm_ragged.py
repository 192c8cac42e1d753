"""Expert products whose fixed reduction is not a whole number of k-tiles (64 bf16, 32 fp32): the last k-tile
reads zeros past the end of each operand row, in full, thin and split tiles, against fp64."""

import itertools

import pytest
import torch

from abacus_amd import _lib

pytestmark = pytest.mark.gpu

call, ptr = _lib.call, _lib.ptr


def _rel(got, want):
    return float((got.double() - want).norm() / want.norm().clamp(min=1e-30))


@pytest.mark.parametrize("dtype,counts,D,M", [
    (torch.bfloat16, [300, 0, 129, 70], 200, 264),     # full and thin tiles, remainders 8
    (torch.bfloat16, [5, 0, 33, 90], 72, 1000),        # a small batch: thin tiles only, remainders 8 and 40
    (torch.bfloat16, [1, 256], 8, 56),                 # shorter than one k-tile
    (torch.bfloat16, [1500, 600, 700], 2056, 2568),    # the down projection's split tail, remainders 8
    (torch.float32, [2000, 2096], 4100, 1028),         # fp32 on the pipelined kernel (a round of tiles), remainders 4
    (torch.float32, [30, 0, 70], 68, 100),             # fp32 on the generic kernel
], ids=["full_thin", "small", "short", "split", "fp32_pipe", "fp32_generic"])
def test_reductions_off_the_k_tile(dtype, counts, D, M):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(31)
    E, R = len(counts), sum(counts)
    offs = [0] + list(itertools.accumulate(counts))
    offsets = torch.tensor(offs, dtype=torch.int32, device=dev)
    dt, s = _lib.dtype_code(dtype), _lib.stream_of(dev)

    def rn(*shape, scale=1.0):
        return (torch.randn(*shape, device=dev, generator=gen) * scale).to(dtype)

    def nan(*shape):
        return torch.full(shape, float("nan"), dtype=dtype, device=dev)

    xp, dy, h, gate, up, dg, du = rn(R, D), rn(R, D), rn(R, M), rn(R, M), rn(R, M), rn(R, M), rn(R, M)
    wg, wu, wd = rn(E, D, M, scale=0.05), rn(E, D, M, scale=0.05), rn(E, M, D, scale=0.05)
    G, U, H, Y, dG, dU, dX = nan(R, M), nan(R, M), nan(R, M), nan(R, D), nan(R, M), nan(R, M), nan(R, D)
    dWd, dWg, dWu = nan(E, M, D), nan(E, D, M), nan(E, D, M)
    call("abacus_moe_gateup_fwd", ptr(xp), ptr(wg), ptr(wu), ptr(offsets), R, D, M, E, dt, ptr(G), ptr(U), ptr(H), s)
    nbytes = _lib.query("abacus_moe_down_fwd_ws_bytes", R, M, D, E, dt)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev) if nbytes else None
    call("abacus_moe_down_fwd", ptr(h), ptr(wd), ptr(offsets), R, M, D, E, dt, ptr(Y), ptr(ws), nbytes, s)
    call("abacus_moe_down_bwd", ptr(dy), ptr(wd), ptr(gate), ptr(up), ptr(h), ptr(offsets), R, M, D, E, dt, ptr(dG),
         ptr(dU), ptr(dWd), ptr(_lib.tile_ctr(dev)), s)
    call("abacus_moe_gateup_bwd", ptr(dg), ptr(du), ptr(wg), ptr(wu), ptr(xp), ptr(offsets), R, D, M, E, dt, ptr(dX),
         ptr(dWg), ptr(dWu), ptr(_lib.tile_ctr(dev)), s)
    torch.cuda.synchronize()
    # one bf16 rounding is 2^-9 of a value at most (0.2%), and at most four meet in dG; an fp32 sum of n <= 4100
    # products is off by at most sqrt(n) 2^-24 of its norm (4e-6) for random terms
    tol = 1e-2 if dtype == torch.bfloat16 else 1e-5
    for e in range(E):
        a, b = offs[e], offs[e + 1]
        if a == b:
            for t in (dWd, dWg, dWu):
                assert torch.count_nonzero(t[e]) == 0
            continue
        d = lambda t: t[a:b].double()
        g64, u64 = d(gate), d(up)
        sg = torch.sigmoid(g64)
        dh = d(dy) @ wd[e].double().t()
        Gd, Ud = d(G), d(U)
        for name, got, want in (
            ("G", G[a:b], d(xp) @ wg[e].double()),
            ("U", U[a:b], d(xp) @ wu[e].double()),
            ("H", H[a:b], Gd * torch.sigmoid(Gd) * Ud),
            ("Y", Y[a:b], d(h) @ wd[e].double()),
            ("dG", dG[a:b], dh * u64 * sg * (1 + g64 * (1 - sg))),
            ("dU", dU[a:b], dh * g64 * sg),
            ("dX", dX[a:b], d(dg) @ wg[e].double().t() + d(du) @ wu[e].double().t()),
            ("dWd", dWd[e], d(h).t() @ d(dy)),
            ("dWg", dWg[e], d(xp).t() @ d(dg)),
            ("dWu", dWu[e], d(xp).t() @ d(du)),
        ):
            assert not torch.isnan(got).any(), f"{name} expert {e}: unwritten elements"
            assert _rel(got, want) < tol, f"{name} expert {e}: {_rel(got, want):.3g}"

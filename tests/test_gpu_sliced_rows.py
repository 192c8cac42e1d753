"""Launches whose tiles are too few for the GPU run as slices of the reduction (down forward, gate/up data gradient):
the same products against fp64, repeatable bit for bit, with the weight gradients beside them unchanged."""

import itertools

import pytest
import torch

from abacus_amd import _lib

pytestmark = pytest.mark.gpu

call, ptr = _lib.call, _lib.ptr


@pytest.mark.parametrize("dtype,counts,D,M", [
    (torch.bfloat16, [300, 0, 129, 70, 1], 200, 6008),   # full and thin tiles, an empty expert, a ragged last k-tile
    (torch.bfloat16, [5, 0, 33], 64, 4096),              # thin tiles only
    (torch.bfloat16, [130, 257], 264, 2731),             # a hidden size off the vector (slices cross the gate/up halves)
    (torch.float32, [300, 0, 129, 70, 1], 200, 2808),
    (torch.float32, [260, 256], 1024, 1408),
], ids=["full_thin", "thin", "odd", "fp32", "fp32_dense"])
def test_sliced_products_match_fp64(dtype, counts, D, M):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(51)
    E, R = len(counts), sum(counts)
    offs = [0] + list(itertools.accumulate(counts))
    offsets = torch.tensor(offs, dtype=torch.int32, device=dev)
    dt, s = _lib.dtype_code(dtype), _lib.stream_of(dev)
    vec = 8 if dtype == torch.bfloat16 else 4
    ld = -(-M // vec) * vec

    def rn(*shape, scale=1.0):
        return (torch.randn(*shape, device=dev, generator=gen) * scale).to(dtype)

    def pitched(t):  # rows of ld, zero past M
        return torch.nn.functional.pad(t, (0, ld - M)).contiguous()

    xp, h, dg, du = rn(R, D), pitched(rn(R, M)), pitched(rn(R, M)), pitched(rn(R, M))
    wg, wu, wd = rn(E, D, M, scale=0.05), rn(E, D, M, scale=0.05), rn(E, M, D, scale=0.05)
    wgp, wup = pitched(wg), pitched(wu)
    outs = []
    for _ in range(2):
        nan = lambda *shape: torch.full(shape, float("nan"), dtype=dtype, device=dev)
        y, dx, dwg, dwu = nan(R, D), nan(R, D), nan(E, D, M), nan(E, D, M)
        n1 = _lib.query("abacus_moe_down_fwd_ws_bytes", R, ld, D, E, dt)
        n2 = _lib.query("abacus_experts_gateup_bwd_ws_bytes", R, D, ld, E, dt)
        assert n1 >= 2 * R * D * 4 and n2 >= 2 * R * D * 4, "these shapes are meant to run sliced"
        ws = torch.full((max(n1, n2) // 4,), float("nan"), device=dev)
        if ld != M:
            call("abacus_experts_down_fwd", ptr(h), ptr(wd), ptr(offsets), R, M, ld, D, E, ptr(y), ptr(ws), n1, s)
        else:
            call("abacus_moe_down_fwd", ptr(h), ptr(wd), ptr(offsets), R, M, D, E, dt, ptr(y), ptr(ws), n1, s)
        call("abacus_experts_gateup_bwd", ptr(dg), ptr(du), ptr(wgp), ptr(wup), ptr(xp), ptr(offsets), R, D, M, ld, E, dt,
             ptr(dx), ptr(dwg), ptr(dwu), ptr(_lib.tile_ctr(dev)), ptr(ws), n2, s)
        torch.cuda.synchronize()
        outs.append((y, dx, dwg, dwu))
    for a, b in zip(*outs):
        assert torch.equal(a, b) and not torch.isnan(a).any()
    y, dx, dwg, dwu = outs[0]
    # one rounding to bf16 (2^-9); fp32 sums of at most 5616 terms: sqrt(n) 2^-24 of their norm
    tol = 4e-3 if dtype == torch.bfloat16 else 1e-5
    for e in range(E):
        a, b = offs[e], offs[e + 1]
        if a == b:
            continue
        d = lambda t: t[a:b].double()
        for name, got, want in (
            ("y", y[a:b], d(h)[:, :M] @ wd[e].double()),
            ("dx", dx[a:b], d(dg)[:, :M] @ wg[e].double().t() + d(du)[:, :M] @ wu[e].double().t()),
            ("dwg", dwg[e], d(xp).t() @ d(dg)[:, :M]),
            ("dwu", dwu[e], d(xp).t() @ d(du)[:, :M]),
        ):
            err = float((got.double() - want).norm() / want.norm())
            assert err < tol, f"{name} expert {e}: {err:.3g}"


@pytest.mark.parametrize("dtype,counts,D,M", [
    (torch.float32, [104, 145, 0, 128, 129, 3, 260], 256, 2816),  # experts on both sides of the thin tiles' rows
    (torch.float32, [0] * 7 + [500], 512, 2048),                 # all rows on one expert
    (torch.float32, [1085] * 4 + [1084] * 4, 184, 876),          # the down product sliced for what even rows gain
    (torch.float32, [0] * 7 + [8676], 184, 876),                 # ... on one expert
], ids=["fp32_mixed", "fp32_one_expert", "fp32_for_even_rows", "fp32_for_even_rows_one_expert"])
def test_uneven_sliced_products_match_fp64(dtype, counts, D, M):
    test_sliced_products_match_fp64(dtype, counts, D, M)


@pytest.mark.parametrize("R,D,M,E", [(1024, 1024, 2816, 16), (2048, 1024, 2816, 16), (800, 1024, 2816, 16),
                                     (600, 512, 2048, 8), (512, 128, 2376, 64), (256, 2048, 1408, 32)])
def test_fp32_slices_bound_a_full_tile(R, D, M, E):
    """However the rows are spread, no full 256-row tile's slice (7 us per 32 of the reduction) takes longer than the
    whole launch does unsliced (2.4 us), which an expert with most of the rows would show."""
    n = _lib.query("abacus_moe_down_fwd_ws_bytes", R, M, D, E, _lib.F32)
    slices, k_tiles = max(1, n // (R * D * 4)), -(-M // 32)
    assert slices == 1 or 7.0 * -(-k_tiles // slices) + 8.0 < 2.4 * k_tiles, slices


@pytest.mark.parametrize("counts", [[64] * 8, [0] * 7 + [512]], ids=["even", "one_expert"])
def test_small_fp32_data_gradient(counts):
    """A gate/up data gradient that is sliced although its down product is not, against fp64."""
    R, D, M, E = sum(counts), 128, 256, len(counts)
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(52)
    rn = lambda *shape: torch.randn(*shape, device=dev, generator=gen)
    n = _lib.query("abacus_experts_gateup_bwd_ws_bytes", R, D, M, E, _lib.F32)
    assert n >= 2 * R * D * 4 and _lib.query("abacus_moe_down_fwd_ws_bytes", R, M, D, E, _lib.F32) == 0
    dg, du, x, wg, wu = rn(R, M), rn(R, M), rn(R, D), rn(E, D, M) * 0.05, rn(E, D, M) * 0.05
    offs = [0] + list(itertools.accumulate(counts))
    offsets = torch.tensor(offs, dtype=torch.int32, device=dev)
    dx, ws = torch.full((R, D), float("nan"), device=dev), torch.full((n // 4,), float("nan"), device=dev)
    ctr = torch.zeros(_lib.TILE_CTR_INTS, dtype=torch.int32, device=dev)
    call("abacus_experts_gateup_bwd", ptr(dg), ptr(du), ptr(wg), ptr(wu), ptr(x), ptr(offsets), R, D, M, M, E, _lib.F32,
         ptr(dx), None, None, ptr(ctr), ptr(ws), n, _lib.stream_of(dev))
    for e in range(E):
        a, b = offs[e], offs[e + 1]
        want = dg[a:b].double() @ wg[e].double().t() + du[a:b].double() @ wu[e].double().t()
        # sums of 512 products in fp32, in four parts: at most 128 roundings of 2^-24 each in one of them
        assert a == b or float((dx[a:b].double() - want).norm() / want.norm()) < 128 * 2 ** -24

"""abacus_attention_any_fwd / _bwd: lengths off the 128-query blocks and 64-key tiles, and head dim 128, against fp64
(the bound is derived where it is applied)."""

import math

import pytest
import torch

from abacus_amd import _lib
from abacus_amd import transformer as tr

pytestmark = pytest.mark.gpu


def _exact(q, k, v, scale):
    qh, kh, vh = (t.permute(0, 2, 1, 3) for t in (q, k, v))
    s = (qh @ kh.transpose(-1, -2).contiguous()) * scale
    L = s.shape[-1]
    s = s.masked_fill(torch.ones(L, L, dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    return (torch.softmax(s, dim=-1) @ vh.contiguous()).permute(0, 2, 1, 3), torch.logsumexp(s, dim=-1)


@pytest.mark.parametrize("K", [64, 128])
@pytest.mark.parametrize("B,L,H", [(1, 1, 1), (2, 63, 3), (1, 65, 2), (1, 128, 2), (3, 129, 1), (2, 200, 2),
                                   (1, 1150, 2)])
def test_any_length_matches_fp64(B, L, H, K):
    g = torch.Generator(device="cuda").manual_seed(17)
    q, k, v, dout = (torch.randn(B, L, H, K, device="cuda", generator=g).to(torch.bfloat16) for _ in range(4))
    scale = 1.0 / math.sqrt(K)
    s = _lib.stream_of(q.device)
    nan = lambda *shape, dtype=torch.bfloat16: torch.full(shape, float("nan"), dtype=dtype, device="cuda")
    o, lse2 = nan(B, L, H, K), nan(B, H, L, dtype=torch.float32)
    _lib.call("abacus_attention_any_fwd", _lib.ptr(q), _lib.ptr(k), _lib.ptr(v), B, L, H, K, scale, 1, _lib.ptr(o),
              _lib.ptr(lse2), s)
    dq, dk, dv = nan(B, L, H, K), nan(B, L, H, K), nan(B, L, H, K)
    nbytes = _lib.query("abacus_attention_bwd_ws_bytes", B, L, H)
    ws = torch.empty(nbytes // 4, dtype=torch.float32, device="cuda")
    _lib.call("abacus_attention_any_bwd", _lib.ptr(q), _lib.ptr(k), _lib.ptr(v), _lib.ptr(o), _lib.ptr(dout),
              _lib.ptr(lse2), B, L, H, K, scale, 1, _lib.ptr(dq), _lib.ptr(dk), _lib.ptr(dv), H * K, _lib.ptr(ws), nbytes, s)
    torch.cuda.synchronize()
    leaves = [t.double().requires_grad_() for t in (q, k, v)]
    want, want_lse = _exact(*leaves, scale)
    grads = torch.autograd.grad(want, leaves, dout.double())
    # bounds: o, dq, dk, dv are rounded once, P and dz once each as MFMA operands (2^-9 each); one query attends to
    # one key only, so dq and dk of L = 1 are zero up to the rounding of o
    floor = float(dout.double().norm()) * 4e-3
    for name, got, ref in zip(("o", "dq", "dk", "dv"), (o, dq, dk, dv), (want, *grads)):
        assert torch.isfinite(got.float()).all(), name
        err = float((got.double() - ref).norm())
        assert err <= max(5e-3 * float(ref.norm()), floor if L == 1 else 0.0), f"{name}: {err / float(ref.norm()):.3g}"
    assert float((lse2.double() * math.log(2.0) - want_lse).abs().max()) < 1e-3


@pytest.mark.parametrize("L,K", [(100, 64), (256, 128)])
def test_module_runs_any_kernels(L, K):
    torch.manual_seed(3)
    attn = tr.MultiHeadAttention(2 * K, 2, K).to(torch.bfloat16).cuda()
    rot = tr.Rotary(K).to(torch.bfloat16).cuda()
    x = torch.randn(2, L, 2 * K, device="cuda").to(torch.bfloat16).requires_grad_()
    timer = _lib.KernelTimer()
    with timer:
        attn(x, rot).sum().backward()
    assert {"abacus_attention_any_fwd", "abacus_attention_any_bwd"} <= set(timer.totals_ms())
    assert torch.isfinite(x.grad.float()).all()


@pytest.mark.parametrize("B,L,H,K", [(2, 256, 3, 64), (1, 75, 2, 128), (3, 1, 1, 64)])
def test_joint_node_equals_separate_nodes(B, L, H, K):
    """The attention as one node against the separate nodes (which run while a KernelTimer is active): the same
    kernels on the same operands, so every output and gradient agrees bit for bit; frozen parameters get none."""
    torch.manual_seed(8)
    dim = 96
    attn = tr.MultiHeadAttention(dim, H, K).to(torch.bfloat16).cuda()
    rot = tr.Rotary(K).to(torch.bfloat16).cuda()
    x = torch.randn(B, L, dim, device="cuda").to(torch.bfloat16)
    dy = torch.randn(B, L, dim, device="cuda").to(torch.bfloat16)

    def run():
        xi = x.clone().requires_grad_()
        attn.zero_grad(set_to_none=True)
        y = attn(xi, rot)
        y.backward(dy)
        return [y.detach(), xi.grad] + [p.grad for p in attn.parameters()]

    joint = run()
    with _lib.KernelTimer():
        separate = run()
    for name, a, b in zip(["out", "dx"] + [n for n, _ in attn.named_parameters()], joint, separate):
        assert torch.equal(a, b), name
    with torch.no_grad():
        assert torch.equal(attn(x, rot), joint[0])
    attn.w_k_DHK.requires_grad_(False)
    attn.q_norm.w_gamma_D.requires_grad_(False)
    attn.zero_grad(set_to_none=True)
    attn(x, rot).backward(dy)  # x needs no gradient either
    assert attn.w_k_DHK.grad is None and attn.q_norm.w_gamma_D.grad is None
    assert torch.equal(attn.w_q_DHK.grad, joint[2]) and torch.equal(attn.w_v_DHK.grad, joint[4])


def test_joint_node_takes_weights_at_any_element():
    """Weights that are views into a flat buffer, off the 16-byte vector, give the same gradients."""
    torch.manual_seed(9)
    attn = tr.MultiHeadAttention(64, 2, 64).to(torch.bfloat16).cuda()
    rot = tr.Rotary(64).to(torch.bfloat16).cuda()
    x = torch.randn(2, 70, 64, device="cuda").to(torch.bfloat16)

    def run():
        xi = x.clone().requires_grad_()
        attn.zero_grad(set_to_none=True)
        attn(xi, rot).sum().backward()
        return [xi.grad, attn.w_q_DHK.grad, attn.w_k_DHK.grad, attn.w_v_DHK.grad]

    want = run()
    for name in ("w_q_DHK", "w_k_DHK", "w_v_DHK"):
        w = getattr(attn, name).detach()
        flat = torch.empty(w.numel() + 1, dtype=w.dtype, device="cuda")
        view = flat[1:].view(w.shape).copy_(w)
        setattr(attn, name, torch.nn.Parameter(view))
        assert getattr(attn, name).data_ptr() % 16 != 0
    for a, b in zip(run(), want):
        # the projections' products may be other library kernels at this alignment: one bf16 rounding of the forward
        assert float((a.double() - b.double()).norm()) <= 1.2e-2 * float(b.double().norm())


def test_block_cast_after_a_forward_refuses_the_old_tables():
    """Rotary's tables of an fp32 forward at this length do not fit the block once it is cast to bf16."""
    torch.manual_seed(10)
    attn, rot = tr.MultiHeadAttention(64, 1, 64).cuda(), tr.Rotary(64).cuda()
    x = torch.randn(2, 70, 64, device="cuda")
    with torch.no_grad():
        attn(x, rot)
        attn, rot = attn.to(torch.bfloat16), rot.to(torch.bfloat16)
        with pytest.raises(RuntimeError):
            attn(x.to(torch.bfloat16), rot)
        assert torch.isfinite(attn(x[:, :69].to(torch.bfloat16), rot).float()).all()


def test_any_rejects_head_dims():
    q = torch.zeros(1, 100, 1, 32, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(RuntimeError, match="head_dim"):
        _lib.call("abacus_attention_any_fwd", *([_lib.ptr(q)] * 3), 1, 100, 1, 32, 0.1, 1, _lib.ptr(q), _lib.ptr(q), None)

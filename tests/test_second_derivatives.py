"""Derivatives of the attention block's gradients (create_graph): the kernel nodes have torch's for the same function."""

import contextlib

import pytest
import torch

from abacus_amd import _lib
from abacus_amd import transformer as tr


def _second(block, x, dy, params):
    """d/d(x, params) of a function of every first gradient, (x, dy, params) given."""
    first = torch.autograd.grad(block(x), [x, *params], dy, create_graph=True)
    g = torch.Generator().manual_seed(2)
    loss = sum((f.double() * torch.randn(f.shape, generator=g).to(f.device)).sum() for f in first)
    return torch.autograd.grad(loss, [x, dy, *params])


def test_recorded_gradients_match_torch():
    """_KernelGradient beside autograd's own second derivatives, with one first gradient not asked for (fp32 sums)."""
    torch.manual_seed(1)
    x, gamma, dy = torch.randn(3, 8, requires_grad=True), torch.randn(8, requires_grad=True), torch.randn(3, 8, requires_grad=True)
    op = lambda x, g: tr._norm_op(x, g, 1e-5)
    want = torch.autograd.grad(torch.autograd.grad(op(x, gamma), x, dy, create_graph=True)[0].square().sum(), (x, gamma, dy))
    with torch.no_grad():
        first = torch.autograd.functional.vjp(op, (x, gamma), dy)[1][0]
    assert tr._recorded(op, (first, None), dy, x, gamma)[1] is None
    with torch.no_grad():
        assert tr._recorded(op, (first, None), dy, x, gamma)[0] is first
    got = torch.autograd.grad(tr._recorded(op, (first, None), dy, x, gamma)[0].square().sum(), (x, gamma, dy))
    for a, b in zip(got, want):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("separate", [False, True])
@pytest.mark.parametrize("L,K", [(128, 64), (75, 64), (40, 128)])
def test_attention_block_matches_fp64(L, K, separate):
    """The joint node, and the separate ones (while a KernelTimer is active).  The derivatives are taken in fp32 of
    bf16 operands; the block's intermediates, first gradients and results pass at most 15 bf16 roundings (2^-9 each,
    relative to norms that the sums between them at most keep): 3e-2."""
    torch.manual_seed(11)
    dim, H = 96, 2
    attn, rot = tr.MultiHeadAttention(dim, H, K).to(torch.bfloat16), tr.Rotary(K).to(torch.bfloat16)
    x, dy = (torch.randn(2, L, dim).to(torch.bfloat16) for _ in range(2))

    exact = tr.MultiHeadAttention(dim, H, K).double()
    exact.load_state_dict({k: v.double() for k, v in attn.state_dict().items()})
    cos, sin = (t.reshape(L, K).double() for t in rot(x, seq_dim=1))

    def reference(xi):
        q, k, v = ((xi @ w.flatten(1)).unflatten(2, (H, K)) for w in (exact.w_q_DHK, exact.w_k_DHK, exact.w_v_DHK))
        q, k = (tr._norm_op(t, n.w_gamma_D, 1e-5) for t, n in ((q, exact.q_norm), (k, exact.k_norm)))
        q, k = (t * cos[:, None] + tr.rotate_half(t) * sin[:, None] for t in (q, k))
        return tr._causal_op(q, k, v).flatten(2) @ exact.w_o_HKD.flatten(0, 1)

    leaf = lambda t: t.detach().clone().requires_grad_()
    want = _second(reference, leaf(x.double()), leaf(dy.double()), list(exact.parameters()))
    attn, rot = attn.cuda(), tr.Rotary(K).to(torch.bfloat16).cuda()
    with _lib.KernelTimer() if separate else contextlib.nullcontext():
        got = _second(lambda xi: attn(xi, rot), leaf(x.cuda()), leaf(dy.cuda()), list(attn.parameters()))
    names = ["x", "dy"] + [n for n, _ in attn.named_parameters()]
    for name, a, b in zip(names, got, want):
        err = float((a.double().cpu() - b).norm() / b.norm())
        assert err < 3e-2, f"{name}: {err:.3g}"

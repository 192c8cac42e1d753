"""abacus_token_wgrad (A^T B over the tokens, sliced) against fp64: outputs below, at and past a 256 x 256 tile, token
counts off the 64-token step, slices of unequal length, one and three parts; and the attention block on its route."""

import pytest
import torch

from abacus_amd import _lib
from abacus_amd import transformer as tr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,M,N,parts", [(1, 8, 24, 3), (63, 256, 264, 1), (65, 264, 248, 1), (130, 512, 768, 3),
                                         (1000, 72, 2048, 1), (5003, 200, 312, 3), (4097, 1024, 1024, 1),
                                         (300, 2056, 6144, 3)])
def test_token_wgrad_matches_fp64(T, M, N, parts):
    gen = torch.Generator(device="cuda").manual_seed(T + M)
    a, b = (torch.randn(T, n, device="cuda", generator=gen).to(torch.bfloat16) for n in (M, N))
    nbytes = _lib.query("abacus_token_wgrad_ws_bytes", T, M, N)
    ws = torch.full((nbytes // 4,), float("nan"), dtype=torch.float32, device="cuda")
    out = [torch.full((M, N // parts), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(parts)]
    _lib.call("abacus_token_wgrad", _lib.ptr(a), _lib.ptr(b), T, M, N, parts, *map(_lib.ptr, out + [None] * (3 - parts)),
              _lib.ptr(ws), nbytes, _lib.stream_of(a.device))
    got, want = torch.cat(out, dim=1).double(), a.double().t() @ b.double()
    err = float((got - want).norm() / want.norm())
    assert err < 2 ** -8, err  # one bf16 rounding (at most 2^-9) of fp32 sums


def test_token_wgrad_rejects():
    x = torch.zeros(64, 64, dtype=torch.bfloat16, device="cuda")
    p = _lib.ptr(x)
    for T, M, N, parts, msg in ((8, 12, 8, 1, "not taken"), (8, 8, 8, 2, "parts"), (8, 8, 8, 3, "parts"), (8, 8, 8, 1, "workspace")):
        with pytest.raises(RuntimeError, match=msg):
            _lib.call("abacus_token_wgrad", p, p, T, M, N, parts, p, p, p, p, 0, None)
    assert _lib.query("abacus_token_wgrad_ws_bytes", 8, 12, 8) == -1


def test_attention_block_weight_gradients(monkeypatch):
    """4200 tokens take the sliced kernel: the block's weight gradients against the library's products."""
    torch.manual_seed(3)
    attn = tr.MultiHeadAttention(192, 3, 64).to(torch.bfloat16).cuda()
    rot = tr.Rotary(64).to(torch.bfloat16).cuda()
    x = torch.randn(3, 1400, 192, device="cuda").to(torch.bfloat16)
    dy = torch.randn(3, 1400, 192, device="cuda").to(torch.bfloat16)

    def grads():
        attn.zero_grad(set_to_none=True)
        attn(x, rot).backward(dy)
        return {n: p.grad.double() for n, p in attn.named_parameters()}

    assert _lib.query("abacus_token_wgrad_pays", 4200, 192, 192) == 1
    own = grads()
    monkeypatch.setattr(tr, "_token_wgrad", lambda *_: None)
    for name, want in grads().items():
        assert float((own[name] - want).norm()) <= 2 ** -7 * float(want.norm()), name  # a bf16 rounding on each side


def test_second_derivative_of_the_output_projection():
    """A backward with create_graph keeps the differentiable product."""
    o, dy = (torch.randn(4096, 64, device="cuda").to(torch.bfloat16).requires_grad_() for _ in range(2))
    w = torch.randn(64, 64, device="cuda").to(torch.bfloat16).requires_grad_()
    assert _lib.query("abacus_token_wgrad_pays", 4096, 64, 64) == 1
    (dw,) = torch.autograd.grad(tr._OutProjection.apply(o, w), w, dy, create_graph=True)
    (got,) = torch.autograd.grad(dw.float().sum(), dy)
    want = o.detach().float().sum(dim=1, keepdim=True).expand(4096, 64)  # d/d dy of sum(o^T dy)
    assert float((got.float() - want).norm()) <= 2 ** -8 * float(want.norm())

"""The bf16 layer with a hidden size that is not whole 16-byte vectors (activations padded in their pitch, weights and
their gradients at M columns) against the layer with the same weights zero-padded to whole vectors."""

import pytest
import torch
import torch.nn.functional as F

from abacus_amd.moe import MoE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,D,M,E,K", [
    (300, 64, 129, 4, 2),    # M % 8 = 1: a lone column in the last vector; M % 64 = 1 row past the k-tile
    (700, 72, 263, 8, 2),    # M % 8 = 7
    (2103, 256, 2730, 4, 2),  # M % 8 = 2, the down projection's split tail
    (64, 128, 5, 4, 1),      # less than a vector
    (90, 128, 260, 16, 4),   # thin tiles, experts with few rows
], ids=["mod1", "mod7", "split", "below_vector", "few_rows"])
def test_matches_padded_weights(T, D, M, E, K):
    torch.manual_seed(5)
    a = MoE(D, E, K, hidden_dim=M).to("cuda", torch.bfloat16).eval()
    Mp = -(-M // 8) * 8
    b = MoE(D, E, K, hidden_dim=Mp).to("cuda", torch.bfloat16).eval()
    pad = {"w_gate_EDM": (0, Mp - M), "w_up_EDM": (0, Mp - M), "w_down_EMD": (0, 0, 0, Mp - M)}
    with torch.no_grad():
        for (n, p), (_, q) in zip(a.named_parameters(), b.named_parameters()):
            p.normal_(0.0, 0.05)
            q.copy_(F.pad(p, pad[n]) if n in pad else p)
    x = torch.randn(1, T, D, device="cuda").to(torch.bfloat16)
    dout = torch.randn(1, T, D, device="cuda").to(torch.bfloat16)
    got = []
    for m in (a, b):
        xi = x.clone().requires_grad_()
        out = m(xi)
        out.backward(dout)
        got.append({"out": out.detach(), "dx": xi.grad, **{n: p.grad for n, p in m.named_parameters()}})
    # the padded layer adds exact zeros to the same sums in the same order: equal bit for bit
    for n, g in got[0].items():
        want = got[1][n]
        if n in ("w_gate_EDM", "w_up_EDM"):
            want = want[:, :, :M]
        elif n == "w_down_EMD":
            want = want[:, :M]
        assert torch.equal(g, want), n
    with torch.no_grad():  # without gradients: the same forward, or the decode kernels' where the batch is small
        err = float((a(x).float() - got[0]["out"].float()).norm() / got[0]["out"].float().norm())
    assert err < 1e-2


def test_frozen_weights_get_no_gradient():
    torch.manual_seed(6)
    moe = MoE(64, 4, 2, hidden_dim=100).to("cuda", torch.bfloat16)
    moe.w_up_EDM.requires_grad_(False)
    moe.w_down_EMD.requires_grad_(False)
    moe(torch.randn(1, 50, 64, device="cuda").to(torch.bfloat16)).sum().backward()
    assert moe.w_up_EDM.grad is None and moe.w_down_EMD.grad is None
    assert moe.w_gate_EDM.grad.shape == moe.w_gate_EDM.shape and torch.isfinite(moe.w_gate_EDM.grad.float()).all()

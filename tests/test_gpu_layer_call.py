"""The MoE layer as one call per direction (abacus_layer_fwd / _bwd) against the same entry points called one by one,
which run while a KernelTimer is active; and backwards that are asked for some of the gradients only."""

import contextlib

import pytest
import torch

from abacus_amd import _lib, moe
from abacus_amd.moe import MoE

pytestmark = pytest.mark.gpu

PARAMS = ("router.w_DE", "w_gate_EDM", "w_up_EDM", "w_down_EMD")
BF16, F32 = torch.bfloat16, torch.float32
SHAPES = [  # dtype, T, D, M, E, K
    (BF16, 300, 64, 256, 4, 2),
    (BF16, 300, 64, 129, 4, 2),     # rows of the hidden activations padded to whole vectors
    (BF16, 130, 256, 4100, 8, 2),   # ... with the data gradient in slices
    (BF16, 130, 256, 4096, 8, 2),   # the data gradient in slices
    (F32, 260, 128, 256, 8, 2),
    (BF16, 40, 72, 60, 4, 1),
]


def _layer(dtype, T, D, M, E, K):
    torch.manual_seed(12)
    layer = MoE(D, E, K, hidden_dim=M).to("cuda", dtype)
    x, dy = (torch.randn(1, T, D, device="cuda").to(dtype) for _ in range(2))
    return layer, x, dy


def _run(layer, x, dy, need_x=True):
    layer.zero_grad(set_to_none=True)
    layer.router.expert_bias_E.zero_()
    xi = x.clone().requires_grad_(need_x)
    out = layer(xi)
    out.backward(dy)
    r = layer.router.last_routing
    return {"out": out.detach(), "x": xi.grad, "bias": layer.router.expert_bias_E.clone(),
            **{n: p.grad for n, p in layer.named_parameters()},
            **{n: getattr(r, n).clone() for n in ("logits_TE", "weights_TK", "indices_TK", "counts_E", "offsets_E1",
                                                  "perm_R", "pos_TK")}}


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_one_call_equals_the_entry_points(shape):
    layer, x, dy = _layer(*shape)
    one = _run(layer, x, dy)
    with _lib.KernelTimer():
        separate = _run(layer, x, dy)
    for name, a in one.items():
        assert torch.equal(a, separate[name]), name
    layer.eval()
    with torch.no_grad():
        out = layer(x)
        with _lib.KernelTimer():
            assert torch.equal(out, layer(x))


@pytest.mark.parametrize("separate", [False, True])
@pytest.mark.parametrize("wanted", [{"x"}, {"w_down_EMD"}, {"w_gate_EDM"}, {"router.w_DE"}, {"x", "w_up_EDM"},
                                    {"x", "w_down_EMD", "router.w_DE"}], ids=lambda w: "+".join(sorted(w)))
@pytest.mark.parametrize("shape", SHAPES[:4], ids=str)
def test_some_gradients_only(shape, wanted, separate):
    """The gradients asked for equal those of the whole backward; the others are not formed."""
    layer, x, dy = _layer(*shape)
    whole = _run(layer, x, dy)
    for name, p in layer.named_parameters():
        p.requires_grad_(name in wanted)
    with _lib.KernelTimer() if separate else contextlib.nullcontext():
        some = _run(layer, x, dy, need_x="x" in wanted)
    for name in ("x", *PARAMS):
        if name not in wanted:
            assert some[name] is None, name
            continue
        # (alone, a gradient's launch may choose other slices of its sums: one bf16 rounding apart)
        err = float((some[name].double() - whole[name].double()).norm() / whole[name].double().norm())
        assert err <= 2 ** -8, (name, err)


def test_frozen_experts_hand_the_backward_no_weight_gradients(monkeypatch):
    """A hidden size off the vector too: no product is formed for weights that want no gradient."""
    layer, x, dy = _layer(*SHAPES[1])
    for name, p in layer.named_parameters():
        p.requires_grad_(name == "router.w_DE")
    made, call = [], moe.call
    monkeypatch.setattr(moe, "call", lambda name, *args: (made.append((name, args)), call(name, *args))[1])
    _run(layer, x, dy)
    (args,) = [a for n, a in made if n == "abacus_layer_bwd"]
    assert args[-4:-1] == (None, None, None)  # dw_gate, dw_up, dw_down


def test_routing_record_may_be_changed():
    """The layer's routing record belongs to the caller: what the backward does not read may change before it."""
    layer, x, dy = _layer(*SHAPES[0])
    want = _run(layer, x, dy)
    layer.zero_grad(set_to_none=True)
    layer.router.expert_bias_E.zero_()
    xi = x.clone().requires_grad_()
    out = layer(xi)
    r = layer.router.last_routing
    for t in (r.logits_TE, r.indices_TK, r.counts_E, r.perm_R):
        t.zero_()
    out.backward(dy)
    assert torch.equal(xi.grad, want["x"]) and torch.equal(layer.w_up_EDM.grad, want["w_up_EDM"])
    out = layer(xi)
    layer.router.last_routing.weights_TK.zero_()  # the backward reads these
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(dy)

"""Performance cases of the framework: what a program that uses it calls, over the sizes it calls it with.

Each listed case is one public entry point (the MoE layer in inference and in training, the attention block,
the token loss, the optimizer, a whole decoder step) at a size taken from this repository's workloads, tests and
benchmark, or a plain generic one; ``draw`` gives further cases of the same ranges.  The path a case takes is
in its ``"path"``:

  moe_infer   MoE.forward in eval mode under no_grad (decode steps and prompt chunks)
  moe_train   MoE.forward + backward in train mode (router bias step included), gradients of x and all weights
  attention   MultiHeadAttention forward + backward (projections, q/k norm + rotary embedding, causal attention)
  loss        cross_entropy forward + backward over (tokens, vocabulary) logits
  optimizer   one AdamW step
  decoder     TransformerMoe forward, next-token loss and backward
"""

from __future__ import annotations

import math

import torch

from abacus.attention import MultiHeadAttention
from abacus.kernels.liger import cross_entropy
from abacus.moe.moe import MoE
from abacus.optimizers.adamw import AdamW
from abacus.rope import Rotary
from abacus.transformer_moe import TransformerMoe
from abacus_amd.train import next_token_loss
from abacus_amd.workloads import zipf_bias

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _moe(path, batch, seq, dim, hidden, experts, top_k, dtype, skew=False):
    return {"path": path, "batch": batch, "seq": seq, "dim": dim, "hidden": hidden, "experts": experts,
            "top_k": top_k, "dtype": dtype, "skew": skew}


def _attention(batch, seq, heads, head_dim, dtype):
    return {"path": "attention", "batch": batch, "seq": seq, "heads": heads, "head_dim": head_dim, "dtype": dtype}


def listed():
    cases = {
        # one token of one sequence through the Mixtral-shaped layer: the latency of a decode step
        "infer_mixtral_T1": _moe("moe_infer", 1, 1, 4096, 14336, 8, 2, "bf16"),
        # a decode step of 64 sequences through a many-expert layer with Zipf-skewed routing
        "infer_skewed_T64": _moe("moe_infer", 64, 1, 2048, 1408, 64, 6, "bf16", skew=True),
        # a prompt chunk (or a large decode batch) of 512 tokens through the same layer
        "infer_skewed_T512": _moe("moe_infer", 1, 512, 2048, 1408, 64, 6, "bf16", skew=True),
        # the smallest training layer, where launches and host time are most of the step
        "train_tiny_fp32": _moe("moe_train", 2, 128, 128, 256, 8, 2, "fp32"),
        # the largest layer: the Mixtral shape, 4096 tokens
        "train_mixtral_bf16": _moe("moe_train", 2, 2048, 4096, 14336, 8, 2, "bf16"),
        # a fine-grained layer: many small experts
        "train_finegrained_bf16": _moe("moe_train", 4, 2048, 2048, 768, 128, 8, "bf16"),
        # sizes nobody rounded: hidden = int(8 / 3 * dim), a token count off every tile
        "train_ragged_bf16": _moe("moe_train", 3, 701, 1024, 2730, 16, 2, "bf16"),
        # the decoder's attention block at its training size
        "attention_L2048_bf16": _attention(4, 2048, 16, 64, "bf16"),
        # the same block on sequences as long as the data has them
        "attention_L1500_bf16": _attention(3, 1500, 16, 64, "bf16"),
        # the token loss over a 32000-word vocabulary
        "loss_V32000_bf16": {"path": "loss", "tokens": 8192, "vocab": 32000, "dtype": "bf16"},
        # the optimizer over one large block's weights and the token tables
        "optimizer_bf16": {"path": "optimizer", "dim": 2048, "experts": 8, "dtype": "bf16"},
        # two layers of the decoder in fp32, whole: forward, loss and backward (its MoE layer is the mid-size one)
        "decoder_fp32": {"path": "decoder", "batch": 4, "seq": 512, "dim": 1024, "heads": 16, "blocks": 2,
                         "vocab": 32000, "experts": 16, "top_k": 2, "hidden": 2816, "dtype": "fp32"},
    }
    return [{"name": name, **case} for name, case in cases.items()]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _draw_layer(rng, largest_hidden):
    dim = 64 * _log(rng, 4, 64) if rng.random() < 0.7 else 8 * _log(rng, 32, 512)
    kind = rng.random()
    hidden = (64 * _log(rng, 4, largest_hidden // 64) if kind < 0.6 else 8 * _log(rng, 32, largest_hidden // 8)
              if kind < 0.8 else _log(rng, 256, largest_hidden))
    experts = rng.choice((4, 8, 8, 16, 16, 32, 64, 64, 128))
    top_k = rng.choice([k for k in (1, 2, 2, 4, 6, 8) if k <= experts // 2])
    return dim, hidden, experts, top_k


def draw(rng):
    path = rng.choice(("moe_infer", "moe_infer", "moe_infer", "moe_train", "moe_train", "moe_train", "attention",
                       "loss", "optimizer", "decoder"))
    if path in ("moe_infer", "moe_train"):
        train = path == "moe_train"
        while True:
            dim, hidden, experts, top_k = _draw_layer(rng, 14336)
            tokens = _log(rng, 128, 16384) if train else _log(rng, 1, 2048)
            dtype = "fp32" if rng.random() < 0.25 else "bf16"
            flops = (18.0 if train else 6.0) * tokens * top_k * dim * hidden
            weights = 3.0 * experts * dim * hidden
            if weights <= 1.5e9 and flops <= (8e12 if dtype == "bf16" else 8e11):
                break
        skew = rng.random() < 0.5 and experts >= 16
        return _moe(path, 1, tokens, dim, hidden, experts, top_k, dtype, skew)
    if path == "attention":
        seq = _log(rng, 64, 4096)
        return _attention(rng.randint(1, max(1, min(8, 12288 // seq))), seq, rng.choice((8, 12, 16)),
                          rng.choice((64, 64, 64, 128)), rng.choice(("bf16", "bf16", "bf16", "fp32")))
    if path == "loss":
        return {"path": "loss", "tokens": _log(rng, 128, 8192), "vocab": rng.choice((32000, 50257, 65536)),
                "dtype": rng.choice(("bf16", "bf16", "fp32"))}
    if path == "optimizer":
        return {"path": "optimizer", "dim": 64 * _log(rng, 4, 32), "experts": rng.choice((4, 8)),
                "dtype": rng.choice(("bf16", "fp32"))}
    return {"path": "decoder", "batch": rng.randint(1, 3), "seq": _log(rng, 64, 512), "dim": rng.choice((512, 768, 1024)),
            "heads": 8, "blocks": 2, "vocab": rng.choice((8000, 32000)), "experts": rng.choice((8, 16)), "top_k": 2,
            "hidden": 128 * rng.randint(4, 16), "dtype": "fp32"}


def _generator(case, seed):
    return torch.Generator(device="cuda").manual_seed(1_000_003 * (seed + 1) % (1 << 40))


def _normal(gen, shape, std, dtype):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(0.0, std, generator=gen)


def _on_gpu(make, dtype):
    """The module with its storage on the GPU, in `dtype`, values still to be drawn."""
    with torch.device("meta"):
        module = make()
    return module.to(dtype).to_empty(device="cuda")


def _fill_moe(moe, gen, skew):
    with torch.no_grad():
        for p in (moe.router.w_DE, moe.w_gate_EDM, moe.w_up_EDM, moe.w_down_EMD):
            p.normal_(0.0, 0.02, generator=gen)
        moe.router.expert_bias_E.zero_()
        if skew:
            moe.router.expert_bias_E.copy_(zipf_bias(moe.n_experts))


def _fill_attention(attention, gen):
    with torch.no_grad():
        for p in (attention.w_q_DHK, attention.w_k_DHK, attention.w_v_DHK, attention.w_o_HKD):
            p.normal_(0.0, attention.dim ** -0.5, generator=gen)
        for norm in (attention.q_norm, attention.k_norm):
            norm.w_gamma_D.normal_(1.0, 0.1, generator=gen)


def _rotary(head_dim, dtype):
    return Rotary(head_dim).to(device="cuda", dtype=dtype)


def _optimizer_shapes(case):
    D, E = case["dim"], case["experts"]
    return [(8000, D), (D,), (D, D), (D, D), (D, D), (D, D), (64,), (64,), (D,), (D, E), (E, D, 2 * D + 8),
            (E, D, 2 * D + 8), (E, 2 * D + 8, D), (D,), (D, 8000)]


class _Weights(torch.nn.Module):
    def __init__(self, tensors):
        super().__init__()
        self.tensors = torch.nn.ParameterList(tensors)


def prepare(case, seed):
    gen, dtype, path = _generator(case, seed), DTYPES[case["dtype"]], case["path"]
    state = {"path": path}
    if path in ("moe_infer", "moe_train"):
        moe = _on_gpu(lambda: MoE(case["dim"], case["experts"], case["top_k"], hidden_dim=case["hidden"]), dtype)
        _fill_moe(moe, gen, case["skew"])
        shape = (case["batch"], case["seq"], case["dim"])
        state["module"], state["x"] = moe, _normal(gen, shape, 1.0, dtype)
        if path == "moe_infer":
            moe.eval()
        else:
            moe.train()
            state["x"].requires_grad_()
            state["dout"] = _normal(gen, shape, 1.0 / (case["batch"] * case["seq"]), dtype)
    elif path == "attention":
        dim = case["heads"] * case["head_dim"]
        attention = _on_gpu(lambda: MultiHeadAttention(dim, case["heads"], case["head_dim"]), dtype)
        _fill_attention(attention, gen)
        shape = (case["batch"], case["seq"], dim)
        state.update(module=attention, rotary=_rotary(case["head_dim"], dtype),
                     x=_normal(gen, shape, 1.0, dtype).requires_grad_(),
                     dout=_normal(gen, shape, 1.0 / (case["batch"] * case["seq"]), dtype))
    elif path == "loss":
        shape = (case["tokens"], case["vocab"])
        state["logits"] = _normal(gen, shape, 2.0, dtype).requires_grad_()
        targets = torch.randint(0, case["vocab"], (case["tokens"],), device="cuda", generator=gen)
        padded = torch.rand(case["tokens"], device="cuda", generator=gen) < 0.02
        state["targets"] = targets.masked_fill(padded, -100)
    elif path == "optimizer":
        shapes = _optimizer_shapes(case)
        state["model"] = _Weights([_normal(gen, s, 0.02, dtype) for s in shapes])
        for p in state["model"].parameters():
            p.grad = _normal(gen, p.shape, 1e-3, dtype)
        state["optimizer"] = AdamW(state["model"])
    else:
        model = _on_gpu(lambda: TransformerMoe(case["dim"], case["heads"], case["dim"] // case["heads"],
                                               case["blocks"], case["vocab"], case["experts"], case["top_k"],
                                               hidden_dim=case["hidden"]), dtype)
        model.rotary = _rotary(case["dim"] // case["heads"], dtype)
        with torch.no_grad():
            model.embedding.w_vocab_D.normal_(0.0, 1.0, generator=gen)
            model.w_D_vocab.normal_(0.0, case["dim"] ** -0.5, generator=gen)
            model.norm.w_gamma_D.normal_(1.0, 0.1, generator=gen)
            for block in model.blocks:
                block.norm_attention.w_gamma_D.normal_(1.0, 0.1, generator=gen)
                block.norm_mlp.w_gamma_D.normal_(1.0, 0.1, generator=gen)
                _fill_attention(block.attention, gen)
                _fill_moe(block.moe, gen, False)
        model.train()
        state["module"] = model
        state["tokens"] = torch.randint(0, case["vocab"], (case["batch"], case["seq"]), device="cuda", generator=gen)
    return state


def _grads(module):
    return {name: p.grad for name, p in module.named_parameters()}


def run(state):
    path = state["path"]
    if path == "moe_infer":
        with torch.no_grad():
            return {"out": state["module"](state["x"])}
    if path in ("moe_train", "attention"):
        module, x = state["module"], state["x"]
        module.zero_grad(set_to_none=True)
        x.grad = None
        out = module(x) if path == "moe_train" else module(x, state["rotary"])
        out.backward(state["dout"])
        got = {"out": out.detach(), "dx": x.grad, **_grads(module)}
        if path == "moe_train":
            got["bias"] = module.router.expert_bias_E
        return got
    if path == "loss":
        logits = state["logits"]
        logits.grad = None
        loss = cross_entropy(logits, state["targets"])
        loss.backward()
        return {"loss": loss.detach(), "dlogits": logits.grad}
    if path == "optimizer":
        optimizer = state["optimizer"]
        optimizer.step()
        return {"weights": [p.detach() for p in optimizer.params],
                "moments": [optimizer.state[id(p)][m] for p in optimizer.params for m in ("exp_avg", "exp_avg_sq")]}
    model = state["module"]
    model.zero_grad(set_to_none=True)
    logits = model(state["tokens"])
    loss = next_token_loss(logits, state["tokens"])
    loss.backward()
    return {"logits": logits.detach(), "loss": loss.detach(), **_grads(model)}


def _bytes(case):
    return 2 if case["dtype"] == "bf16" else 4


def work(case):
    s, path = _bytes(case), case["path"]
    if path in ("moe_infer", "moe_train"):
        D, M, E, K, T = case["dim"], case["hidden"], case["experts"], case["top_k"], case["batch"] * case["seq"]
        touched = E * (1.0 - (1.0 - K / E) ** T)  # experts that a batch of T tokens reaches, routed evenly
        if path == "moe_infer":
            return {"bytes": s * (3 * touched * D * M + 2 * T * D + D * E), "flops": 6.0 * T * K * D * M + 2.0 * T * D * E}
        return {"bytes": s * (3 * (touched + E) * D * M + 4 * T * D + 2 * D * E),
                "flops": 18.0 * T * K * D * M + 6.0 * T * D * E}
    if path == "attention":
        T, H = case["batch"] * case["seq"], case["heads"]
        D = H * case["head_dim"]
        return {"bytes": s * (4 * T * D + 8 * D * D), "flops": 24.0 * T * D * D + 7.0 * T * case["seq"] * D}
    if path == "loss":
        n = case["tokens"] * case["vocab"]
        return {"bytes": 2.0 * s * n, "flops": 6.0 * n}
    if path == "optimizer":
        n = sum(math.prod(shape) for shape in _optimizer_shapes(case))
        return {"bytes": 7.0 * s * n, "flops": 12.0 * n}
    D, L, V, T = case["dim"], case["seq"], case["vocab"], case["batch"] * case["seq"]
    block_weights = 4 * D * D + 3 * case["experts"] * D * case["hidden"]
    flops = case["blocks"] * (24.0 * T * D * D + 7.0 * T * L * D + 18.0 * T * case["top_k"] * D * case["hidden"])
    return {"bytes": s * (2.0 * (case["blocks"] * block_weights + 2 * V * D) + T * V), "flops": flops + 6.0 * T * D * V}


def tolerance(case):
    fine = case["dtype"] == "fp32"
    if case["path"] == "optimizer":
        # one rounding of the update in the weights' type, moments rounded at each step of their sum
        return {"rel": 1e-6, "max": 1e-4} if fine else {"rel": 4e-3, "max": 0.05}
    if case["path"] == "loss":
        return {"rel": 2e-6, "max": 1e-4} if fine else {"rel": 4e-3, "max": 0.05}
    if fine:
        return {"rel": 1e-5, "max": 2e-3}
    # bf16 layers: every product is rounded to bf16 before the next one reads it
    return {"rel": 1.2e-2, "max": 0.5}


# ---------------------------------------------------------------------------
# The same results in 64 bits, in plain torch.  Routing is the one discrete step: experts are picked on the logits
# and scores as the layer's type holds them, ties to the lower index.
# ---------------------------------------------------------------------------


def _exact_moe(x, w_DE, bias, w_gate, w_up, w_down, top_k, dtype):
    logits = x @ w_DE
    held = logits.detach().float().to(dtype).double()
    score = torch.sigmoid(held).float().to(dtype)
    value = (score.float() + bias.float()).to(dtype)
    picked = torch.sort(value, dim=-1, descending=True, stable=True).indices[:, :top_k]
    chosen = torch.sigmoid(logits).gather(1, picked)
    weights = chosen / chosen.sum(dim=-1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(w_DE.shape[1]):
        token, slot = torch.nonzero(picked == e, as_tuple=True)
        if token.numel() == 0:
            continue
        rows = x[token]
        gate = rows @ w_gate[e].double()
        y = (gate * torch.sigmoid(gate) * (rows @ w_up[e].double())) @ w_down[e].double()
        out = out.index_add(0, token, y * weights[token, slot].unsqueeze(1))
    return out, picked


def _exact_norm(x, gamma):
    return gamma * x / torch.sqrt(x.square().mean(dim=-1, keepdim=True) + 1e-5)


def _exact_attention(x, p, heads, cos, sin):
    B, L, D = x.shape
    K = D // heads

    def rotated(t):
        return t * cos + torch.cat((-t[..., K // 2:], t[..., :K // 2]), dim=-1) * sin

    q, k, v = ((x.reshape(B * L, D) @ p[n].reshape(D, D)).view(B, L, heads, K) for n in ("w_q_DHK", "w_k_DHK", "w_v_DHK"))
    q, k = rotated(_exact_norm(q, p["q_norm.w_gamma_D"])), rotated(_exact_norm(k, p["k_norm.w_gamma_D"]))
    later = torch.ones(L, L, dtype=torch.bool, device=x.device).triu_(1)
    outs = []
    for b in range(B):
        s = q[b].transpose(0, 1).contiguous() @ k[b].permute(1, 2, 0).contiguous() / math.sqrt(K)
        outs.append((torch.softmax(s.masked_fill(later, float("-inf")), dim=-1) @ v[b].transpose(0, 1).contiguous())
                    .transpose(0, 1).reshape(L, D))
    return torch.stack(outs) @ p["w_o_HKD"].reshape(D, D)


def _doubles(module):
    return {n: p.detach().double().requires_grad_() for n, p in module.named_parameters()}


def _tables(rotary, x, seq):
    cos, sin = rotary._angles(x, torch.arange(seq, device="cuda"))
    return cos.double().reshape(seq, 1, -1), sin.double().reshape(seq, 1, -1)


def exact(case, seed):
    state, path, dtype = prepare(case, seed), case["path"], DTYPES[case["dtype"]]
    if path in ("moe_infer", "moe_train"):
        moe, train = state["module"], path == "moe_train"
        x = state["x"].detach().double().requires_grad_(train)
        p = {n: (t.detach().double() if train else t.detach()).requires_grad_(train) for n, t in moe.named_parameters()}
        w_DE = p["router.w_DE"].double()
        with torch.set_grad_enabled(train):
            out, _ = _exact_moe(x.reshape(-1, case["dim"]), w_DE, moe.router.expert_bias_E, p["w_gate_EDM"],
                                p["w_up_EDM"], p["w_down_EMD"], case["top_k"], dtype)
            out = out.view(x.shape)
        if not train:
            return {"out": out}
        out.backward(state["dout"].double())
        got = {"out": out.detach(), "dx": x.grad, "bias": None}
        for n, t in p.items():
            got[n] = torch.zeros_like(t) if t.grad is None else t.grad
        if case["top_k"] == 1:  # a lone weight is 1 whatever the logit: the gradient is zero, and nothing but rounding here
            got["router.w_DE"] = None
        return got
    if path == "attention":
        x, p = state["x"].detach().double().requires_grad_(), _doubles(state["module"])
        cos, sin = _tables(state["rotary"], state["x"], case["seq"])
        out = _exact_attention(x, p, case["heads"], cos, sin)
        out.backward(state["dout"].double())
        return {"out": out.detach(), "dx": x.grad, **{n: t.grad for n, t in p.items()}}
    if path == "loss":
        logits = state["logits"].detach().double().requires_grad_()
        loss = torch.nn.functional.cross_entropy(logits, state["targets"])
        loss.backward()
        return {"loss": loss.detach(), "dlogits": logits.grad}
    if path == "optimizer":
        lr, b1, b2, eps, decay = 1e-3, 0.9, 0.999, 1e-8, 1e-2
        weights, moments = [], []
        for p in state["model"].parameters():
            g = p.grad.double()
            m, v = (1 - b1) * g, (1 - b2) * g * g
            weights.append(p.detach().double() * (1 - lr * decay) - lr * (m / (1 - b1)) / ((v / (1 - b2)).sqrt() + eps))
            moments += [m, v]
        return {"weights": weights, "moments": moments}
    model, tokens = state["module"], state["tokens"]
    p = _doubles(model)
    x = p["embedding.w_vocab_D"][tokens]
    cos, sin = _tables(model.rotary, model.w_D_vocab, case["seq"])
    for i, block in enumerate(model.blocks):
        own = {n[len("blocks.%d." % i):]: t for n, t in p.items() if n.startswith("blocks.%d." % i)}
        attention = {n[len("attention."):]: t for n, t in own.items() if n.startswith("attention.")}
        x = x + _exact_attention(_exact_norm(x, own["norm_attention.w_gamma_D"]), attention, case["heads"], cos, sin)
        h = _exact_norm(x, own["norm_mlp.w_gamma_D"]).reshape(-1, case["dim"])
        y, _ = _exact_moe(h, own["moe.router.w_DE"], block.moe.router.expert_bias_E, own["moe.w_gate_EDM"],
                          own["moe.w_up_EDM"], own["moe.w_down_EMD"], case["top_k"], dtype)
        x = x + y.view(x.shape)
    logits = _exact_norm(x, p["norm.w_gamma_D"]) @ p["w_D_vocab"]
    loss = torch.nn.functional.cross_entropy(logits[:, :-1].reshape(-1, case["vocab"]), tokens[:, 1:].reshape(-1))
    loss.backward()
    return {"logits": logits.detach(), "loss": loss.detach(), **{n: t.grad for n, t in p.items()}}

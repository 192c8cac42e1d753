"""Which attention inputs reach the GPU kernels, decided on the host: checked without a GPU on fake CUDA tensors, with
the library's calls recorded instead of made."""

import contextlib

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from abacus_amd import transformer as tr


@pytest.fixture
def calls(monkeypatch):
    made = []
    monkeypatch.setattr(tr._lib, "call", lambda name, *args: made.append(name))
    monkeypatch.setattr(tr._lib, "ptr", lambda t: 0)
    monkeypatch.setattr(tr._lib, "stream_of", lambda device: 0)
    with FakeTensorMode():
        yield made


def _block(head_dim=64, dtype=torch.bfloat16):
    with torch.device("cuda"):
        attn, rot = tr.MultiHeadAttention(2 * head_dim, 2, head_dim), tr.Rotary(head_dim)
    for module in attn.modules():
        for name, p in list(module.named_parameters(recurse=False)):
            setattr(module, name, torch.nn.Parameter(p.detach().to(dtype)))
    rot.inv_freq = rot.inv_freq.to(dtype)
    return attn, rot


def _x(head_dim=64, dtype=torch.bfloat16):
    return torch.empty(2, 9, 2 * head_dim, device="cuda", dtype=dtype)


def test_tables_of_the_inputs_type_take_the_joint_node(calls):
    attn, rot = _block()
    attn(_x(), rot)
    assert calls == ["abacus_qk_norm_rope_fwd", "abacus_attention_any_fwd"]


@pytest.mark.parametrize("stale", [dict(dtype=torch.float32), dict(device="cpu")])
def test_tables_cached_for_another_type_or_device_are_refused(calls, stale):
    """Rotary caches its tables by length alone, so a module cast or moved afterwards hands on the old ones: no kernel
    reads them (torch's products refuse them on the GPU; fake tensors let a type through)."""
    attn, rot = _block()
    rot(_x(), seq_dim=1)
    rot.cos_cached, rot.sin_cached = rot.cos_cached.to(**stale), rot.sin_cached.to(**stale)
    with contextlib.suppress(RuntimeError):
        attn(_x(), rot)
    assert not any("rope" in name for name in calls)


def test_block_without_rotary_takes_any_norms():
    """Without a rotary embedding the q and k norms are only called: any module will do."""
    attn = tr.MultiHeadAttention(16, 2, 8)
    attn.q_norm, attn.k_norm = torch.nn.Identity(), torch.nn.LayerNorm(8)
    assert attn(torch.randn(2, 5, 16)).shape == (2, 5, 16)


def test_norm_weights_of_another_length_stay_with_torch(calls):
    """A weight that broadcasts over the row is not the row of weights that the kernels read."""
    attn, rot = _block()
    attn.q_norm.w_gamma_D = torch.nn.Parameter(torch.empty(1, device="cuda", dtype=torch.bfloat16))
    assert attn(_x(), rot).shape == (2, 9, 128)
    assert "abacus_rmsnorm_fwd" in calls and not any("rope" in name for name in calls)  # k_norm's kernel only
    assert calls.count("abacus_rmsnorm_fwd") == 1

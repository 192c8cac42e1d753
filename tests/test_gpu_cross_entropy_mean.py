"""cross_entropy's mean on the device: row sums and counts of one and several passes of the mean kernel, vocabularies
off the vector (rows at any alignment), an ignore index of its own, no rows left, against fp64."""

import math

import pytest
import torch
import torch.nn.functional as F

from abacus_amd import _lib
from abacus_amd.train import cross_entropy, next_token_loss

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("N,V,ignore", [(1, 7, -100), (1024, 64, 3), (1025, 65, -100), (3001, 50257, -100),
                                        (5000, 129, 0), (37, 1030, -100)])
def test_mean_matches_fp64(dtype, N, V, ignore):
    g = torch.Generator(device="cuda").manual_seed(N + V)
    x = (torch.randn(N, V, device="cuda", generator=g) * 3).to(dtype).requires_grad_()
    t = torch.randint(0, V, (N,), device="cuda", generator=g)
    t[1::5] = ignore
    loss = cross_entropy(x, t, ignore_index=ignore)
    upstream = torch.tensor(0.75, device="cuda", dtype=dtype)
    (grad,) = torch.autograd.grad(loss, x, upstream)
    ref_x = x.detach().double().requires_grad_()
    ref = F.cross_entropy(ref_x, t, ignore_index=ignore)
    (ref_grad,) = torch.autograd.grad(ref, ref_x, upstream.double())
    # one rounding to the dtype (bf16 2^-9) over fp32 sums
    assert loss.dtype == dtype and loss.shape == ()
    assert abs(float(loss.detach()) - float(ref.detach())) <= (2 ** -8 if dtype == torch.bfloat16 else 1e-5) * abs(float(ref.detach()))
    err = float((grad.double() - ref_grad).norm() / ref_grad.norm())
    assert err <= (4e-3 if dtype == torch.bfloat16 else 1e-5), err
    assert torch.count_nonzero(grad[t == ignore]) == 0


def test_no_rows_left_is_nan():
    x = torch.randn(4, 16, device="cuda").requires_grad_()
    loss = cross_entropy(x, torch.full((4,), -100, device="cuda"))
    assert torch.isnan(loss.detach())
    loss.backward()
    assert torch.count_nonzero(x.grad) == 0
    assert torch.isnan(cross_entropy(torch.randn(0, 16, device="cuda"), torch.zeros(0, dtype=torch.int64, device="cuda")))



def test_count_of_many_rows_is_rounded_once():
    """More rows than fp32 counts exactly: the count is the exact one, rounded once."""
    N, V = 3 << 24, 8
    x = torch.zeros(N, V, device="cuda", dtype=torch.bfloat16)
    t = torch.zeros(N, device="cuda", dtype=torch.int64)
    for wave in range(9, 16):  # odd sums of the waves past the first 2^24 rows
        t[wave * 64:wave * 64 + 3] = -100
    rows = torch.empty(2, N, device="cuda")
    loss, count = torch.empty((), device="cuda", dtype=torch.bfloat16), torch.empty((), device="cuda")
    _lib.call("abacus_cross_entropy_mean_fwd", _lib.ptr(x), _lib.ptr(t), N, V, -100, _lib.BF16, rows.data_ptr(),
              rows[1].data_ptr(), _lib.ptr(loss), _lib.ptr(count), _lib.stream_of(x.device))
    assert float(count) == float((t != -100).sum().float())


def test_sum_of_many_rows_keeps_its_digits():
    """The row losses of a large batch are added without the error of a long fp32 chain (row losses: 1e-6)."""
    N = 1 << 24
    x = torch.zeros(N, 4, device="cuda")
    loss = cross_entropy(x, torch.zeros(N, device="cuda", dtype=torch.int64))
    assert abs(float(loss) - math.log(4.0)) <= 2e-6 * math.log(4.0)


def test_targets_on_the_cpu_raise():
    x, t = torch.randn(1, 5, 16, device="cuda"), torch.zeros(1, 5, dtype=torch.int64)
    with pytest.raises(RuntimeError):
        cross_entropy(x[0], t[0])
    with pytest.raises(RuntimeError):
        next_token_loss(x, t)

"""The mean of the loss and its gradient in one launch each, and the squared norm, against 64 bits."""

import pytest
import torch

from llmctl import ops
from llmctl.ops._lib import native

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("T", [1, 63, 1025, 32768, 32769])
def test_mean_and_gradient(T):
    torch.manual_seed(T)
    logits = torch.randn(T, 41, device="cuda").bfloat16()
    labels = torch.randint(0, 41, (T,), device="cuda")
    labels[::7] = -100
    rows, lse = native().cross_entropy_fwd(logits, labels, -100)
    want = rows.double().sum() / (T + 2)
    x = logits.clone().requires_grad_()
    loss = ops.cross_entropy(x, labels, reduction_denom=float(T + 2))
    # one launch: summed in 64 bits, rounded twice; beyond 32768 rows the library's sum of 32-bit partial sums (some 64 additions a thread and its tree) and quotient
    assert loss.shape == () and (loss.double() - want).abs() <= (4 if T <= 32768 else 64) * 2.0 ** -24 * want.abs() + 1e-30
    (loss * 3).backward()
    dloss = ((torch.tensor(3.0, device="cuda") / float(T + 2)).expand(T)).contiguous()
    assert torch.equal(x.grad, native().cross_entropy_bwd(dloss, logits, lse, labels, -100, False))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [1, 7, 8, 8191, 8193, 1_000_003, 5_000_008])
def test_squared_norm(n, dtype):
    torch.manual_seed(n)
    x = torch.randn(n, device="cuda").to(dtype)
    out = torch.full((1,), 2.0, device="cuda")
    native().l2norm_sq_(x, out)
    want = x.double().square().sum() + 2
    # an eight's products and additions, a workgroup's sum (its own are 64-bit) and each one's addition to the result
    assert (out.double() - want).abs() <= (9 + min(n // 8192 + 1, 512)) * 2.0 ** -24 * want


@pytest.mark.parametrize("denom", [3, 1e38, 1e39])
def test_any_denominator(denom):
    """The quotient is rounded once, whether or not the denominator is a 32-bit number."""
    logits, labels = torch.randn(64, 41, device="cuda").bfloat16(), torch.zeros(64, dtype=torch.int64, device="cuda")
    want = native().cross_entropy_fwd(logits, labels, -100)[0].double().sum() / denom
    assert abs(float(ops.cross_entropy(logits, labels, reduction_denom=denom)) - float(want)) <= 2.0 ** -24 * float(want)

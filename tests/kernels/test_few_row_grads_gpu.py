"""Products of a few rows whose operands need gradients: the forms without a backward leave them to autograd."""

import pytest
import torch

from llmctl import ops
from llmctl.ops import hybrid as hops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("needs", ["x", "w", "b"])
@pytest.mark.parametrize("M", [4, 40])
@pytest.mark.parametrize("form", ["linear", "linear_f32", "decode_linear"])
def test_gradients_of_few_row_products(form, M, needs):
    g = torch.Generator(device="cuda").manual_seed(M)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    t = dict(x=r(M, 72), w=r(64, 72), b=r(64))  # (a size that no kernel of the older kind takes)
    if needs == "b" and form == "linear_f32":
        pytest.skip("no bias")
    t[needs].requires_grad_()
    y = {"linear": lambda: hops.linear(t["x"], t["w"], t["b"]), "linear_f32": lambda: hops.linear_f32(t["x"], t["w"]),
         "decode_linear": lambda: ops.decode_linear(t["x"], t["w"], t["b"])}[form]()
    dy = r(M, 64)
    y.backward(dy.to(y.dtype))
    # (one rounding of the gradient; of dy too where the result was fp32)
    want = {"x": lambda: dy.float() @ t["w"].float(), "w": lambda: dy.float().t() @ t["x"].float(), "b": lambda: dy.float().sum(0)}[needs]()
    assert (t[needs].grad.float() - want).norm() <= 2.0 ** -7 * want.norm()


def test_gradients_of_latent_values():
    g = torch.Generator(device="cuda").manual_seed(0)
    o, w = (torch.randn(*s, generator=g, device="cuda").bfloat16() for s in ((5, 3, 64), (3, 64, 16)))
    w.requires_grad_()
    y = hops.latent_values(o, w)
    dy = torch.randn(y.shape, generator=g, device="cuda").bfloat16()
    y.backward(dy)
    want = torch.stack([o[:, h].float().t() @ dy[:, h * 16:(h + 1) * 16].float() for h in range(3)])
    assert (w.grad.float() - want).norm() <= 2.0 ** -7 * want.norm()


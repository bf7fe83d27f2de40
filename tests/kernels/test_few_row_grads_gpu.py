"""Products of a few rows and routed experts whose operands need gradients: the forms without a backward leave them to autograd."""

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



@pytest.mark.parametrize("T", [6, 80])
@pytest.mark.parametrize("kind", ["group", "softmax"])
def test_gradients_of_expert_down_weights(kind, T):
    """The grouped expert products have no backward; the layer's general form gives its last projections their gradients."""
    from llmctl.models.moe import BiasedSoftmaxMoE, GroupLimitedMoE

    torch.manual_seed(T)
    W, ff, E = 64, 32, 4
    kw = dict(device="cuda", dtype=torch.bfloat16)
    m = GroupLimitedMoE(W, ff, E, 2, 2, 1, **kw) if kind == "group" else BiasedSoftmaxMoE(W, ff, E, 2, "relu2", shared_ff=ff, **kw)
    down = list(m.experts_down) if kind == "group" else [m.w_down, m.w_sdown]
    for p in m.parameters():
        p.requires_grad_(any(p is d for d in down))
    x, dy = torch.randn(T, W, device="cuda").bfloat16(), torch.randn(T, W, device="cuda")
    m(x).backward(dy)
    with torch.no_grad():
        logits = torch.nn.functional.linear(x.float(), m.w_router)
        topi, topw = hops.group_topk_router(logits, 2, 2, 1) if kind == "group" else hops.bias_topk_router(logits, m.bias, 2, 1, 1, True)
        for e in range(E):
            t, k = (topi == e).nonzero(as_tuple=True)
            if not len(t):
                continue
            u = x[t].float() @ m.experts_up[e].float().t()
            a = torch.nn.functional.silu(u[:, :ff]) * u[:, ff:] if kind == "group" else torch.relu(u).square()
            want = (dy[t] * topw[t, k].float()[:, None]).t() @ a
            got = m.experts_down[e].grad if kind == "group" else m.w_down.grad[:, e * ff:(e + 1) * ff]
            # bf16: the rows that the activation reads, the activation itself, dy and the result, 2^-8 each (the square doubles the first)
            assert (got.float() - want).norm() <= 5 * 2.0 ** -8 * want.norm()
        if kind == "softmax":
            want = dy.t() @ torch.relu(x.float() @ m.w_sup[:ff].float().t()).square()
            assert (m.w_sdown.grad.float() - want).norm() <= 5 * 2.0 ** -8 * want.norm()

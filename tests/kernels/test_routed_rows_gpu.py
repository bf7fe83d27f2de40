"""The kernels that norm a step's few rows and route them (``router_rows.h``): the norm's results are those without a router, and the choice and its
weights are the router's on the same rows.  Router outputs at the edges of the passes of eight and of the 16 lanes, groups, biases, rows on
either side of a thread's quads and rows that only the general forms take."""

import pytest
import torch

from llmctl.ops import hybrid as hops

pytestmark = pytest.mark.gpu


def _same(routed, h, router):
    nat = hops.native_hybrid()
    w, bias, top, groups, keep, softmax, renorm = router
    idx, wgt = routed
    ri, rw = nat.moe_route(h, *router)
    z = h.double() @ w.double().t()
    # fp32 sums of W products in another order: 2^-20 of the terms' size; rows whose choice such a change of the logits could move are left out
    eps = 2.0 ** -20 * (h.double().abs() @ w.double().abs().t())
    pick = lambda z: (hops.bias_topk_router(z.float().contiguous(), bias, top, groups, keep, renorm) if softmax
                      else hops.group_topk_router(z.float().contiguous(), top, groups, keep))[0]
    base, safe = pick(z), torch.ones(h.shape[0], dtype=torch.bool, device="cuda")
    for s in range(4):
        noise = (torch.rand(z.shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(s)).double() - 0.5) * 4 * eps
        safe &= (pick(z + noise) == base).all(1)
    assert len(safe) < 16 or safe.float().mean() > 0.9
    assert torch.equal(idx[safe], ri[safe]) and torch.equal(idx.long()[safe], base[safe])
    assert torch.allclose(wgt[safe], rw[safe], rtol=1e-4, atol=1e-6)


@pytest.mark.parametrize("E,top,groups,keep", [(1, 1, 1, 1), (7, 3, 1, 1), (8, 2, 2, 1), (9, 2, 3, 2), (16, 4, 4, 2), (17, 2, 1, 1), (64, 5, 8, 3), (128, 8, 8, 3)])
@pytest.mark.parametrize("W", [8, 1024, 1032, 2048, 4096, 4104])
@pytest.mark.parametrize("T,kind", [(1, "sigmoid"), (33, "softmax"), (64, "bias")])
def test_routed_rows(E, top, groups, keep, W, T, kind):
    g = torch.Generator(device="cuda").manual_seed(E + W + T)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    bf = torch.bfloat16
    router = (r(E, W) * W ** -0.5, 0.1 * r(E) if kind == "bias" else None, top, groups, keep, kind != "sigmoid", kind == "bias")
    w, b, w2 = r(W), r(W), r(W)
    table, ids = r(50, W).to(bf), torch.arange(T, device="cuda") * 7 % 50
    x, h, routed = hops.embed_layernorm_route(ids, table, 1.5, w, b, 1e-5, router)
    x0, h0 = hops.embed_layernorm_f32(ids, table, 1.5, w, b, 1e-5)
    assert torch.equal(x, x0) and torch.equal(h, h0)
    _same(routed, h, router)
    for pad in (0, 2):  # rows aligned for quads, and not
        a = r(T, W + pad).to(bf)[:, pad:]
        n = T * 2
        s = hops.ExpertSum(r(n, W), torch.randint(0, 3, (T, 2), generator=g, device="cuda").to(torch.int32), r(T, 2).abs(), r(T, W).to(bf), None, None, 3)
        x1, x2 = x.clone(), x.clone()
        h1, routed = hops.add_layernorm_route_(x1, a, s, w, b, 1e-5, bf, router)
        assert torch.equal(h1, hops.add_layernorm_f32_(x2, a, s, w, b, 1e-5, bf)) and torch.equal(x1, x2)
        _same(routed, h1, router)
        x1, x2 = x.clone(), x.clone()
        h1, routed = hops.gated_norm_add_norm_route_(x1, h0, a, w, w2, 1e-5, bf, router)
        assert torch.equal(h1, hops.gated_norm_add_norm_f32_(x2, h0, a, w, w2, 1e-5, bf)) and torch.equal(x1, x2)
        _same(routed, h1, router)

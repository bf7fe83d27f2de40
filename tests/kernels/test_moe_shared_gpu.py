"""A shared expert's products of a few rows in the experts' own launches: the same bits as in launches of their own."""

import pytest
import torch

from llmctl.models.moe import BiasedSoftmaxMoE
from llmctl.ops import hybrid as hops

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("T", [1, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("width, ff, shared_ff, experts, act, opts", [
    (256, 32, 64, 4, "relu2", {}),
    (520, 40, 264, 3, "gelu", {"side": 8}),  # ragged tiles and K steps; more workgroups of the shared expert than an expert's row of the grid
    (512, 512, 1016, 8, "relu2", {"side": 7, "shared_gate": True, "identity": 2}),
    (2048, 1024, 2048, 8, "relu2", {"side": 16}),
])
def test_shared_expert_in_the_experts_launches(T, width, ff, shared_ff, experts, act, opts, monkeypatch):
    torch.manual_seed(T + width)
    m = BiasedSoftmaxMoE(width, ff, experts, 2, act, shared_ff=shared_ff, device="cuda", dtype=torch.bfloat16, **opts).requires_grad_(False)
    if m.b_sup is not None:
        m.b_sup.normal_()
    x = torch.randn(T, width + 8, device="cuda").bfloat16()[:, :width]
    calls = []
    rides = hops.shared_rides
    monkeypatch.setattr(hops, "shared_rides", lambda *a: calls.append(rides(*a)) or calls[-1])
    got = m(x)
    assert calls == [True]
    monkeypatch.setattr(hops, "shared_rides", lambda *a: False)
    want = m(x)
    for a, b in zip(got if m.side else [got], want if m.side else [want]):
        assert torch.equal(a, b)


def test_shared_expert_stays_apart_where_its_form_is_another():
    kw = dict(device="cuda", dtype=torch.bfloat16)
    x = torch.randn(33, 512, **kw)
    w = torch.randn(8192, 512, **kw)
    d = torch.randn(512, 8192, **kw)
    assert not hops.shared_rides(x, w[:1024], None, 1024, d[:, :1024], "relu2")  # more rows than a step
    assert not hops.shared_rides(x[:16], w[:1024], None, 1024, d[:, :1024], "swiglu")
    assert not hops.shared_rides(x[:4], w, None, 8192, d, "relu2")  # two waves a workgroup
    assert not hops.shared_rides(x[:16], w[:1020], None, 1016, d[:, :1016], "relu2")  # rows that are not aligned
    assert hops.shared_rides(x[:16], w[:1024], None, 1024, d[:, :1024], "relu2")

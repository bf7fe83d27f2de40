"""The residual updates that take the routed experts' weighted sum in their own pass, against the sum as a tensor and the plain update (the same
operations in the same order: the same bits): one to five experts a token, experts without weights, a shared expert with and without its gate,
few tokens (fp32 results) and many (bf16), widths on either side of a thread's quads, strided rows, rows that only the general form takes."""

import pytest
import torch

from llmctl.ops import hybrid as hops

pytestmark = pytest.mark.gpu


def _sum(T, W, top, dtype, shared, identity):
    g = torch.Generator(device="cuda").manual_seed(T + W + top)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    E = 6
    idx = torch.stack([torch.randperm(E + identity, generator=g, device="cuda")[:top] for _ in range(T)]).to(torch.int32)
    rows = r(T * top, W).to(dtype)
    rows[idx.reshape(-1) >= E] = float("nan")  # entries that no product writes
    wide = r(T, 2 * W + 8).bfloat16()
    return hops.ExpertSum(rows, idx, r(T, top).abs(), wide[:, 8:8 + W], wide[:, W + 8:] if shared else None,
                          wide[:, 7:8] if shared == "gate" else None, E)


@pytest.mark.parametrize("W", [8, 1024, 1032, 2048, 4096, 4104])
@pytest.mark.parametrize("T,dtype", [(1, torch.float32), (33, torch.float32), (70, torch.bfloat16)])
@pytest.mark.parametrize("top,identity,shared", [(1, 0, None), (2, 0, None), (2, 2, "plain"), (3, 1, "gate"), (5, 3, None)])
def test_sums_in_the_residual_update(W, T, dtype, top, identity, shared):
    s = _sum(T, W, top, dtype, shared, identity)
    g = torch.Generator(device="cuda").manual_seed(W)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, w, b = r(T, W), r(W), r(W)
    bf = torch.bfloat16
    for pad in (0, 2):  # rows aligned for quads, and not
        a = r(T, W + pad).to(bf)[:, pad:]
        x1, x2 = x.clone(), x.clone()
        h1, h2 = hops.add_layernorm_f32_(x1, a, s, w, b, 1e-5, bf), hops.add_layernorm_f32_(x2, a, s.total(), w, b, 1e-5, bf)
        assert torch.equal(x1, x2) and torch.equal(h1, h2) and not h1.isnan().any()
        hops.residual_add_(x1, a, s)
        hops.residual_add_(x2, a, s.total())
        assert torch.equal(x1, x2)
        for nxt in (b, None):
            h1, h2 = hops.gated_norm_add_norm_f32_(x1, s, a, w, nxt, 1e-5, bf), hops.gated_norm_add_norm_f32_(x2, s.total(), a, w, nxt, 1e-5, bf)
            assert torch.equal(x1, x2) and (h1 is h2 is None or torch.equal(h1, h2))

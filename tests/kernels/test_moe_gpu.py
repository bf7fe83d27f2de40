"""Grouped expert kernels (``llmctl/ops/csrc/hybrid/moe.hip``) against the same layer in float64, at the edges of
their tiles: single rows, the last small step (64 tokens) and the first tiled one, partial row and column tiles, K tails,
experts that nobody chose and one that everybody chose, experts without weights, gated shared experts."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(T, W, ff, E, act, seed=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, W, generator=g).bfloat16()
    router = torch.randn(E, W, generator=g) * W ** -0.5
    rows = 2 * ff if act == "swiglu" else ff
    up = (torch.randn(E, rows, W, generator=g) * W ** -0.5).bfloat16()
    down = (torch.randn(W, E * ff, generator=g) * ff ** -0.5).bfloat16()
    return x.cuda(), router.cuda(), up.cuda(), down.cuda()


def _plain(x, idx, w, up, down, act, E):
    x, up, down = x.double(), up.double(), down.double()
    out = torch.zeros_like(x)
    ff = down.shape[-1]
    for e in range(E):
        t, k = (idx == e).nonzero(as_tuple=True)
        u = x[t] @ up[e].t()
        if act == "swiglu":
            u = torch.nn.functional.silu(u[:, :ff]) * u[:, ff:]
        elif act == "relu2":
            u = torch.relu(u).square()
        else:
            u = torch.nn.functional.gelu(u)
        out.index_add_(0, t, (u @ down[e].t()) * w[t, k].double()[:, None])
    t, k = (idx >= E).nonzero(as_tuple=True)
    out.index_add_(0, t, x[t] * w[t, k].double()[:, None])
    return out


@pytest.mark.parametrize("act", ["swiglu", "relu2", "gelu"])
@pytest.mark.parametrize("T,W,ff,E,top", [
    (1, 64, 8, 4, 2), (3, 72, 24, 5, 3), (16, 256, 64, 8, 2), (17, 136, 40, 8, 2), (33, 128, 16, 3, 1), (64, 2048, 96, 8, 2),
    (65, 64, 8, 4, 2), (66, 72, 24, 5, 5), (129, 136, 40, 128, 4), (300, 256, 200, 8, 2), (511, 1024, 512, 4, 2),
    (1024, 192, 136, 2, 1), (2050, 128, 72, 16, 2)])
def test_experts_against_float64(T, W, ff, E, top, act):
    from llmctl.ops import hybrid as hops

    x, router, up, down = _case(T, W, ff, E, act, seed=T)
    d3 = down.view(W, E, ff).transpose(0, 1)
    assert hops.experts_ok(x, up, d3, E)
    nat = hops.native_hybrid()
    idx, w = nat.moe_route(x, router, None, top, 1, 1, True, True)
    got = nat.moe_experts(x, idx, w, [up], [d3], hops._EXPERT_ACTS[act])
    want = _plain(x, idx.long(), w, up, d3, act, E)
    # up to three bf16 roundings (first product, activation, expert result) of relative size 2^-9 each, over sums of ff and of top terms
    assert (got.double() - want).norm() <= 2.0 ** -7 * want.norm()
    again = nat.moe_experts(x, idx, w, [u.contiguous() for u in up.unbind(0)], [u.contiguous() for u in d3.unbind(0)],
                            hops._EXPERT_ACTS[act])
    assert torch.equal(got, again)  # a list of expert weights is the same product, and no atomics: bit for bit


@pytest.mark.parametrize("act", ["swiglu", "relu2", "gelu"])
@pytest.mark.parametrize("W,ff,top", [(256, 256, 1), (384, 640, 1), (1024, 256, 2)])
@pytest.mark.parametrize("counts", [[1, 33, 128, 129, 0, 256, 257], [288, 289, 127, 544, 0, 545, 32], [0, 0, 0, 0, 0, 0, 2305]])
def test_wide_tiles_at_their_edges(counts, W, ff, top, act):
    """Rows that just fill a half tile, a tile, a tile and its ninth block, and one more; widths of the shortest K range and of uneven ones; copies of no expert between."""
    from llmctl.ops import hybrid as hops

    E = len(counts)
    chosen = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)] + [torch.full((40,), E)])
    chosen = chosen[torch.randperm(len(chosen), generator=torch.Generator().manual_seed(W))]
    T = -(-len(chosen) // top)
    idx = torch.full((T * top,), E, dtype=torch.int32)
    idx[:len(chosen)] = chosen.int()
    idx = idx.view(T, top).cuda()
    x, _, up, down = _case(T, W, ff, E, act, seed=sum(counts))
    d3 = down.view(W, E, ff).transpose(0, 1)
    w = torch.rand(T, top, device="cuda")
    want = _plain(x, idx.long(), w, up, d3, act, E)
    for form in (0, 2):  # (which the rule takes, and these tiles)
        got = hops.native_hybrid().moe_experts(x, idx, w, [up], [d3], hops._EXPERT_ACTS[act], None, None, form)
        # as above, row by row: a wrong row would not show in the norm of all
        assert bool(((got.double() - want).norm(dim=1) <= 2.0 ** -7 * want.norm(dim=1) + 1e-12).all())


@pytest.mark.parametrize("T,top,E", [(8192, 2, 8), (8193, 2, 8), (9000, 2, 9), (16385, 1, 3), (11000, 3, 40), (20000, 2, 8)])
@pytest.mark.parametrize("form", [1, 2])
def test_more_copies_than_the_registers_hold(T, top, E, form):
    """The grouping keeps 16384 copies in registers and reads the rest again, and the wide tiles' lanes hold 64 row tiles; unlike shares, an expert that nobody chose and copies of none between."""
    from llmctl.ops import hybrid as hops

    W = ff = 256
    x, _, up, down = _case(T, W, ff, E, "relu2", seed=T)
    d3 = down.view(W, E, ff).transpose(0, 1)
    g = torch.Generator().manual_seed(T)
    share = torch.rand(E + 1, generator=g) + 0.05
    share[E // 2] = 0.0
    idx = torch.multinomial(share.expand(T, -1), top, generator=g).int().cuda()
    w = torch.rand(T, top, generator=g).cuda()
    got = hops.native_hybrid().moe_experts(x, idx, w, [up], [d3], 0, None, None, form)
    want = _plain(x, idx.long(), w, up, d3, "relu2", E)
    # roundings to bf16 (2^-8 at most) of the first product, which the square doubles, of the activation and of the result, whose rows can hang on a few large activations
    assert bool(((got.double() - want).norm(dim=1) <= 2.0 ** -6 * want.norm(dim=1) + 1e-12).all())


def test_tiles_that_pay():
    """The rule of the wide tiles against the times that its figures are from."""
    import re
    from pathlib import Path

    from llmctl.ops import hybrid as hops

    pays = hops.native_hybrid().moe_wide_pays
    picks, taken, best = [], 0.0, 0.0
    for line in (Path(__file__).resolve().parents[2] / "profiles" / "expert_tiles.txt").read_text().splitlines():
        if m := re.match(r"(\d+) (\d+) (\d+) (\d+) (\d+) (\w+) \| ([\d.]+) \| ([\d.]+)$", line):
            T, W, ff, E, top = map(int, m.groups()[:5])
            other, wide = float(m[7]), float(m[8])
            own = wide if pays(T * top, E, W, ff, m[6] == "swiglu") else other
            picks.append(own / min(other, wide))
            taken, best = taken + own, best + min(other, wide)
    assert len(picks) == 1803 and max(picks) < 1.2 and sum(p > 1.05 for p in picks) <= 25 and taken < 1.0025 * best
    assert not any(pays(N, E, W, ff, True) for N, E, W, ff in ((0, 8, 2048, 1024), (383, 8, 2048, 1024), (4096, 8, 2048, 1000), (4096, 8, 2040, 1024), (4096, 8, 128, 1024), (4096, 0, 2048, 1024)))


@pytest.mark.parametrize("T", [5, 64, 65, 700])
def test_one_expert_takes_all_and_experts_without_weights(T):
    from llmctl.ops import hybrid as hops

    W, ff, E = 128, 48, 6  # output 7 is an expert without weights
    x, _, up, down = _case(T, W, ff, E, "swiglu")
    d3 = down.view(W, E, ff).transpose(0, 1)
    nat = hops.native_hybrid()
    idx = torch.tensor([[3, 7]], dtype=torch.int32, device="cuda").repeat(T, 1)
    w = torch.rand(T, 2, device="cuda")
    shared = torch.randn(T, W + 8, device="cuda").bfloat16()
    got = nat.moe_experts(x, idx, w, [up], [d3], 1, shared[:, :W], shared[:, W:W + 1])
    want = _plain(x, idx.long(), w, up, d3, "swiglu", E) + torch.sigmoid(shared[:, W:W + 1].double()) * shared[:, :W].double()
    assert (got.double() - want).norm() <= 2.0 ** -7 * want.norm()


@pytest.mark.parametrize("T,W,E,top,groups,keep", [(1, 64, 8, 2, 1, 1), (7, 72, 8, 2, 4, 2), (130, 256, 128, 8, 8, 3), (1025, 2048, 8, 2, 2, 1),
                                                   (1030, 136, 9, 9, 3, 3)])
@pytest.mark.parametrize("kind", ["sigmoid", "softmax", "softmax+bias"])
def test_route_matches_the_choice_kernels(T, W, E, top, groups, keep, kind):
    """The fused router chooses and weighs as the choice kernels do on the float64 logits (rows whose choice hangs on less
    than the fp32 product's rounding are left out)."""
    from llmctl.ops import hybrid as hops

    x, router, _, _ = _case(T, W, 8, E, "relu2", seed=3)
    bias = torch.randn(E, device="cuda") * 0.1 if kind == "softmax+bias" else None
    idx, w = hops.native_hybrid().moe_route(x, router, bias, top, groups, keep, kind != "sigmoid", True if kind != "sigmoid" else False)
    z = x.double() @ router.double().t()
    pick = (lambda l: hops.group_topk_router(l, top, groups, keep)) if kind == "sigmoid" else (
        lambda l: hops.bias_topk_router(l, bias, top, groups, keep, True))
    ri, rw = pick(z.float().contiguous())
    # a perturbation of the size of the product's rounding (W terms) that leaves the choice alone marks a safe row
    eps = 4e-6 * z.abs().max().float()
    safe = torch.ones(T, dtype=torch.bool, device="cuda")
    for s in range(4):
        noise = (torch.rand(z.shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(s)) - 0.5) * 2 * eps
        safe &= (pick((z.float() + noise).contiguous())[0] == ri).all(1)
    assert safe.float().mean() > 0.9
    assert torch.equal(idx.long()[safe], ri[safe])
    assert torch.allclose(w[safe], rw[safe], rtol=1e-4, atol=1e-6)


@pytest.mark.parametrize("layout", ["off by four bytes", "transposed"])
@pytest.mark.parametrize("T", [6, 80])
@pytest.mark.parametrize("kind", ["group", "softmax"])
def test_routers_in_other_layouts(kind, T, layout):
    """A router that is a slice of a larger buffer, or a transposed matrix: the layer's general form takes it."""
    from llmctl.models.moe import BiasedSoftmaxMoE, GroupLimitedMoE

    torch.manual_seed(0)
    kw = dict(device="cuda", dtype=torch.bfloat16)
    m = GroupLimitedMoE(64, 32, 4, 2, 2, 1, **kw) if kind == "group" else BiasedSoftmaxMoE(64, 32, 4, 2, "relu2", **kw)
    x = torch.randn(T, 64, device="cuda").bfloat16()
    with torch.no_grad():
        want = m(x)
        w = m.w_router.detach()
        buf = torch.zeros(w.numel() + 1, device="cuda")
        other = buf[1:].view_as(w) if layout != "transposed" else torch.empty(64, 4, device="cuda").t()
        other.copy_(w)
        m.w_router.data = other
        assert not m.w_router.is_contiguous() or m.w_router.data_ptr() % 16
        got = m(x)
    assert (got - want).norm() <= 2.0 ** -7 * want.norm()  # the general form rounds every expert's result to bf16


@pytest.mark.parametrize("kind", ["group", "softmax"])
def test_large_experts_with_many_rows_take_library_products(kind, monkeypatch):
    """On either side of the line, with it moved to a size for tests: the same results, and the form that the rule names."""
    from llmctl.models.moe import BiasedSoftmaxMoE, GroupLimitedMoE
    from llmctl.ops import hybrid as hops

    assert hops.experts_pay(1 << 20, 2, 8, 16384, 2048) and hops.experts_pay(4096, 2, 8, 16384, 4096)
    assert not hops.experts_pay(16384, 2, 8, 16384, 4096) and not hops.experts_pay(4096, 2, 8, 28672, 4096) and hops.experts_pay(4095, 2, 8, 28672, 4096)
    torch.manual_seed(0)
    kw = dict(device="cuda", dtype=torch.bfloat16)
    m = GroupLimitedMoE(64, 32, 4, 2, 2, 1, **kw) if kind == "group" else BiasedSoftmaxMoE(64, 32, 4, 2, "relu2", **kw)
    x = torch.randn(80, 64, device="cuda").bfloat16()
    grouped, calls = hops.routed_experts, []
    monkeypatch.setattr(hops, "routed_experts", lambda *a: calls.append(1) or grouped(*a))
    with torch.no_grad():
        want = m(x)
        assert calls and m.on_device(80)
        monkeypatch.setattr(hops, "experts_pay", lambda *a: False)
        got = m(x)
        assert len(calls) == 1 and (kind == "softmax" or not m.on_device(80))
    assert (got - want).norm() <= 2.0 ** -7 * want.norm()

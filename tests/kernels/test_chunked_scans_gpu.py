"""The chunked recurrences on the fp32 matrix cores (``llmctl/ops/csrc/hybrid/mlstm_chunk.hip``, ``gla_chunk.hip``) against the
token-by-token formulas in float64: chunk edges, one-token and empty portions beside long ones, carried and fresh states, key and value
sizes that fill no tile, strided rows, weak and strong gates (decays from nearly one to nearly nothing within a chunk)."""

import pytest
import torch

from llmctl.ops import hybrid as hops

pytestmark = pytest.mark.gpu
LENS = [[41], [256], [300, 1, 0, 63, 64, 65], [17, 513, 128]]


def _cu(lens):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return cu


def _rows(T, H, dk, dv, dtype, g):
    z = torch.randn(T, 2 * H * dk + H * dv + 8, generator=g).to(dtype)  # q | k | v | other columns
    q, k = z[:, :H * dk].unflatten(1, (H, dk)), z[:, H * dk:2 * H * dk].unflatten(1, (H, dk))
    return z, q, k, z[:, 2 * H * dk:2 * H * dk + H * dv].unflatten(1, (H, dv))


def _check(got, want, terms):
    """``terms``: the magnitude of what each result sums up; fp32 sums and exponentials of pairwise exact differences, relative 2^-17."""
    assert ((got.double().cpu() - want).abs() <= 2.0 ** -17 * terms + 1e-7).all(), ((got.double().cpu() - want).abs() / (terms + 1e-7)).max()


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("H,dk,dv,dtype,gain", [(2, 8, 8, torch.float32, 1.0), (3, 64, 128, torch.bfloat16, 1.0), (2, 24, 40, torch.bfloat16, 20.0),
                                                (1, 128, 72, torch.float32, 20.0), (2, 100, 136, torch.bfloat16, 4.0), (2, 33, 16, torch.float32, 1.0)])
def test_mlstm_chunks(H, dk, dv, dtype, gain, lens):
    g = torch.Generator().manual_seed(dk + dv)
    cu, T, ns = _cu(lens), sum(lens), len(lens)
    z, q, k, v = _rows(T, H, dk, dv, dtype, g)
    raw, b_i, b_f = torch.randn(T, 2 * H, generator=g) * gain, torch.randn(H, generator=g), torch.randn(H, generator=g) + 2
    cap, qs = 15.0, dk ** -0.5
    slots = torch.randperm(ns + 2, generator=g)[:ns].int()
    start = torch.tensor([0 if i % 2 else 9 for i in range(ns)], dtype=torch.int32)
    S, n, m = (torch.randn(s, generator=g) for s in ((ns + 2, H, dk, dv), (ns + 2, H, dk), (ns + 2, H)))
    Sd, nd, md, zd = S.cuda(), n.cuda(), m.cuda(), z.cuda()
    d = lambda t, a, w: zd[:, a:a + H * w].unflatten(1, (H, w))
    got = hops.mlstm_scan(d(z, 0, dk), d(z, H * dk, dk), d(z, 2 * H * dk, dv), raw.cuda(), b_i.cuda(), b_f.cuda(), cap, qs, Sd, nd, md,
                          slots.cuda(), torch.tensor(cu, dtype=torch.int32).cuda(), start.cuda(), cu_host=cu)
    i = cap * torch.tanh((raw[:, :H].double() + b_i) / cap)
    f = torch.nn.functional.logsigmoid(cap * torch.tanh((raw[:, H:].double() + b_f) / cap))
    for s in range(ns):
        sl, fresh = int(slots[s]), int(start[s]) == 0
        if lens[s] == 0:
            assert torch.equal(Sd[sl].cpu(), S[sl]) and torch.equal(md[sl].cpu(), m[sl])
            continue
        C, N, M = (torch.zeros_like(t[sl]).double() if fresh else t[sl].double() for t in (S, n, m))
        Ca, Na = C.abs(), N.abs()  # the magnitudes behind them
        for t in range(cu[s], cu[s + 1]):
            Mn = torch.maximum(f[t] + M, i[t])
            a, b = torch.exp(f[t] + M - Mn), torch.exp(i[t] - Mn)
            kt, vt, qt = k[t].double(), v[t].double(), q[t].double() * qs
            C, N = a[:, None, None] * C + b[:, None, None] * kt[:, :, None] * vt[:, None, :], a[:, None] * N + b[:, None] * kt
            Ca = a[:, None, None] * Ca + b[:, None, None] * kt[:, :, None].abs() * vt[:, None, :].abs()
            Na = a[:, None] * Na + b[:, None] * kt.abs()
            M = Mn
            den = torch.maximum((N * qt).sum(-1).abs(), torch.exp(-M)) + 1e-6
            num, numa = torch.einsum("hkv,hk->hv", C, qt), torch.einsum("hkv,hk->hv", Ca, qt.abs())
            want = num / den[:, None]
            _check(got[t], want, numa / den[:, None] + want.abs() * ((Na * qt.abs()).sum(-1) / den)[:, None])
        _check(Sd[sl], C, Ca), _check(nd[sl], N, Na), _check(md[sl], M, M.abs() + 1)


@pytest.mark.parametrize("lens", LENS[1:])
@pytest.mark.parametrize("H,dk,dv,dtype,gain", [(2, 8, 8, torch.float32, 1.0), (3, 64, 128, torch.bfloat16, 1.0), (2, 24, 40, torch.bfloat16, 100.0),
                                                (1, 128, 72, torch.float32, 3000.0), (2, 100, 136, torch.bfloat16, 10.0), (2, 33, 16, torch.float32, 1.0),
                                                (1, 136, 16, torch.float32, 1.0)])
def test_gla_chunks(H, dk, dv, dtype, gain, lens):
    g = torch.Generator().manual_seed(dk + dv)
    cu, T, ns = _cu(lens), sum(lens), len(lens)
    z, q, k, v = _rows(T, H, dk, dv, dtype, g)
    zl, zb, tau, qs = torch.randn(T, H * dk, generator=g) * gain, torch.randn(H * dk, generator=g), 16.0, dk ** -0.5
    slots = torch.randperm(ns + 2, generator=g)[:ns].int()
    start = torch.tensor([0 if i % 2 else 9 for i in range(ns)], dtype=torch.int32)
    S = torch.randn(ns + 2, H, dk, dv, generator=g)
    Sd, zd = S.cuda(), z.cuda()
    d = lambda a, w: zd[:, a:a + H * w].unflatten(1, (H, w))
    got = hops.gla_scan(d(0, dk), d(H * dk, dk), d(2 * H * dk, dv), zl.cuda(), zb.cuda(), tau, qs, Sd, slots.cuda(),
                        torch.tensor(cu, dtype=torch.int32).cuda(), start.cuda(), cu_host=cu)
    la = (torch.nn.functional.logsigmoid((zl + zb).double()) / tau).view(T, H, dk)
    for s in range(ns):
        sl = int(slots[s])
        if lens[s] == 0:
            assert torch.equal(Sd[sl].cpu(), S[sl])
            continue
        C = torch.zeros_like(S[sl]).double() if int(start[s]) == 0 else S[sl].double()
        Ca = C.abs()
        for t in range(cu[s], cu[s + 1]):
            a, kt, vt, qt = torch.exp(la[t]), k[t].double(), v[t].double(), q[t].double() * qs
            C = a[:, :, None] * C + kt[:, :, None] * vt[:, None, :]
            Ca = a[:, :, None] * Ca + kt[:, :, None].abs() * vt[:, None, :].abs()
            _check(got[t], torch.einsum("hkv,hk->hv", C, qt), torch.einsum("hkv,hk->hv", Ca, qt.abs()))
        _check(Sd[sl], C, Ca)


def test_the_layers_of_a_step_share_one_plan(monkeypatch):
    from llmctl.serve.engine import InferenceEngine
    from llmctl.serve.scheduler import PrefillChunk

    e = InferenceEngine("lenitar-w128-l8", device="cuda", max_batch_size=2, num_kv_blocks=32, block_size=16, max_model_len=256, prefix_caching=False)
    assert sum(type(m).__name__ == "MLSTM" for m in e.model.modules()) >= 2
    calls, plan = [], hops.mlstm_chunk_plan
    monkeypatch.setattr(hops, "mlstm_chunk_plan", lambda *a: calls.append(1) or plan(*a))
    for _ in range(2):
        s = e.open_sequence(list(range(1, 90)))
        e.prefill([PrefillChunk(s, 0, 89)])
    assert len(calls) == 2  # one a step
    e.close()


@pytest.mark.parametrize("slab", [False, True])
@pytest.mark.parametrize("ns,H,dk,dv", [(300, 16, 64, 256), (128, 16, 32, 200), (64, 8, 16, 64)])
def test_mlstm_decode_rows_of_many_sequences(ns, H, dk, dv, slab):
    """One token each: every value tile of a head starts from the carried normaliser and log-scale, however late it begins."""
    from llmctl.ops._lib import native_hybrid

    g = torch.Generator(device="cuda").manual_seed(ns)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    q, k, v = r(ns, H, dk), r(ns, H, dk), r(ns, H, dv)
    z = torch.cat([t.reshape(ns, -1) for t in (q, k, v)], 1).contiguous()  # rows of one projection
    q, k, v = (z[:, a:a + H * w].unflatten(1, (H, w)) for a, w in ((0, dk), (H * dk, dk), (2 * H * dk, dv)))
    raw, b_i, b_f, cap, qs = r(ns, 2 * H), r(H), r(H) + 2, 15.0, dk ** -0.5
    S, n, m = r(ns, H, dk, dv), r(ns, H, dk), r(ns, H)
    slots = torch.randperm(ns, generator=torch.Generator().manual_seed(1)).int().cuda()
    i32 = lambda n: torch.arange(n, dtype=torch.int32, device="cuda")
    for _ in range(4):
        i = cap * torch.tanh((raw[:, :H].double() + b_i) / cap)
        f = torch.nn.functional.logsigmoid(cap * torch.tanh((raw[:, H:].double() + b_f) / cap))
        S0, n0, m0 = S[slots.long()].double(), n[slots.long()].double(), m[slots.long()].double()
        m1 = torch.maximum(f + m0, i)
        a, b = torch.exp(f + m0 - m1), torch.exp(i - m1)
        S1 = a[..., None, None] * S0 + b[..., None, None] * k.double()[..., None] * v.double()[:, :, None]
        n1 = a[..., None] * n0 + b[..., None] * k.double()
        den = torch.maximum((n1 * q.double() * qs).sum(-1).abs(), torch.exp(-m1)) + 1e-6
        num = (S1 * q.double()[..., None] * qs).sum(2)
        got = native_hybrid().mlstm_scan(q, k, v, raw, b_i, b_f, cap, qs, S, n, m, slots, i32(ns + 1), torch.ones_like(slots), slab)
        # the quotient's parts are fp32 sums of dk products: 2^-17 of their terms' size each
        size = (S1.abs() * q.double().abs()[..., None] * qs).sum(2) / den[..., None]
        rel = (n1.abs() * q.double().abs() * qs).sum(-1) / den
        assert ((got.double() - num / den[..., None]).abs() <= 2.0 ** -16 * (size + rel[..., None] * (num / den[..., None]).abs()) + 1e-6).all()
        for pool, want in ((S, S1), (n, n1), (m, m1)):
            assert (pool[slots.long()].double() - want).norm() <= 2.0 ** -18 * want.norm()


@pytest.mark.parametrize("lens,chunks", [([255], True), ([64], True), ([40], "mlstm"), ([63], "mlstm"), ([100] + [1] * 16, True), ([64] + [1] * 64, False), ([40] * 64, False), ([1] * 8, False),
                                         ([256] + [1] * 64, True)])
@pytest.mark.parametrize("op", ["mlstm", "gla"])
def test_short_portions_of_many_sequences_are_scanned(op, lens, chunks):
    """Which form a step takes, and that both agree there (the same recurrence, in chunks or token by token)."""
    from llmctl.ops._lib import native_hybrid

    H, dk, dv, nat = 16, 64, 128, native_hybrid()
    plan = (hops.mlstm_chunk_plan if op == "mlstm" else hops.gla_plan)(_cu(lens), torch.device("cuda"), H, dk, dv)
    assert (plan is not None) == (chunks is True or chunks == op)
    g = torch.Generator().manual_seed(len(lens))
    T, ns = sum(lens), len(lens)
    z, q, k, v = _rows(T, H, dk, dv, torch.bfloat16, g)
    zd = z.cuda()
    q, k, v = (zd[:, a:a + H * w].unflatten(1, (H, w)) for a, w in ((0, dk), (H * dk, dk), (2 * H * dk, dv)))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32).cuda()
    slots, start, cu = i32(list(range(ns))), i32([5] * ns), i32(_cu(lens))
    S, n, m = (torch.randn(s, generator=g).cuda() for s in ((ns, H, dk, dv), (ns, H, dk), (ns, H)))
    S2, n2, m2 = S.clone(), n.clone(), m.clone()
    if op == "mlstm":
        raw, b_i, b_f = torch.randn(T, 2 * H, generator=g).cuda(), torch.zeros(H).cuda(), torch.full((H,), 2.0).cuda()
        got = hops.mlstm_scan(q, k, v, raw, b_i, b_f, 15.0, dk ** -0.5, S, n, m, slots, cu, start, cu_host=_cu(lens))
        want = nat.mlstm_scan(q, k, v, raw, b_i, b_f, 15.0, dk ** -0.5, S2, n2, m2, slots, cu, start, False)
    else:
        zl, zb = torch.randn(T, H * dk, generator=g).cuda(), torch.zeros(H * dk).cuda()
        got = hops.gla_scan(q, k, v, zl, zb, 16.0, dk ** -0.5, S, slots, cu, start, cu_host=_cu(lens))
        want = nat.gla_scan(q, k, v, zl, zb, 16.0, dk ** -0.5, S2, slots, cu, start, None, True, True)
    for a, b in ((got, want), (S, S2)):  # fp32 sums of some hundred terms in another order (the mLSTM's quotient may cancel)
        assert (a - b).norm() <= 1e-4 * b.norm()

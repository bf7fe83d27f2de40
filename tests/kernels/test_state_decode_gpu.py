"""One token per sequence through a matrix memory with its gates and head norm in one launch: against float64, over key and value sizes at the edges of the lanes'
split, views with odd strides, fresh and carried memories, and ranks and widths that fill no whole round of loads."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0**-24


def _rows(g, T, H, d, pad):
    return torch.randn(T, H * d + pad, generator=g, device="cuda").bfloat16()[:, :H * d].unflatten(1, (H, d))


class _Batch:
    def __init__(self, T, slots, g):
        self.Tp = 0
        self.state = torch.randperm(slots, generator=g, device="cuda")[:T].int()
        self.start = torch.arange(T, device="cuda", dtype=torch.int32) % 3 * 5  # every third begins


def _finish(o, err, w, g, eps, silu):
    """(the result, a bound of what errors ``err`` of o and the rounding of the rest make of it), rows [T, H, dv]"""
    rms = (o.pow(2).mean(2, keepdim=True) + eps).sqrt()
    f = w * torch.sigmoid(g) * (g if silu else 1.0)
    # the mean's relative error is at most twice o's over its root mean square; four roundings, an exponential of 2 ulp; then bf16
    y, spread = o / rms * f, err / rms + o.abs() / rms * (err.pow(2).mean(2, keepdim=True).sqrt() / rms)
    return y, 2.0**-8 * y.abs() + 2.0 * spread * f.abs() + 32 * EPS * y.abs() + 1e-30


SIZES = [(1, 1, 1, 4, 1), (3, 2, 16, 64, 4), (5, 3, 17, 68, 7), (16, 4, 64, 128, 16), (33, 2, 65, 60, 24), (2, 1, 128, 124, 8), (4, 2, 200, 128, 64), (2, 2, 256, 8, 3)]


@pytest.mark.parametrize("T,H,dk,dv,rank", SIZES)
def test_gla_decode(T, H, dk, dv, rank):
    from llmctl.ops import hybrid as hops

    g = torch.Generator(device="cuda").manual_seed(T * dk + dv)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    q, k, v = _rows(g, T, H, dk, 3), _rows(g, T, H, dk, 1), _rows(g, T, H, dv, 5)
    a, w, bias = rand(T, rank + 1).bfloat16()[:, :rank], (rand(H * dk, rank) * rank**-0.5).bfloat16(), rand(H * dk)
    gate, norm, S = rand(T, H * dv + 7).bfloat16()[:, :H * dv], rand(H * dv), rand(T + 2, H, dk, dv)
    b, tau, scale = _Batch(T, T + 2, g), 16.0, dk**-0.5
    assert hops.state_decode_ok(v.flatten(1), S, b, dv)
    D, old = torch.Tensor.double, S.clone()
    z = D(a) @ D(w).t() + D(bias)
    f = (torch.nn.functional.logsigmoid(z) / tau).exp().unflatten(1, (H, dk))[..., None]
    s0 = D(S)[b.state.long()] * (b.start != 0)[:, None, None, None]
    kv = D(k)[..., None] * D(v)[:, :, None]
    want = f * s0 + kv
    # the logit's sums and the functions after it move the decay by this much of itself
    df = (rank + 4) * EPS * ((D(a).abs() @ D(w).abs().t() + D(bias).abs()) / tau).unflatten(1, (H, dk))[..., None] + 8 * EPS
    err = (f * s0).abs() * df + 2 * EPS * ((f * s0).abs() + kv.abs())
    qd = (D(q) * scale)[..., None]
    o, eo = (want * qd).sum(2), ((err + (dk + 2) * EPS * want.abs()) * qd.abs()).sum(2)
    y, tol = _finish(o, eo, D(norm).view(H, dv), D(gate).unflatten(1, (H, dv)), 1e-5, True)
    got = hops.gla_decode(q, k, v, a, w, bias, tau, scale, S, b, norm, gate, 1e-5)
    assert got.dtype == torch.bfloat16 and bool(((D(got).unflatten(1, (H, dv)) - y).abs() <= tol).all())
    idx = b.state.long()
    assert bool(((D(S)[idx] - want).abs() <= err).all())
    rest = torch.ones(T + 2, dtype=torch.bool, device="cuda")
    rest[idx] = False
    assert torch.equal(S[rest], old[rest])


@pytest.mark.parametrize("T,H,dk,dv,rank", SIZES)
@pytest.mark.parametrize("few", [True, False])
def test_mlstm_decode(T, H, dk, dv, rank, few):
    from llmctl.ops import hybrid as hops

    g = torch.Generator(device="cuda").manual_seed(T * dk + dv)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    W = 4 * rank if few else 4 * rank + 1  # (rows in no quads: the product of their own)
    q, k, v, h = _rows(g, T, H, dk, 3), _rows(g, T, H, dk, 1), _rows(g, T, H, dv, 5), rand(T, W).bfloat16()
    w_if, b_i, b_f = rand(2 * H, W) * W**-0.5, rand(H), rand(H) + 2.0
    gate, norm, S, n, m = rand(T, H * dv + 7).bfloat16()[:, :H * dv], rand(H * dv), rand(T + 2, H, dk, dv), rand(T + 2, H, dk), rand(T + 2, H)
    b, cap, scale = _Batch(T, T + 2, g), 15.0, dk**-0.5
    D, idx = torch.Tensor.double, b.state.long()
    z, dz = D(h) @ D(w_if).t(), (W + 8) * EPS * (D(h).abs() @ D(w_if).abs().t() + 4.0)
    zi, zf = z[:, :H] + D(b_i), z[:, H:] + D(b_f)
    on = (b.start != 0)[:, None]
    i, f = cap * torch.tanh(zi / cap), torch.nn.functional.logsigmoid(cap * torch.tanh(zf / cap))
    m0 = D(m)[idx] * on
    mn = torch.maximum(f + m0, i)
    da, db = (f + m0 - mn).exp(), (i - mn).exp()
    # both exponents' errors: the logits' and the roundings of numbers of up to 15 + |m|
    de = dz[:, :H] + dz[:, H:] + 16 * EPS * (cap + m0.abs() + 1.0)
    s0, n0 = D(S)[idx] * on[..., None, None], D(n)[idx] * on[..., None]
    kv = D(k)[..., None] * D(v)[:, :, None]
    e4, x = lambda t: t[..., None, None], lambda t: t[..., None]
    want, nw = e4(da) * s0 + e4(db) * kv, x(da) * n0 + x(db) * D(k)
    es = (2 * e4(de) + 4 * EPS) * ((e4(da) * s0).abs() + (e4(db) * kv).abs())
    en = (2 * x(de) + 4 * EPS) * ((x(da) * n0).abs() + (x(db) * D(k)).abs())
    qd = D(q) * scale
    num, enum = (want * qd[..., None]).sum(2), ((es + (dk + 2) * EPS * want.abs()) * qd.abs()[..., None]).sum(2)
    nq, enq = (nw * qd).sum(2), ((en + (dk + 2) * EPS * nw.abs()) * qd.abs()).sum(2)
    den = torch.maximum(nq.abs(), (-mn).exp()) + 1e-6
    eden = torch.maximum(enq, (-mn).exp() * 2 * de) + 2 * EPS * den
    o = num / x(den)
    eo = (enum + o.abs() * x(eden)) / x(den) * 1.1 + 2 * EPS * o.abs()
    y, tol = _finish(o, eo, D(norm).view(H, dv), D(gate).unflatten(1, (H, dv)), 1e-5, False)
    got = hops.mlstm_decode(q, k, v, h, w_if, b_i, b_f, cap, scale, S, n, m, b, norm, gate, 1e-5)
    assert got.dtype == torch.bfloat16 and bool(((D(got).unflatten(1, (H, dv)) - y).abs() <= tol).all())
    assert bool(((D(S)[idx] - want).abs() <= es).all()) and bool(((D(n)[idx] - nw).abs() <= en).all())
    assert bool(((D(m)[idx] - mn).abs() <= 2 * de).all())

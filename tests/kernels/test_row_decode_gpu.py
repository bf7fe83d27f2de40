"""Decode rows over a paged row cache (``llmctl/ops/csrc/hybrid/row_decode.hip``) against the plain formula in float64, at the
edges of the kernel: one key, the last key of a 64-key step and the first of the next, windows and chunks that begin inside a step,
kept first keys, more than 16 heads and counts that do not fill a tile, key and value widths that are no multiple of 32 or
that need more than one value tile, several kv groups, every option, and contexts that split over workgroups or do not."""

import pytest
import torch

from llmctl.ops import hybrid as hops

pytestmark = pytest.mark.gpu
NO = hops.NO_LIMIT


def _case(H, R, rk, groups, koff, rs, ctxs, bs, seed):
    g = torch.Generator().manual_seed(seed)
    maxb = max((c + bs - 1) // bs for c in ctxs)
    nb = maxb * len(ctxs) + 1
    cache = torch.randn(nb, bs, groups * rs, generator=g).bfloat16()
    bt = torch.randperm(nb, generator=g)[: maxb * len(ctxs)].view(len(ctxs), maxb).int()
    qa = torch.randn(len(ctxs), H, R, generator=g).bfloat16()
    return qa, cache, bt, torch.tensor(ctxs, dtype=torch.int32)


def _plain(qa, cache, bt, ctx, window, sink, scale, rk, groups, koff, chunk, hscale, ofreq, sig_bias, dist_a, dist_b, softcap, keep):
    ns, H, R = qa.shape
    rs = cache.shape[2] // groups
    out = torch.empty(ns, H, rk, dtype=torch.float64)
    for n in range(ns):
        c = int(ctx[n])
        rows = cache[bt[n].long()].reshape(-1, groups, rs)[:c].double()
        j, pos = torch.arange(c), c - 1
        c0 = (pos // chunk) * chunk
        seen = (j >= c0) & ((pos - j < window) | (j < keep))
        for h in range(H):
            k, v = rows[:, h // (H // groups), koff:koff + R], rows[:, h // (H // groups), :rk]
            s = k @ qa[n, h].double() * scale * (hscale[h].double() if hscale is not None else 1.0)
            if softcap:
                s = softcap * torch.tanh(s / softcap)
            if sig_bias is not None:
                if dist_a is not None:
                    s = s - dist_a[h].double() * torch.log1p(dist_b[h].double() * (pos - j).double())
                w = torch.sigmoid(s + sig_bias[h].double()) * seen
            else:
                s = s.masked_fill(~seen, float("-inf"))
                top = s.max() if sink is None else torch.maximum(s.max(), sink[h].double())
                e = torch.exp(s - top)
                w = e / (e.sum() + (0 if sink is None else torch.exp(sink[h].double() - top)))
            o = w @ v
            if ofreq is not None:
                a = pos * ofreq.double()
                u, t = o[0::2].clone(), o[1::2].clone()
                o[0::2], o[1::2] = u * a.cos() + t * a.sin(), t * a.cos() - u * a.sin()
            out[n, h] = o
    return out


EDGES = [1, 2, 63, 64, 65, 127, 128, 129, 200]


@pytest.mark.parametrize("H,R,rk,groups,koff,rs,bs", [
    (4, 64, 64, 1, 0, 64, 16), (16, 576, 512, 1, 0, 576, 64), (17, 40, 24, 1, 0, 40, 8), (40, 136, 64, 1, 72, 208, 16),
    (6, 200, 136, 3, 136, 336, 12), (8, 256, 256, 2, 256, 512, 16), (3, 640, 600, 1, 0, 640, 16), (2, 8, 8, 1, 8, 16, 1),
    (32, 128, 128, 4, 128, 256, 32), (5, 264, 520, 1, 520, 784, 16)])
@pytest.mark.parametrize("form", ["plain", "sink", "window", "chunk", "keep", "scale", "cap", "turn", "sigmoid"])
def test_decode_rows_against_float64(H, R, rk, groups, koff, rs, bs, form):
    if form in ("cap", "turn", "sigmoid") and R > 256:
        pytest.skip("keys this wide take these options in the generic kernel")
    g = torch.Generator().manual_seed(H * R + rk)
    ctxs = EDGES if H * rk <= 2048 else EDGES[:6]
    qa, cache, bt, ctx = _case(H, R, rk, groups, koff, rs, ctxs, bs, seed=R)
    window, chunk, keep, cap, sink, hscale, ofreq, sb, da, db = NO, NO, 0, 0.0, None, None, None, None, None, None
    if form == "sink":
        sink, window = torch.randn(H, generator=g), 70
    elif form == "window":
        window = 66
    elif form == "chunk":
        chunk, window = 96, 80
    elif form == "keep":
        keep, window, chunk = 5, 33, 100
    elif form == "scale":
        hscale = torch.rand(H, generator=g) + 0.5
    elif form == "cap":
        cap = 2.0
    elif form == "turn":
        ofreq = torch.rand(rk // 2, generator=g) * 0.1
        sink = torch.randn(H, generator=g)
    elif form == "sigmoid":
        sb, da, db = -torch.rand(H, generator=g) * 4, torch.rand(H, generator=g), torch.rand(H, generator=g)
        window = 100
    scale = R ** -0.5
    want = _plain(qa, cache, bt, ctx, window, sink, scale, rk, groups, koff, chunk, hscale, ofreq, sb, da, db, cap, keep)
    dev = lambda t: None if t is None else t.cuda()
    args = [dev(t) for t in (qa, cache, bt, ctx)]
    for max_ctx in (0, max(ctxs)):  # sizes the split of the keys
        got = hops.latent_attention_decode(*args, window, dev(sink), scale, rk, True, groups, koff, chunk, dev(hscale), dev(ofreq),
                                           max_ctx, dev(sb), dev(da), dev(db), cap, keep).double().cpu()
        # weights (the second product's operand) and results round to bf16, 2^-9 each: sum_j w_j |v_j| over the values' norm is at
        # most 4 here (|v| < 4 everywhere but in rare tails), and weights sum to 1 (sigmoids: to the number of keys)
        size = want.abs().amax(-1, keepdim=True).clamp(min=1.0)
        assert ((got - want).abs() <= 2.0 ** -7 * size).all(), (form, max_ctx, ((got - want).abs() / size).amax((1, 2)))


def test_empty_splits_and_long_context():
    # one short and one long sequence in one launch: most splits of the short one see no key
    qa, cache, bt, ctx = _case(8, 128, 128, 1, 0, 128, [3, 5000], 16, seed=1)
    want = _plain(qa, cache, bt, ctx, NO, None, 0.09, 128, 1, 0, NO, None, None, None, None, None, 0.0, 0)
    got = hops.latent_attention_decode(qa.cuda(), cache.cuda(), bt.cuda(), ctx.cuda(), NO, None, 0.09, 128, max_ctx=5000).double().cpu()
    assert ((got - want).abs() <= 2.0 ** -7 * want.abs().amax(-1, keepdim=True).clamp(min=1.0)).all()


def _plain_rows(qa, cache, bt, ctx, window, sink, scale, rk, groups, koff, chunk, hscale, ofreq, sig_bias, dist_a, dist_b, softcap, keep):
    """``_plain`` with a row's heads at once, float64 on the operands' device."""
    ns, H, R = qa.shape
    P, rs = H // groups, cache.shape[2] // groups
    out = torch.empty(ns, H, rk, dtype=torch.float64, device=qa.device)
    up = lambda t: None if t is None else t.double()[:, None]
    sink, hscale, sig_bias, dist_a, dist_b = map(up, (sink, hscale, sig_bias, dist_a, dist_b))
    for n in range(ns):
        c = int(ctx[n])
        rows = cache[bt[n, :(c + cache.shape[1] - 1) // cache.shape[1]].long()].reshape(-1, groups, rs)[:c].double()
        j, pos = torch.arange(c, device=qa.device), c - 1
        seen = (j >= (pos // chunk) * chunk) & ((pos - j < window) | (j < keep))
        k, v = rows[:, :, koff:koff + R].permute(1, 2, 0).contiguous(), rows[:, :, :rk].transpose(0, 1).contiguous()
        s = torch.bmm(qa[n].double().view(groups, P, R), k).view(H, c) * scale * (1.0 if hscale is None else hscale)
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        if sig_bias is not None:
            w = torch.sigmoid(s - dist_a * torch.log1p(dist_b * (pos - j).double()) + sig_bias) * seen
        else:
            s = s.masked_fill(~seen, float("-inf"))
            top = s.amax(1, keepdim=True) if sink is None else torch.maximum(s.amax(1, keepdim=True), sink)
            e = torch.exp(s - top)
            w = e / (e.sum(1, keepdim=True) + (0 if sink is None else torch.exp(sink - top)))
        o = torch.bmm(w.view(groups, P, c), v).view(H, rk)
        if ofreq is not None:
            a = pos * ofreq.double()
            u, t = o[:, 0::2].clone(), o[:, 1::2].clone()
            o[:, 0::2], o[:, 1::2] = u * a.cos() + t * a.sin(), t * a.cos() - u * a.sin()
        out[n] = o
    return out


@pytest.mark.parametrize("H,R,rk,groups,koff,rs,bs,ns", [
    (128, 64, 64, 1, 0, 64, 16, 260), (72, 136, 64, 2, 72, 208, 16, 290), (130, 40, 24, 1, 0, 40, 8, 200), (96, 320, 256, 1, 0, 320, 16, 70),
    (128, 576, 512, 1, 0, 576, 64, 40), (40, 640, 600, 1, 0, 640, 12, 90)])
@pytest.mark.parametrize("form", ["plain", "sink", "window", "keep", "scale", "cap", "turn", "sigmoid"])
def test_many_heads_of_a_group(H, R, rk, groups, koff, rs, bs, ns, form):
    """Many heads over the same keys in many rows, at contexts around the edges of a tile and over splits, some of them empty: sizes that run in
    tiles of up to 128 heads (``decode_tiles_pay``), and the same rows few at a time, which do not."""
    if form in ("cap", "turn", "sigmoid") and R > 256:
        pytest.skip("keys this wide take these options in the generic kernel")
    g = torch.Generator().manual_seed(H * R + rk)
    qa, cache, bt, ctx = (t.cuda() for t in _case(H, R, rk, groups, koff, rs, [EDGES[i % len(EDGES)] + 64 * (i // 64) for i in range(ns)], bs, seed=R))
    bt = torch.nn.functional.pad(bt, (0, 8192 // bs))  # room for longer contexts
    opt = dict(window=NO, sink=None, chunk=NO, hscale=None, ofreq=None, sig_bias=None, dist_a=None, dist_b=None, softcap=0.0, keep=0)
    rnd = lambda n: torch.rand(n, generator=g).cuda()
    if form in ("sink", "turn"):
        opt["sink"] = torch.randn(H, generator=g).cuda()
    if form == "window":
        opt.update(window=130, chunk=192)
    elif form == "keep":
        opt.update(window=100, keep=70)
    elif form == "scale":
        opt["hscale"] = rnd(H) + 0.5
    elif form == "cap":
        opt["softcap"] = 2.0
    elif form == "turn":
        opt["ofreq"] = rnd(rk // 2) * 0.1
    elif form == "sigmoid":
        opt.update(sig_bias=-4 * rnd(H), dist_a=rnd(H), dist_b=rnd(H))
    o, scale = opt, R ** -0.5
    want = _plain_rows(qa, cache, bt, ctx, o["window"], o["sink"], scale, rk, groups, koff, o["chunk"], o["hscale"], o["ofreq"], o["sig_bias"], o["dist_a"],
                       o["dist_b"], o["softcap"], o["keep"])
    run = lambda q, t, c, m: hops.latent_attention_decode(q, cache, t, c, o["window"], o["sink"], scale, rk, True, groups, koff, o["chunk"], o["hscale"], o["ofreq"], m,
                                                          o["sig_bias"], o["dist_a"], o["dist_b"], o["softcap"], o["keep"]).double()
    size = want.abs().amax(-1, keepdim=True).clamp(min=1.0)  # (the bound: see above)
    for got in (run(qa, bt, ctx, 0), run(qa, bt, ctx, int(ctx.max())), torch.cat([run(qa[i:i + 3], bt[i:i + 3], ctx[i:i + 3], int(ctx.max())) for i in range(0, ns, 3)])):
        assert ((got - want).abs() <= 2.0 ** -7 * size).all(), ((got - want).abs() / size).amax((1, 2))

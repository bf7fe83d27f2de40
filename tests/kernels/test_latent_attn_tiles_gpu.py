"""Prompt attention over row caches on the matrix cores (``latent_attn_mfma``) against the plain form: key widths around the 12- and 16-step forms, heads
dealt to the XCDs or not, portions around a block of 128 queries, masks at the edges of a tile of 64 keys."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,rk,koff,H,G", [(192, 128, 0, 8, 1), (136, 128, 0, 3, 1), (200, 128, 0, 16, 1), (128, 128, 128, 16, 4), (64, 64, 64, 8, 2), (256, 256, 0, 2, 1)])
@pytest.mark.parametrize("lens,window,keep", [([129, 1, 64], 1 << 30, 0), ([300], 100, 0), ([65, 200], 64, 5)])
@pytest.mark.parametrize("sig", [False, True])
def test_prompt_tiles(native_lib, R, rk, koff, H, G, lens, window, keep, sig):
    """Scores and sums in fp32, weights rounded to bf16 (2^-9), as the result: 2^-7 of the row's size covers both."""
    from llmctl.ops import hybrid as hops
    from llmctl.ops import ref_hybrid as ref

    g = torch.Generator().manual_seed(R + H)
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).cuda()  # noqa: E731
    past, bs, rs = 70, 16, max(R + koff, rk)
    ctx = torch.tensor([n + past * (i % 2) for i, n in enumerate(lens)], dtype=torch.int32)
    mb = int(ctx.max()) // bs + 1
    bt = torch.randperm(mb * len(lens), generator=g).view(len(lens), mb).int().cuda()
    cache = r(mb * len(lens), bs, G * rs)
    qa = r(sum(lens), H, R)
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    h = dict(sig_bias=-torch.rand(H, generator=g).cuda(), dist_a=torch.rand(H, generator=g).cuda() * 0.1, dist_b=torch.rand(H, generator=g).cuda()) if sig else {}
    args = (cu, ctx.cuda(), window, None, R ** -0.5, rk)
    got = hops.latent_attention_prefill(qa, cache, bt, *args, max(lens), groups=G, koff=koff, keep_first=keep, **h)
    want = ref.latent_attention(qa.float().cpu(), cache.float().cpu(), bt.cpu(), args[0].cpu(), ctx, *args[2:], groups=G, koff=koff, keep_first=keep,
                                **{k: v.cpu() for k, v in h.items()})
    err = (got.float().cpu().view(want.shape) - want).norm(dim=-1)
    assert (err <= 2.0 ** -7 * want.norm(dim=-1) + 2.0 ** -7 * want.norm() / want[..., 0].numel() ** 0.5).all()


@pytest.mark.parametrize("R,rk", [(136, 64), (192, 128), (200, 96), (256, 128)])
@pytest.mark.parametrize("past,window,chunk", [(0, 1 << 30, 1 << 30), (70, 40, 1 << 30), (50, 10, 1 << 30), (32, 1 << 30, 32), (200, 64, 96)])
@pytest.mark.parametrize("opt", ["", "sink", "sink above", "sink below", "cap", "scale", "sink cap scale"])
def test_two_groups_of_waves_share_a_tiles_keys(native_lib, R, rk, past, window, chunk, opt):
    """Keys of 129 to 256 columns: the first group takes a tile's first 32 keys, the second the rest, and their maxima, denominators and outputs meet at the end.  Portions of which only
    the first half of a tile is visible (20 tokens, no past), or only the second (windows of 10 and chunks of 32 behind them), and rows that see both; the sink counts once."""
    from llmctl.ops import hybrid as hops
    from llmctl.ops import ref_hybrid as ref

    H, G, bs, lens = 4, 2, 16, [1, 20, 33, 150]
    g = torch.Generator().manual_seed(R + past)
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).cuda()  # noqa: E731
    ctx = torch.tensor([n + past for n in lens], dtype=torch.int32)
    mb = int(ctx.max()) // bs + 1
    bt = torch.randperm(mb * len(lens), generator=g).view(len(lens), mb).int().cuda()
    cache, qa = r(mb * len(lens), bs, G * R), r(sum(lens), H, R)
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    sink = torch.randn(H, generator=g) + (12.0 if "above" in opt else -30.0 if "below" in opt else 0.0) if "sink" in opt else None
    kw = dict(groups=G, chunk=chunk, hscale=torch.rand(H, generator=g) * 2 if "scale" in opt else None, softcap=3.0 if "cap" in opt else 0.0)
    cuda = lambda t: t.cuda() if torch.is_tensor(t) else t  # noqa: E731
    got = hops.latent_attention_prefill(qa, cache, bt, cu, ctx.cuda(), window, cuda(sink), R ** -0.5, rk, max(lens), **{k: cuda(v) for k, v in kw.items()})
    want = ref.latent_attention(qa.float().cpu(), cache.float().cpu(), bt.cpu(), cu.cpu(), ctx, window, sink, R ** -0.5, rk, **kw)
    # scores and sums in fp32, weights rounded to bf16 (2^-8 at most, each their own way), as the result: a row's error is at most 2^-8 of its size and 2^-8 of its values' under their weights
    err = (got.float().cpu().view(want.shape) - want).norm(dim=-1)
    size = ref.latent_attention(qa.float().cpu(), torch.cat([cache.float().cpu().view(-1, G, R)[..., :rk].abs(), cache.float().cpu().view(-1, G, R)], 2).view(mb * len(lens), bs, -1), bt.cpu(),
                                cu.cpu(), ctx, window, sink, R ** -0.5, rk, **{**kw, "koff": rk})
    assert (err <= 2.0 ** -8 * (want.norm(dim=-1) + size.norm(dim=-1)) + 1e-30).all()

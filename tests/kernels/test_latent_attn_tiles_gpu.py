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

"""Attention over row caches with a gate on its output, in the kernels that store it and after those that do not, against the same attention and a pass of its own for the gate:
a gate per column and per head, prompts and decode rows whose keys are split over workgroups or not, several value tiles, turned outputs, sigmoid weights, fp32."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# heads, kv groups, key width, value width, contexts of the decode rows
@pytest.mark.parametrize("H,G,R,rk", [(1, 1, 8, 8), (16, 4, 128, 128), (8, 8, 192, 128), (3, 1, 256, 200), (16, 1, 576, 512), (64, 1, 128, 128), (2, 1, 20, 12)])
@pytest.mark.parametrize("form", ["plain", "turn", "sigmoid", "fp32"])
@pytest.mark.parametrize("each", [True, False])
def test_gate(H, G, R, rk, form, each):
    from llmctl.ops import hybrid as hops

    if form == "turn" and (rk % 2 or R > 256):
        pytest.skip("turned outputs are even and of keys up to 256 wide")
    dtype = torch.float32 if form == "fp32" else torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(H + R)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    ctx = torch.tensor([1, 70, 900], dtype=torch.int32, device="cuda")
    bs, mb = 16, 57
    cache = r(3 * mb, bs, G * max(R, rk)).to(dtype)
    bt = torch.randperm(3 * mb, generator=g, device="cuda").view(3, mb).int()
    opt = dict(groups=G)
    if form == "turn":
        opt["ofreq"] = torch.rand(rk // 2, generator=g, device="cuda")
    if form == "sigmoid":
        opt["sig_bias"] = r(H)

    def check(call, rows, off=4):
        qa = r(rows, H, R).to(dtype)
        gate = (3.0 * r(rows, off + (H * rk if each else H))).to(dtype)[:, off:]  # (quads, and none)
        want = hops.sigmoid_gate_mul(call(qa).reshape(rows, H * rk), gate)
        got = call(qa, gate=gate).reshape(rows, H * rk)
        # the same product of the same rounded output, but for an ulp of the exponential and of the reciprocal: next to a tie it rounds to the neighbour, at most 2^-7 away in bf16
        assert got.dtype == want.dtype and bool(((got.double() - want.double()).abs() <= (2.0**-7 if dtype == torch.bfloat16 else 2.0**-21) * want.double().abs()).all())

    check(lambda qa, **kw: hops.latent_attention_decode(qa, cache, bt, ctx, hops.NO_LIMIT, None, R**-0.5, rk, max_ctx=900, **opt, **kw), 3, 3)
    check(lambda qa, **kw: hops.latent_attention_decode(qa, cache, bt, ctx, 50, None, R**-0.5, rk, max_ctx=900, **opt, **kw), 3)  # a single split
    for lens in ([1, 60, 140], [1, 3, 5]):
        cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
        check(lambda qa, **kw: hops.latent_attention_prefill(qa, cache, bt, cu, ctx, 100, None, R**-0.5, rk, max(lens), **opt, **kw), sum(lens), 3 + lens[1] % 2)

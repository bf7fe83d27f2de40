"""Vector gradients written by their kernels (``llmctl/ops/csrc/col_sum.hip``, ``norm_bwd_into``) and the unrotated QKV attention
(``flash_attn_bwd_qkv`` without tables), against float64 sums and the sliced form: one row, row and column remainders, widths on
either side of a column block, strided rows, fp32 and bf16 targets, stored and added."""

import pytest
import torch

from llmctl import ops
from llmctl.ops._lib import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("T,N,pad", [(1, 8, 0), (7, 248, 8), (8, 256, 0), (31, 264, 0), (33, 768, 0), (257, 2304, 16), (5000, 40, 0), (9000, 1600, 0)])
def test_column_sums(T, N, pad, f32):
    g = torch.Generator().manual_seed(T + N)
    x = torch.randn(T, N + pad, generator=g).bfloat16().cuda()[:, :N]
    out = torch.randn(N, generator=g).to(torch.float32 if f32 else torch.bfloat16).cuda()
    old, want = out.double(), x.double().sum(0)
    size = x.double().abs().sum(0) + old.abs()
    tol = (2.0 ** -20 if f32 else 0.0) * size + (0.0 if f32 else 2.0 ** -8) * (want.abs() + old.abs() + 1e-3) + 2.0 ** -20 * size
    for add in (False, True):  # fp32 sums of at most 2^14 terms (relative 2^-20 of their magnitudes), one rounding to bf16 at the end
        native().col_sum_(x, out, add)
        assert ((out.double() - (want + (old if add else 0))).abs() <= tol).all()
        out.copy_(old)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("T,H", [(1, 64), (5, 520), (300, 768), (2100, 1600), (2100, 2304), (600, 4096), (40, 5120)])
@pytest.mark.parametrize("ln", [False, True])
def test_norm_gradients_into_vectors(T, H, ln, f32):
    g = torch.Generator().manual_seed(T + H)
    r = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()
    x, dy, w, b, dres = r(T, H), r(T, H), r(H), r(H), r(T, H)
    if ln:
        _, mu, rstd = native().layernorm_fwd(x, w, b, 1e-5)
        dx0, dw0, db0 = native().layernorm_bwd(dy, x, w, mu, rstd, dres)
    else:
        _, rstd = native().rmsnorm_fwd(x, w, 1e-5)
        mu = db0 = None
        dx0, dw0 = native().rmsnorm_bwd(dy, x, w, rstd, dres)
    xd, dyd = x.double(), dy.double()
    xh = (xd - (mu.double()[:, None] if ln else 0)) * rstd.double()[:, None]
    sums = [(dyd * xh).sum(0)] + ([dyd.sum(0)] if ln else [])
    mags = [(dyd * xh).abs().sum(0)] + ([dyd.abs().sum(0)] if ln else [])
    for add in (False, True):
        olds = [torch.randn(H, generator=g).to(torch.float32 if f32 else torch.bfloat16).cuda() for _ in sums]
        outs = [o.clone() for o in olds]
        dx = native().norm_bwd_into(dy, x, w, mu, rstd, dres, outs[0], add, outs[1] if ln else None, add)
        assert torch.equal(dx, dx0)
        for out, old, s, m in zip(outs, olds, sums, mags):
            want = s + (old.double() if add else 0)
            # fp32 sums (relative 2^-18 of the terms' magnitudes: products of rounded factors), one rounding to bf16
            tol = 2.0 ** -18 * (m + old.double().abs()) + (0.0 if f32 else 2.0 ** -8) * want.abs()
            assert ((out.double() - want).abs() <= tol).all()
    if not f32:
        outs = [torch.empty(H, device="cuda").bfloat16() for _ in sums]
        native().norm_bwd_into(dy, x, w, mu, rstd, dres, outs[0], False, outs[1] if ln else None, False)
        assert torch.equal(outs[0], dw0) and (not ln or torch.equal(outs[1], db0))


@pytest.mark.parametrize("docs", [False, True])
@pytest.mark.parametrize("B,S,nq,nkv,D", [(1, 1, 2, 2, 64), (2, 65, 4, 2, 64), (1, 300, 3, 3, 128), (2, 128, 12, 12, 64)])
def test_unrotated_qkv_attention(B, S, nq, nkv, D, docs):
    g = torch.Generator().manual_seed(S)
    qkv = torch.randn(B * S, (nq + 2 * nkv) * D, generator=g).bfloat16().cuda().requires_grad_()
    do = torch.randn(B, S, nq, D, generator=g).bfloat16().cuda()
    ds = (torch.arange(S) // 40 * 40).int().expand(B, S).contiguous().cuda() if docs else None
    o = ops.qkv_flash_attention(qkv, nq, nkv, B, S, ds)
    o.backward(do)
    ref = qkv.detach().clone().requires_grad_()
    q, k, v = (t.contiguous() for t in ref.view(B, S, -1, D).split((nq, nkv, nkv), dim=2))
    o2 = ops.flash_attention(q, k, v, causal=True, doc_start=ds)
    o2.backward(do)
    assert torch.equal(o, o2) and torch.equal(qkv.grad, ref.grad)  # the same kernels on other strides


def test_a_bias_gradient_can_be_differentiated():
    from llmctl.exec.linear import linear

    g = torch.Generator().manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()
    x, w, b = r(24, 64), r(32, 64), r(32).requires_grad_()
    y = linear(x, w, b)
    (gb,) = torch.autograd.grad((y.float() ** 3).sum(), b, create_graph=True)  # sum over rows of 3 y^2
    (ggb,) = torch.autograd.grad(gb.float().sum(), b)  # sum over rows of 6 y
    want = 6 * (x.double() @ w.double().t() + b.double()).sum(0)
    assert (ggb.double() - want).norm() <= 2.0 ** -5 * want.norm()

"""A decode step's LayerNorm and projection in one launch (``llmctl/ops/csrc/norm_linear.hip``) against float64: row
counts on either side of a wave's batches, row lengths that fill no 512-column piece or 32-deep step, outputs that fill no tile, with and
without residual, bias and activation; and QKV to bf16 and fp8 caches with a row that goes nowhere."""

import pytest
import torch

from llmctl import ops
from llmctl.ops._lib import native

pytestmark = pytest.mark.gpu


def _case(M, K, N, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    return r(M, K) * 3, r(M, K), r(K), r(K), r(N, K) * K ** -0.5, r(N)


def _exact(x, q, nw, nb, w, b, act):
    """float64 of the same bf16 inputs (the residual rounded once, as both forms do), and the bound: the normalised row is a bf16
    operand and the result a bf16 number (2^-9 each of the terms' magnitudes; twice that, for fp32 sums and the activation's slope)."""
    x = (x.float() + q.float()).bfloat16().double() if q is not None else x.double()
    xn = (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, unbiased=False, keepdim=True) + 1e-5) * nw.double() + nb.double()
    y = xn @ w.double().t() + (0 if b is None else b.double())
    bound = 2.0 ** -8 * (xn.abs() @ w.double().abs().t() + (0 if b is None else b.double().abs()))
    if act:
        y = torch.nn.functional.gelu(y, approximate="tanh" if act == 2 else "none")
    return y, bound


@pytest.mark.parametrize("M,K,N", [(1, 8, 4), (1, 768, 3072), (3, 40, 20), (4, 504, 16), (5, 512, 36), (8, 520, 100), (9, 768, 64), (16, 1024, 48),
                                   (12, 1032, 20), (7, 2048, 52), (12, 2048, 16)])
@pytest.mark.parametrize("res,bias,act", [(True, True, 1), (False, True, 0), (True, False, 2)])
def test_norm_linear(M, K, N, res, bias, act):
    x, q, nw, nb, w, b = _case(M, K, N, seed=M + K)
    q, b = (q if res else None), (b if bias else None)
    y, r = native().norm_linear(x, q, nw, nb, 1e-5, w, b, act)
    xn, want_r = ops.add_layernorm(x, q, nw, nb, 1e-5) if res else (ops.layernorm(x, nw, nb, 1e-5), None)
    want, bound = _exact(x, q, nw, nb, w, b, act)
    assert ((y.double() - want).abs() <= bound).all()
    assert torch.equal(r, want_r) if res else r.numel() == 0
    got, r2 = ops.decode_norm_linear(x, q, nw, nb, 1e-5, w, b, act="gelu" if act == 1 else None)
    if act != 2:
        assert ((got.double() - want).abs() <= bound).all()
    assert torch.equal(r2, want_r if res else x)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("M,K,nq,nkv,D", [(1, 768, 12, 12, 64), (5, 64, 4, 2, 8), (16, 256, 3, 1, 40)])
def test_norm_qkv_cache(M, K, nq, nkv, D, fp8):
    x, res, nw, nb, w, b = _case(M, K, (nq + 2 * nkv) * D, seed=M)
    slots = torch.randperm(40, device="cuda")[:M].long()
    if M > 1:
        slots[1] = -1
    caches = [torch.zeros(10, 4, nkv, D, device="cuda").to(torch.float8_e4m3fn if fp8 else torch.bfloat16) for _ in range(4)]
    q, r = ops.decode_norm_qkv_cache(x, res, nw, nb, 1e-5, w, b, nq, nkv, caches[0], caches[1], slots)
    xn, want_r = ops.add_layernorm(x, res, nw, nb, 1e-5)
    want, _, _ = ops.qkv_split_cache(ops.decode_linear(xn, w, b), nq, nkv, caches[2], caches[3], slots)
    exact, bound = _exact(x, res, nw, nb, w, b, 0)
    assert ((q.reshape(M, -1).double() - exact[:, :nq * D]).abs() <= bound[:, :nq * D]).all() and torch.equal(r, want_r)
    for i in (0, 1):
        rows = caches[i].float().reshape(40, -1)
        cols = slice((nq + i * nkv) * D, (nq + (i + 1) * nkv) * D)
        live = slots >= 0
        e, bd = exact[live][:, cols], bound[live][:, cols]
        # fp8 (3 mantissa bits, subnormal step 2^-9): half a step on top
        assert ((rows[slots[live]].double() - e).abs() <= bd + ((2.0 ** -4 * (e.abs() + bd) + 2.0 ** -10) if fp8 else 0)).all()
        rows[slots[live]] = 0
        assert not rows.any()  # nothing else was written
        assert ((caches[i].float() != 0) == (caches[i + 2].float() != 0)).float().mean() > 0.99

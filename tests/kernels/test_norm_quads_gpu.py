"""Residual-and-norm rows in quads (``stream.hip``, ``gated_stream.hip``) on either side of a thread's one, two and four quads, widths that
leave threads idle, rows wider than the quads form or not in fours or not aligned (the general form), strided inputs: against float64."""

import pytest
import torch

from llmctl.ops import hybrid as hops

pytestmark = pytest.mark.gpu
WIDTHS = [4, 100, 1024, 1028, 2048, 2052, 4096, 4100, 1030, 6]


def _near(got, want, size, bf16):
    # fp32 over a row: 2^-18 of the terms' size; a bf16 result rounds once
    assert ((got.double() - want).abs() <= 2.0 ** -18 * size + (2.0 ** -8 if bf16 else 0.0) * want.abs()).all()


@pytest.mark.parametrize("W", WIDTHS)
@pytest.mark.parametrize("bf16,pad", [(True, 0), (True, 8), (False, 0), (True, 2)])
@pytest.mark.parametrize("second", [True, False])
def test_add_layernorm_rows(W, bf16, pad, second):
    g = torch.Generator(device="cuda").manual_seed(W)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, z, w, b = r(5, W), (r(5, W) if second else None), r(W), r(W)
    a = r(5, W + pad).to(torch.bfloat16 if bf16 else torch.float32)[:, pad // 2 * 2:]
    want = x.double() + a.double() + (z.double() if second else 0)
    y = (want - want.mean(-1, keepdim=True)) / torch.sqrt(want.var(-1, unbiased=False, keepdim=True) + 1e-5) * w.double() + b.double()
    h = hops.add_layernorm_f32_(x, a, z, w, b, 1e-5, a.dtype)
    _near(x, want, want.abs() + 4, False)
    _near(h, y, w.double().abs() * 8 + b.double().abs(), bf16)
    x2 = x.clone()
    h2 = hops.layernorm_f32(x2, w, b, 1e-5, a.dtype)  # the norm alone leaves x as it is
    _near(h2, y, w.double().abs() * 8 + b.double().abs(), bf16)
    assert torch.equal(x2, x)
    hops.residual_add_(x2, a, z)  # the sum alone
    _near(x2, want + a.double() + (z.double() if second else 0), want.abs() + 8, False)


@pytest.mark.parametrize("W", WIDTHS)
@pytest.mark.parametrize("ty,tr,pad", [(torch.bfloat16, torch.bfloat16, 0), (torch.float32, torch.bfloat16, 8), (torch.bfloat16, torch.bfloat16, 2)])
@pytest.mark.parametrize("last", [False, True])
def test_gated_norm_add_norm_rows(W, ty, tr, pad, last):
    g = torch.Generator(device="cuda").manual_seed(W)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, wp, wn = r(5, W), r(W), r(W)
    y, gate = r(5, W + pad).to(ty)[:, pad:], r(5, W + pad).to(tr)[:, pad:]
    v = y.double() * torch.sigmoid(gate.double())
    want = x.double() + v / torch.sqrt((v * v).mean(-1, keepdim=True) + 1e-5) * wp.double()
    n = want / torch.sqrt((want * want).mean(-1, keepdim=True) + 1e-5) * wn.double()
    h = hops.gated_norm_add_norm_f32_(x, y, gate, wp, None if last else wn, 1e-5, torch.bfloat16)
    _near(x, want, want.abs() + 8 * wp.double().abs() + 1, False)
    if not last:
        _near(h, n, 8 * wn.double().abs(), True)

"""Per-head products of a decode step (``llmctl/ops/csrc/hybrid/head_rows.hip``) against float64: row counts around a tile, K and N that fill
no step or workgroup, several batches of steps, strided rows, rotary parts of both layouts and none, with and without gate."""

import pytest
import torch

from llmctl.ops import hybrid as hops

pytestmark = pytest.mark.gpu


def _product(x, w):
    """float64 of bf16 inputs, and one bf16 rounding over fp32 sums (2^-8 of the result, 2^-20 of the terms)."""
    y = torch.einsum("thk,hkn->thn", x.double(), w.double())
    return y, 2.0 ** -8 * y.abs() + 2.0 ** -20 * torch.einsum("thk,hkn->thn", x.double().abs(), w.double().abs())


@pytest.mark.parametrize("T,H,dn,dr,rot,rk,inter", [(1, 1, 4, 0, 0, 8, False), (16, 16, 128, 64, 64, 512, False), (17, 3, 36, 8, 4, 40, True),
                                                    (32, 2, 600, 12, 12, 72, True), (5, 4, 32, 16, 8, 32, False)])
def test_latent_queries(T, H, dn, dr, rot, rk, inter):
    g = torch.Generator().manual_seed(T + dn)
    z = torch.randn(T, H * (dn + dr) + 4, generator=g).bfloat16().cuda()
    q = z[:, :H * (dn + dr)].unflatten(1, (H, dn + dr))
    w = (torch.randn(H, dn, rk, generator=g) * dn ** -0.5).bfloat16().cuda()
    pos = torch.randint(0, 3000, (T,), generator=g, dtype=torch.int32).cuda()
    freq = torch.rand(rot // 2, generator=g).cuda()
    assert hops.head_rows_ok(q, w)
    got = hops.latent_queries(q, w, pos, freq, rot, inter, 1.25)
    y, bound = _product(q[:, :, :dn], w)
    assert ((got[:, :, :rk].double() - y).abs() <= bound).all()
    other = hops.latent_q_assemble(y.bfloat16(), q, pos, freq, rot, dn, inter, 1.25)
    assert ((got[:, :, rk:].float() - other[:, :, rk:].float()).abs() <= 2.0 ** -7 * other[:, :, rk:].float().abs() + 1e-4).all()


@pytest.mark.parametrize("T,H,rk,dv", [(1, 1, 4, 8), (16, 16, 512, 128), (15, 2, 44, 24), (31, 3, 700, 136), (4, 5, 64, 32)])
@pytest.mark.parametrize("gated", [False, True])
def test_latent_values(T, H, rk, dv, gated):
    g = torch.Generator().manual_seed(rk)
    o = torch.randn(T, H, rk, generator=g).bfloat16().cuda()
    w = (torch.randn(H, rk, dv, generator=g) * rk ** -0.5).bfloat16().cuda()
    gate = torch.randn(T, H * dv + 8, generator=g).bfloat16().cuda()[:, 8:] if gated else None
    assert hops.head_rows_ok(o, w)
    got = hops.latent_values(o, w, gate).double()
    y, bound = (t.reshape(T, -1) for t in _product(o, w))
    if gated:  # rounded before the gate and after it
        s = torch.sigmoid(gate.double())
        y, bound = y * s, bound * s + 2.0 ** -8 * (y * s).abs()
    assert ((got - y).abs() <= bound).all()

"""Embedding rows of serving steps: with positions, scaled and normed; widths on either side of a thread's one, two and four quads, widths and
addresses that only the general forms take, one row and many, repeated and last ids."""

import pytest
import torch

from llmctl import ops
from llmctl.ops import hybrid as hops
from llmctl.ops import ref_hybrid

pytestmark = pytest.mark.gpu
V = 37


def _table(W, dtype, seed, off=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(V * W + off, generator=g, device="cuda").to(dtype)[off:].view(V, W)


def _ids(T):
    return torch.tensor([(5 * i) % V if i % 3 else V - 1 for i in range(T)], device="cuda")


@pytest.mark.parametrize("T", [1, 16, 300])
@pytest.mark.parametrize("W,off", [(8, 0), (768, 0), (4096, 0), (12, 0), (768, 1)])
@pytest.mark.parametrize("pos", [None, torch.int32, torch.int64])
def test_embed_rows(T, W, off, pos):
    table, ptable, ids = _table(W, torch.bfloat16, 1, off), _table(W, torch.bfloat16, 2, off), _ids(T)
    if pos is None:
        got, want = ops.embed_rows(ids, table), table[ids]
    else:
        p = (ids * 3 % V).to(pos)
        got, want = ops.embed_rows(ids, table, p, ptable), table[ids] + ptable[p.long()]
    assert torch.equal(got, want)


def _near(got, want, size, bf16):
    # fp32 over a row: 2^-18 of the terms' size; a bf16 result rounds once
    assert ((got.double() - want).abs() <= 2.0 ** -18 * size + (2.0 ** -8 if bf16 else 0.0) * want.abs()).all()


@pytest.mark.parametrize("W,off", [(4, 0), (1024, 0), (1028, 0), (2048, 0), (2052, 0), (4096, 0), (4100, 0), (1030, 0), (6, 0), (1024, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [1, 33])
def test_embed_norms(W, off, dtype, T):
    table, ptable, ids = _table(W, dtype, 3, off), _table(W, dtype, 4, off), _ids(T)
    g = torch.Generator(device="cuda").manual_seed(5)
    w, b = torch.randn(W, generator=g, device="cuda"), torch.randn(W, generator=g, device="cuda")
    x, h = hops.embed_layernorm_f32(ids, table, 2.5, w, b, 1e-5)
    assert torch.equal(x, table[ids].float() * 2.5) and h.dtype == dtype
    d = x.double()
    want = (d - d.mean(-1, keepdim=True)) / torch.sqrt(d.var(-1, unbiased=False, keepdim=True) + 1e-5) * w.double() + b.double()
    _near(h, want, w.double().abs() * 8 + b.double().abs(), dtype == torch.bfloat16)
    pos = (ids * 3 % V).to(torch.int32)
    x, h = hops.embed_rmsnorm_f32(ids, pos, table, ptable, w, 1e-5, dtype)
    xr, _ = ref_hybrid.embed_rmsnorm_f32(ids, pos, table, ptable, w, 1e-5, dtype)
    assert torch.equal(x, xr)
    d = x.double()
    _near(h, d / torch.sqrt(d.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double(), w.double().abs() * 8, dtype == torch.bfloat16)

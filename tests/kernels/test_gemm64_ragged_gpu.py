"""The 256 x 256 kernel on rows and columns that fill no whole tile, with bias, gated, with its last round split over K, on strided rows between
others: against float64, and what lies around the operands does not matter."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(M, K, g, lead=8):
    """[M, K] rows inside a larger buffer whose other entries are NaN."""
    buf = torch.full((M + 2, K + 2 * lead), float("nan"), device="cuda", dtype=torch.bfloat16)
    x = buf[1:1 + M, lead:lead + K]
    x.copy_(torch.randn(M, K, generator=g, device="cuda"))
    return x


@pytest.mark.parametrize("M", [1, 128, 255, 256, 257, 700])
@pytest.mark.parametrize("N,K", [(8, 256), (248, 384), (256, 1024), (264, 2048), (1000, 256), (4240, 1024)])
@pytest.mark.parametrize("bias", [False, True])
def test_ragged_product(M, N, K, bias):
    from llmctl.ops._lib import native

    g = torch.Generator(device="cuda").manual_seed(M + N)
    x, w = _rows(M, K, g), _rows(N, K, g)
    b = torch.randn(N, generator=g, device="cuda").bfloat16() if bias else None
    want = x.double() @ w.double().t() + (b.double() if bias else 0)
    got = native().gemm64_fwd(x, w, b)
    # fp32 sums of K bf16 products (errors of at most K ulp, far less in practice), rounded to bf16 once
    size = x.double().abs() @ w.double().abs().t()
    assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -20 * size).all()


@pytest.mark.parametrize("M", [1, 200, 257, 513])
@pytest.mark.parametrize("F,K", [(128, 256), (384, 1024), (1024, 2048)])
def test_ragged_gated_product(M, F, K):
    from llmctl.ops._lib import native

    g = torch.Generator(device="cuda").manual_seed(M + F)
    x, w = _rows(M, K, g), (torch.randn(2 * F, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    z = (x.double() @ w.double().t()).bfloat16().double()
    want = torch.nn.functional.silu(z[:, :F]) * z[:, F:]
    got = native().gemm64_fwd(x, w, None, True)
    # a gate or an up value on a rounding edge may round the other way (2^-8 each), and the result rounds once
    assert ((got.double() - want).abs() <= 2.0 ** -6 * want.abs() + 2.0 ** -7 * (z[:, :F].abs() + z[:, F:].abs() + 1) * 2.0 ** -2).all()
    assert (got.double() - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.parametrize("M,N,K,own", [(2300, 4240, 1024, True), (2200, 4240, 1024, False), (2304, 4096, 1024, False), (2300, 4244, 1024, False), (2300, 4240, 1152, True),
                                       (2300, 4240, 1088, False), (4600, 4240, 896, False)])
def test_rule_of_odd_products(M, N, K, own, monkeypatch):
    from llmctl.ops import functional as F

    g = torch.Generator(device="cuda").manual_seed(M)
    x, w = (torch.randn(n, K, generator=g, device="cuda").bfloat16() for n in (M, N))
    calls, lib = [], torch.nn.functional.linear
    monkeypatch.setattr(torch.nn.functional, "linear", lambda *a: calls.append(1) or lib(*a))
    y = F.odd_linear(x, w)
    assert calls == ([] if own else [1])
    want = x.double() @ w.double().t()
    assert (y.double() - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.parametrize("T,own", [(1100, True), (1000, False), (1024, True)])
def test_rule_of_gated_products(T, own, monkeypatch):
    from llmctl import ops

    g = torch.Generator(device="cuda").manual_seed(T)
    F, K = 5504, 512
    x, w = torch.randn(1, T, K, generator=g, device="cuda").bfloat16(), (torch.randn(2 * F, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    calls, lib = [], torch.nn.functional.linear
    monkeypatch.setattr(torch.nn.functional, "linear", lambda *a: calls.append(1) or lib(*a))
    got = ops.up_swiglu(x, w)
    assert calls == ([] if own else [1]) and got.shape == (1, T, F)
    z = x[0].double() @ w.double().t()
    want = torch.nn.functional.silu(z[:, :F]) * z[:, F:]
    assert (got[0].double() - want).norm() <= 2.0 ** -7 * want.norm()

"""Prompt products on tiles of up to 288 rows x 128: rows that just fill a tile and one more, the shortest K and odd numbers of pairs of K-tiles, outputs that fill no tile, rows wider
than the matrix, a bias; and the route that takes them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 33, 128, 129, 256, 288, 289, 544, 545, 1000])
@pytest.mark.parametrize("N,K,pad", [(8, 256, 0), (128, 384, 8), (264, 640, 0), (1000, 2048, 8)])
@pytest.mark.parametrize("form", [1, 2])
def test_products(M, N, K, pad, form):
    from llmctl.ops._lib import native

    g = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)
    rows = lambda n: torch.randn(n, K + pad, generator=g, device="cuda").bfloat16()[:, :K]
    x, w = rows(M), rows(N)
    b = torch.randn(N, generator=g, device="cuda").bfloat16() if pad else None
    got = native().gemm_rows(x, w, b, form)
    X, W = x.double(), w.double()
    ref, mag = X @ W.t(), X.abs() @ W.abs().t()
    if b is not None:
        ref, mag = ref + b.double(), mag + b.double().abs()
    bound = (K + 1) * 2.0**-24 * mag  # fp32 sums of K exact products in any order; then one rounding
    assert bool(((got.double() - ref).abs() <= bound + 2.0**-8 * (ref.abs() + bound)).all())


@pytest.mark.parametrize("M", [1, 33, 128, 129, 288, 289, 700])
@pytest.mark.parametrize("N,K,splits", [(8, 512, 2), (264, 896, 3), (1000, 2048, 8), (136, 4224, 16)])
@pytest.mark.parametrize("form,act", [(1, 0), (2, 0), (1, 1), (2, 2)])
def test_ranges_of_k_and_activations(M, N, K, splits, form, act):
    """Ranges of 256 on, of unlike length too; erf and tanh GELU of the sum, in the tiles' epilogue and in the pass that adds the ranges."""
    from llmctl.ops._lib import native

    g = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)
    x, w = (torch.randn(n, K, generator=g, device="cuda").bfloat16() for n in (M, N))
    b = torch.randn(N, generator=g, device="cuda").bfloat16()
    X = x.double()
    w = (w.float() * 2.0 ** -round(K.bit_length() / 2)).bfloat16()  # (an exact scale: sums near 1, where the GELUs bend)
    W = w.double()
    ref, mag = X @ W.t() + b.double(), X.abs() @ W.abs().t() + b.double().abs()
    bound = (K + splits + 1) * 2.0**-24 * mag  # fp32 sums of exact products
    if act:
        # both GELUs' slopes stay below 1.13; 3e-7 |sum| for the fp32 forms (erf: 7.3e-8)
        bound = 1.13 * bound + 2.0**-20 * ref.abs()
        ref = torch.nn.functional.gelu(ref, approximate="tanh" if act == 2 else "none")
    for n in (1, splits):
        got = native().gemm_rows(x, w, b, form, n, act)
        assert bool(((got.double() - ref).abs() <= bound + 2.0**-8 * (ref.abs() + bound)).all())
    y = torch.full((M + 1, N // 8, 16), 7.0, device="cuda", dtype=torch.bfloat16)
    native().gemm_rows_into(x, w, b, form, y[:M, :, :8], splits)
    assert torch.equal(y[:M, :, :8].reshape(M, N), native().gemm_rows(x, w, b, form, splits)) and bool((y[:, :, 8:] == 7).all()) and bool((y[M] == 7).all())


def test_route():
    """Sizes of the rule run on these tiles, inside autograd too; other callers keep the library: a wanted gradient outside of it, autocast, batched rows of a transform."""
    import importlib

    L = importlib.import_module("llmctl.exec.linear")
    assert L.rows_form(2048, 2048, 2048) == 2 and L.rows_form(2911, 2048, 1024) == 1
    assert not any(L.rows_form(*s) for s in ((32, 2048, 2048), (2048, 2044, 2048), (2048, 2048, 2000), (2048, 2048, 128), (3379, 8192, 2048), (900, 12288, 4096), (0, 256, 256)))
    assert L.rows_form(128, 4096, 11008) >> 2 and L.rows_form(200, 2048, 2048, False, True) >> 2 and not L.rows_form(200, 2048, 2048)  # (the host's gain alone)
    x, w = (torch.randn(n, 1024, device="cuda", dtype=torch.bfloat16) for n in (1500, 2048))
    b = torch.randn(2048, device="cuda", dtype=torch.bfloat16)
    ref = x.double() @ w.double().t() + b.double()
    for y in (L.rows_linear(x, w, b), L.rows_linear(x.view(3, 500, 1024), w, b).view(1500, 2048)):
        assert float((y.double() - ref).norm() / ref.norm()) < 2.0**-9
    p = w.clone().requires_grad_()
    assert L.rows_linear(x, p, b) is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert L.rows_linear(x, w, b) is None
    assert L.rows_linear(x[:, 1:], w[:, 1:]) is None and L.rows_linear(x.t().contiguous().t(), w) is None and L.rows_linear(x.float(), w.float()) is None
    y = torch.vmap(lambda t: L.forward_linear(t, w, b))(x.view(3, 500, 1024))
    assert float((y.reshape(1500, 2048).double() - ref).norm() / ref.norm()) < 2.0**-8
    xg = x.clone().requires_grad_()
    y = L.linear(xg, p, b)
    y.sum().backward()
    assert float((y.double() - ref).norm() / ref.norm()) < 2.0**-9 and xg.grad is not None and p.grad is not None


@pytest.mark.parametrize("M,K", [(33, 256), (129, 384), (545, 640)])
@pytest.mark.parametrize("groups,n,gap", [(1, 264, 8), (3, 88, 16), (33, 8, 8), (16, 256, 64)])
@pytest.mark.parametrize("form", [1, 2])
def test_into_groups_that_lie_apart(M, K, groups, n, gap, form):
    from llmctl.ops._lib import native

    g = torch.Generator(device="cuda").manual_seed(M + groups)
    x, w = (torch.randn(r, K, generator=g, device="cuda").bfloat16() for r in (M, groups * n))
    y = torch.full((M + 1, groups, n + gap), 7.0, device="cuda", dtype=torch.bfloat16)
    native().gemm_rows_into(x, w, None, form, y[:M, :, :n])
    assert torch.equal(y[:M, :, :n].reshape(M, -1), native().gemm_rows(x, w, None, form))
    assert bool((y[:, :, n:] == 7).all()) and bool((y[M] == 7).all())


def test_linear_into_takes_any_rows():
    from llmctl.ops import hybrid as hops

    for T, dtype in ((1, torch.bfloat16), (20, torch.bfloat16), (300, torch.bfloat16), (40, torch.float32)):
        x, w = torch.randn(T, 512, device="cuda", dtype=dtype), torch.randn(4 * 64, 512, device="cuda", dtype=dtype)
        y = torch.zeros(T, 4, 72, device="cuda", dtype=dtype)
        hops.linear_into(x, w, y[:, :, :64])
        assert torch.equal(y[:, :, :64].reshape(T, 256), hops.linear(x, w)) and not y[:, :, 64:].any()

"""Products of a few rows as sums over ranges of K, and the residual norm that adds them: ragged ranges and outputs, every row count's form, one and two
results, with and without a bias."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(4, 8), (132, 200), (1024, 1024), (2048, 8192), (4096, 264)])
@pytest.mark.parametrize("parts", [1, 2, 4, 16])
def test_parts_add_up(M, N, K, parts):
    from llmctl.ops.hybrid import native_hybrid

    g = torch.Generator(device="cuda").manual_seed(M * N + K)
    x, w = torch.randn(M, K + 8, generator=g, device="cuda").bfloat16()[:, :K], torch.randn(N, K, generator=g, device="cuda").bfloat16()
    p = native_hybrid().rows_parts(x, w, parts)
    assert p.shape[0] <= parts and p.shape[1:] == (M, N)
    ref, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert bool(((p.double().sum(0) - ref).abs() <= K * 2.0**-24 * mag).all())  # fp32 sums of exact products


@pytest.mark.parametrize("M,N", [(1, 6), (3, 6), (5, 10), (7, 513), (17, 1), (32, 4095)])
def test_ranges_that_start_between_quads(M, N):
    """Ranges of M * N sums that are no multiple of four: the second one and later start off 16 bytes, where nothing is stored in quads."""
    from llmctl.ops.hybrid import native_hybrid

    K = 1000
    g = torch.Generator(device="cuda").manual_seed(M * N)
    x, w = torch.randn(M, K, generator=g, device="cuda").bfloat16(), torch.randn(N, K, generator=g, device="cuda").bfloat16()
    p = native_hybrid().rows_parts(x, w, 4)
    part = (K // 4 + 31) // 32 * 32
    for i, got in enumerate(p):
        xi, wi = x[:, i * part:(i + 1) * part].double(), w[:, i * part:(i + 1) * part].double()
        assert bool(((got.double() - xi @ wi.t()).abs() <= part * 2.0**-24 * (xi.abs() @ wi.abs().t())).all())


@pytest.mark.parametrize("T", [1, 7, 32])
@pytest.mark.parametrize("W", [4, 260, 1024, 2048, 4096])
@pytest.mark.parametrize("n1,n2,bias", [(1, 0, False), (4, 0, True), (3, 2, False), (16, 1, True)])
def test_norm_of_parts(T, W, n1, n2, bias):
    from llmctl.ops import hybrid as hops

    g = torch.Generator(device="cuda").manual_seed(T * W + n1)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, y1, y2 = rand(T, W), rand(n1, T, W), rand(n2, T, W) if n2 else None
    b, w = rand(W).bfloat16() if bias else None, rand(W)
    y = 0.5 * (y1.double().sum(0) + (b.double() if bias else 0.0)) + (0.25 * y2.double().sum(0) if n2 else 0.0)
    add = 0.5 * y / (y.pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * (w.double() + 1.0)
    want = x.double() + add
    h = hops.norm_add_f32_(x, hops.RowParts(y1, b), 0.5, hops.RowParts(y2, None) if n2 else None, 0.25, w, 0.5, 1e-6, True, torch.bfloat16)
    size = 0.5 * y1.double().abs().sum(0) + (0.25 * y2.double().abs().sum(0) if n2 else 0.0) + 2.0
    # fp32 sums of n1 + n2 + 2 terms, a norm and four products
    tol = (n1 + n2 + 40) * 2.0**-23 * (x.double().abs() + want.abs() + size * (w.double().abs() + 1.0))
    assert bool(((x.double() - want).abs() <= tol).all())
    assert torch.equal(h, x.bfloat16())


@pytest.mark.parametrize("T,W", [(1, 4), (7, 260), (16, 2048), (32, 4096)])
@pytest.mark.parametrize("parts", [True, False])
def test_norm_with_the_next(T, W, parts):
    """The last residual update and the final norm in one pass: the same stream, and x's own norm."""
    from llmctl.ops import hybrid as hops

    g = torch.Generator(device="cuda").manual_seed(T + W)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x, w, wn, y = rand(T, W), rand(W), rand(W), rand(3, T, W)
    y = hops.RowParts(y, None) if parts else y[0].bfloat16()
    x2 = x.clone()
    hops.norm_add_f32_(x2, y, 0.5, None, 0.0, w, 0.5, 1e-6, True, torch.bfloat16)
    h = hops.norm_add_f32_(x, y, 0.5, None, 0.0, w, 0.5, 1e-6, True, torch.bfloat16, wn)
    assert torch.equal(x, x2)
    xd = x.double()
    want = xd / (xd.pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * (wn.double() + 1.0)
    assert bool(((h.double() - want).abs() <= (2.0**-8 + 1e-5) * want.abs() + 1e-30).all())


# (32 rows 4096 x 512: whole 8.9 us with the norm, in four ranges 9.8)
@pytest.mark.parametrize("M,N,K,parts", [(16, 2048, 8192, 4), (4, 2048, 2048, 2), (32, 4096, 512, 0), (32, 4096, 2048, 4), (33, 1024, 512, 0), (8, 4100, 512, 0), (8, 514, 512, 0)])
def test_rule(M, N, K, parts):
    from llmctl.ops import hybrid as hops

    x, w = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(N, K, device="cuda").bfloat16()
    b = torch.randn(N, device="cuda").bfloat16()
    y = hops.linear_parts(x, w, b)
    assert (y.parts.shape[0] if isinstance(y, hops.RowParts) else 0) == parts
    got = y.total() if parts else y
    ref = x.double() @ w.double().t() + b.double()
    assert bool(((got.double() - ref).abs() <= 2.0**-8 * ref.abs() + K * 2.0**-22 * 8).all())


@pytest.mark.parametrize("T", [1, 4, 5, 16, 17, 32])
@pytest.mark.parametrize("N,K", [(1, 8), (8, 2048), (32, 2056), (6, 4104)])
def test_fp32_weights(T, N, K):
    from llmctl.ops import hybrid as hops

    g = torch.Generator(device="cuda").manual_seed(T * N + K)
    x = torch.randn(T, K + 8, generator=g, device="cuda").bfloat16()[:, :K]
    w = torch.randn(N, K, generator=g, device="cuda")
    got = hops.linear_f32w(x, w, few=True)
    ref, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    err = (got.double() - ref).abs()
    assert bool((err <= (K / 256 + 24) * 2.0**-24 * mag).all())  # a thread's chain of K / 256 and the sums over threads
    lib = (torch.nn.functional.linear(x.float(), w).double() - ref).abs()
    assert err.pow(2).mean() <= 4 * lib.pow(2).mean() + (2.0**-25 * mag).pow(2).mean()


@pytest.mark.parametrize("off", ["w", "w_next", "x"])
def test_norm_vectors_off_16_bytes(off):
    """A norm vector or stream that is an offset view takes the general form, with the same stream."""
    from llmctl.ops import hybrid as hops

    T, W = 7, 260
    g = torch.Generator(device="cuda").manual_seed(5)
    rand = lambda n, name: torch.randn(n + 1, generator=g, device="cuda")[1 if name == off else 0:][:n]
    x, w, wn = rand(T * W, "x").view(T, W), rand(W, "w"), rand(W, "w_next")
    y = torch.randn(3, T, W, generator=g, device="cuda")
    yb = y.sum(0).bfloat16().double()  # (the general form's product is rounded)
    want = x.double() + 0.5 * yb / (yb.pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * (w.double() + 1.0)
    h = hops.norm_add_f32_(x, hops.RowParts(y, None), 1.0, None, 0.0, w, 0.5, 1e-6, True, torch.bfloat16, wn)
    assert bool(((x.double() - want).abs() <= 1e-5 * (x.double().abs() + want.abs() + 1.0)).all())  # an fp32 norm
    hw = want / (want.pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * (wn.double() + 1.0)
    assert bool(((h.double() - hw).abs() <= (2.0**-8 + 1e-5) * hw.abs() + 1e-5).all())

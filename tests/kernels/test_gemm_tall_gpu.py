"""Backward products on 256 x 128 tiles: one tile and several, the shortest K range and uneven ones, each output form, rows wider than the matrix."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(at, M, N, K, pad):
    g = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)
    shape = (K, M) if at else (M, K)
    a = torch.randn(shape[0], shape[1] + pad, generator=g, device="cuda").bfloat16()[:, :shape[1]]
    b = torch.randn(K, N + pad, generator=g, device="cuda").bfloat16()[:, :N]
    return a, b


def _bound(a, b, K, S):
    """fp32 sums of K exact products in any order, and S partial sums: (K + S) 2^-24 of the sum of magnitudes"""
    return (K + S) * 2.0**-24 * (a.abs() @ b.abs())


@pytest.mark.parametrize("at,M,N,K,S,pad", [
    (False, 256, 128, 256, 1, 0), (True, 256, 128, 256, 1, 8),        # one tile, the four peeled K-tiles alone
    (False, 512, 384, 384, 1, 8), (True, 768, 256, 640, 1, 0),        # an odd number of pairs of K-tiles
    (False, 1280, 128, 1152, 4, 0), (True, 256, 384, 1408, 5, 8),     # uneven ranges, tile rows that fill no group of four
    (True, 768, 768, 8192, 12, 0), (False, 8192, 768, 768, 1, 0),
])
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("add", [False, True])
def test_products(at, M, N, K, S, pad, f32, add):
    from llmctl.ops._lib import native

    a, b = _operands(at, M, N, K, pad)
    full = torch.full((M, N + 8), 3.0, device="cuda", dtype=torch.float32 if f32 else torch.bfloat16)
    out = full[:, :N]
    old = out.double() if add else torch.zeros((), device="cuda", dtype=torch.float64)
    if not add:
        out.fill_(float("nan"))
    native().gemm_tall(a, b, out, at, add, S)
    A, B = (a.t() if at else a).double(), b.double()
    ref, bound = A @ B + old, _bound(A, B, K, S + 1)
    if not f32:  # one rounding of the fp32 result
        bound = bound + 2.0**-8 * (ref.abs() + bound)
    assert bool(((out.double() - ref).abs() <= bound + 2.0**-23 * ref.abs()).all())
    assert bool((full[:, N:] == 3.0).all())


@pytest.mark.parametrize("at,M,N,K", [(False, 8192, 768, 2304), (False, 2048, 768, 768), (True, 768, 3072, 1024), (True, 256, 256, 128),
                                      (False, 512, 256, 128)])
@pytest.mark.parametrize("odd_rows", [False, True])
def test_gemm64_takes_either_tile(at, M, N, K, odd_rows):
    """Whatever tile the plan takes, also for output rows of 8 bytes' alignment (those stay with the 256 x 256 tiles)."""
    from llmctl.ops._lib import native

    a, b = _operands(at, M, N, K, 0)
    out = torch.full((M, N + 4), 3.0, device="cuda", dtype=torch.bfloat16)[:, :N] if odd_rows else torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
    native().gemm64_ex(a, b, out, at, True, False, 304)
    A, B = (a.t() if at else a).double(), b.double()
    ref, bound = A @ B, _bound(A, B, K, 16)
    assert bool(((out.double() - ref).abs() <= bound + 2.0**-8 * (ref.abs() + bound)).all())


@pytest.mark.parametrize("M,N,K,S,pad", [(256, 512, 256, 1, 8), (512, 640, 640, 2, 0), (768, 3072, 8192, 3, 0), (2304, 768, 1152, 4, 8)])
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("add", [False, True])
def test_column_sums_ride_along(M, N, K, S, pad, f32, add):
    """The product as without them, the sums of dy's columns beside it."""
    from llmctl.ops._lib import native

    dy, x = _operands(True, M, N, K, pad)
    dy = (dy.float() + 0.5).bfloat16()  # sums that do not cancel
    dt = torch.float32 if f32 else torch.bfloat16
    out, plain = torch.ones(M, N, device="cuda", dtype=dt), torch.ones(M, N, device="cuda", dtype=dt)
    db = torch.linspace(-1, 1, M, device="cuda").to(dt)
    ref = dy.double().sum(0) + (db.double() if add else 0.0)
    bound = (K + S + 1) * 2.0**-24 * dy.double().abs().sum(0)
    native().gemm_tall(dy, x, out, True, add, S, db, add)
    native().gemm_tall(dy, x, plain, True, add, S)
    assert torch.equal(out, plain)
    err = (db.double() - ref).abs()
    assert bool((err <= bound + (0 if f32 else 2.0**-8) * (ref.abs() + bound)).all())


@pytest.mark.parametrize("tokens,out,inn", [(1024, 768, 3072), (2048, 2304, 768), (4096, 4096, 4096), (1000, 768, 768), (1024, 768, 256)])
def test_linear_backward_with_sinks(tokens, out, inn):
    """Both gradients land in their flat views whichever kernel takes the weight's, and each is told of once."""
    from llmctl.exec.linear import GradSink, linear

    torch.manual_seed(1)
    w = torch.nn.Parameter((torch.randn(out, inn, device="cuda") * 0.02).bfloat16())
    b = torch.nn.Parameter(torch.zeros(out, device="cuda", dtype=torch.bfloat16))
    sink, told = GradSink(), []
    sink.callbacks.append(lambda p: told.append(p))
    for p in (w, b):
        p.grad = torch.full_like(p, float("nan"))
        sink.attach(p)
    x, dy = torch.randn(tokens, inn, device="cuda").bfloat16(), torch.randn(tokens, out, device="cuda").bfloat16()
    linear(x, w, b).backward(dy)
    assert len(told) == 2 and {id(p) for p in told} == {id(w), id(b)}
    linear(x, w, b).backward(dy)
    for p, ref in ((w, dy.double().t() @ x.double()), (b, dy.double().sum(0))):
        assert bool(((p.grad.double() - 2 * ref).abs() <= 2.0**-7 * 2 * ref.abs() + 1e-3 * ref.abs().max()).all())


@pytest.mark.parametrize("M,N,tokens", [(8200, 256, 3072), (8440, 512, 3200), (8320, 256, 3072)])
@pytest.mark.parametrize("f32", [False, True])
def test_weight_gradient_of_a_vocabulary(M, N, tokens, f32, monkeypatch):
    """Rows that fill no whole tile: both parts of the gradient, stored and added to."""
    import importlib

    from llmctl.exec.linear import _wgrad_whole, wgrad_into

    monkeypatch.setattr(importlib.import_module("llmctl.exec.linear"), "_whole_pays", lambda *a: True)  # (the rule takes larger ones)
    dy, x = _operands(True, M, N, tokens, 0)
    g = torch.full((M, N), float("nan"), device="cuda", dtype=torch.float32 if f32 else torch.bfloat16)
    assert f32 or _wgrad_whole(g, dy, x)
    A, B = dy.t().double(), x.double()
    ref, bound = A @ B, _bound(A, B, tokens, 16)
    wgrad_into(g, dy, x, False)
    first = g.double()
    # an fp32 gradient takes the library's product, rounded to bf16; each write of a bf16 one rounds once
    assert bool(((first - ref).abs() <= bound + 2.0**-8 * (ref.abs() + bound)).all())
    wgrad_into(g, dy, x, True)
    assert bool(((g.double() - first - ref).abs() <= bound + 2.0**-7 * (ref.abs() + first.abs() + bound)).all())


def test_adding_a_vocabularys_gradient_stays_off_mixed_adds():
    """Rows behind the whole tiles are added in fp32 by the product itself, not by an elementwise add of two types."""
    from torch.profiler import ProfilerActivity, profile

    from llmctl.exec.linear import _wgrad_whole, wgrad_into

    M, N, tokens = 8200, 2048, 4096
    dy, x = _operands(True, M, N, tokens, 0)
    g = torch.randn(M, N, device="cuda").bfloat16()
    assert _wgrad_whole(g, dy, x)
    before = g.double()
    with profile(activities=[ProfilerActivity.CPU]) as prof:
        wgrad_into(g, dy, x, True)
    assert "aten::add_" not in {e.key for e in prof.key_averages()}
    A, B = dy.t().double(), x.double()
    ref, bound = A @ B, _bound(A, B, tokens, 16)
    assert bool(((g.double() - before - ref).abs() <= bound + 2.0**-8 * (ref.abs() + before.abs() + bound)).all())


@pytest.mark.parametrize("K,S", [(257, 1), (300, 1), (319, 1), (383, 1), (385, 2), (513, 2), (640, 2), (1000, 3), (3912, 4), (8191, 12)])
@pytest.mark.parametrize("M,N,pad", [(256, 512, 0), (512, 640, 8)])
@pytest.mark.parametrize("bias", [False, True])
def test_any_number_of_tokens(K, S, M, N, pad, bias):
    """A weight gradient whose last K-tiles are part full: nothing of what lies behind the last token (NaN here) comes in."""
    from llmctl.ops._lib import native

    g = torch.Generator(device="cuda").manual_seed(K + N)
    full = [torch.full((K + 160, n + pad), float("nan"), device="cuda", dtype=torch.bfloat16) for n in (M, N)]
    dy, x = full[0][:K, :M], full[1][:K, :N]
    for t in (dy, x):
        t.copy_(torch.randn(t.shape, generator=g, device="cuda"))
    out = torch.full((M, N), float("nan"), device="cuda")
    db = torch.full((M,), float("nan"), device="cuda") if bias else None
    native().gemm_tall(dy, x, out, True, False, S, db, False)
    A, B = dy.t().double(), x.double()
    assert bool(((out.double() - A @ B).abs() <= _bound(A, B, K, S)).all())
    if bias:
        assert bool(((db.double() - A.sum(1)).abs() <= (K + S) * 2.0**-24 * A.abs().sum(1)).all())


@pytest.mark.parametrize("tokens,out,inn", [(3912, 768, 3072), (300, 2304, 768), (1111, 768, 256), (255, 768, 768), (2080, 4096, 4096)])
@pytest.mark.parametrize("f32", [False, True])
def test_weight_gradients_of_odd_batches(tokens, out, inn, f32):
    """Whichever kernel or library product takes them; each gradient stored once and added to once."""
    from llmctl.exec.linear import GradSink, linear

    torch.manual_seed(1)
    w = torch.nn.Parameter((torch.randn(out, inn, device="cuda") * 0.02).bfloat16())
    b = torch.nn.Parameter(torch.zeros(out, device="cuda", dtype=torch.bfloat16))
    sink = GradSink()
    for p in (w, b):
        p.main_grad = torch.full(p.shape, float("nan"), device="cuda", dtype=torch.float32 if f32 else torch.bfloat16)
        sink.attach(p)
    x, dy = torch.randn(tokens, inn, device="cuda").bfloat16(), torch.randn(tokens, out, device="cuda").bfloat16()
    for _ in range(2):
        linear(x, w, b).backward(dy)
    for p, ref in ((w, dy.double().t() @ x.double()), (b, dy.double().sum(0))):
        assert bool(((p.main_grad.double() - 2 * ref).abs() <= 2.0**-7 * 2 * ref.abs() + 1e-3 * ref.abs().max()).all())


def test_refusals_are_kept_by_size(monkeypatch):
    """Sizes that the 256 x 128 tiles leave to others are asked about once, not in every backward."""
    import importlib

    from llmctl.ops._lib import native

    L = importlib.import_module("llmctl.exec.linear")
    L._bias_rides.cache_clear()
    K, M, N = 300, 6144, 2048
    assert native().gemm64_wgrad_splits(M, N, K, True) == 0
    calls = []

    class Counting:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(native(), name)

    monkeypatch.setattr("llmctl.ops._lib.native", lambda: Counting())
    dy, x = torch.randn(K, M, device="cuda").bfloat16(), torch.randn(K, N, device="cuda").bfloat16()
    g, gb = torch.empty(M, N, device="cuda", dtype=torch.bfloat16), torch.empty(M, device="cuda", dtype=torch.bfloat16)
    for _ in range(3):
        assert not L.wgrad_bias_into(g, dy, x, False, gb, False)
    assert calls == ["gemm64_wgrad_splits"]


@pytest.mark.parametrize("M,N,K,ranges", [(2560, 2560, 16384, 0), (5120, 1280, 6144, 0), (6144, 2048, 16384, 0), (3072, 1024, 12288, 0), (1536, 2048, 8192, 0), (768, 3072, 8192, 3),
                                          (2304, 768, 8192, 4), (2048, 2048, 2048, 1), (1024, 4096, 6144, 2), (4096, 4096, 8192, 0)])
def test_sizes_of_the_rule(M, N, K, ranges):
    """Weight gradients on both sides of the line (``profiles/backward_tiles.txt``)."""
    from llmctl.ops._lib import native

    assert native().gemm64_wgrad_splits(M, N, K, True) == ranges


@pytest.mark.parametrize("T,O,I,S,pad", [(256, 256, 128, 1, 0), (257, 256, 640, 1, 8), (511, 512, 512, 1, 0), (640, 768, 512, 2, 8), (1000, 256, 768, 3, 0),
                                         (1326, 2304, 768, 1, 0), (8192, 768, 512, 5, 0)])  # data gradients' last rows, either kind of workgroup first
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("add", [False, True])
@pytest.mark.parametrize("bias", [False, True])
def test_both_gradients_in_one_launch(T, O, I, S, pad, f32, add, bias):
    from llmctl.ops._lib import native

    if bias and I < 512:
        pytest.skip("column sums ride from 512 inputs on")
    g = torch.Generator(device="cuda").manual_seed(T + O + I)
    rows = lambda n, c: torch.randn(n, c + pad, generator=g, device="cuda").bfloat16()[:, :c]
    dy, w, x = rows(T, O), rows(O, I), rows(T, I)
    dt = torch.float32 if f32 else torch.bfloat16
    dx = torch.full((T + 2, I), 3.0, device="cuda", dtype=torch.bfloat16)
    gw, gb = (torch.full(s, 2.0 if add else float("nan"), device="cuda", dtype=dt) for s in ((O, I), (O,)))
    native().gemm_tall_back(dy, w, dx[:T], x, gw, add, S, gb if bias else None, add)
    D, W, X = dy.double(), w.double(), x.double()
    old = 2.0 if add else 0.0
    for out, ref, mag, n, half in ((dx[:T], D @ W, D.abs() @ W.abs(), O, True), (gw, D.t() @ X + old, D.t().abs() @ X.abs(), T, not f32),
                                   *([(gb, D.sum(0) + old, D.abs().sum(0), T, not f32)] if bias else [])):
        bound = (n + S + 1) * 2.0**-24 * mag + 2.0**-23 * ref.abs()
        if half:  # one rounding of the fp32 result
            bound = bound + 2.0**-8 * (ref.abs() + bound)
        assert bool(((out.double() - ref).abs() <= bound).all())
    assert bool((dx[T:] == 3.0).all())


@pytest.mark.parametrize("tokens,out,inn,bias", [(8192, 768, 768, True), (1326, 2304, 768, True), (640, 768, 3072, False)])
def test_layers_take_the_one_launch(tokens, out, inn, bias, monkeypatch):
    import importlib

    L = importlib.import_module("llmctl.exec.linear")
    calls, back = [], L.tall_back
    monkeypatch.setattr(L, "tall_back", lambda *a: calls.append(back(*a)) or calls[-1])
    sink = L.GradSink()
    w = torch.nn.Parameter(torch.randn(out, inn, device="cuda", dtype=torch.bfloat16) * 0.05)
    b = torch.nn.Parameter(torch.zeros(out, device="cuda", dtype=torch.bfloat16)) if bias else None
    for p in (w, b) if bias else (w,):
        p.grad = torch.full_like(p, float("nan"))
        sink.attach(p)
    x = torch.randn(tokens, inn, device="cuda", dtype=torch.bfloat16).requires_grad_()
    dy = torch.randn(tokens, out, device="cuda", dtype=torch.bfloat16)
    L.linear(x, w, b).backward(dy)
    assert len(calls) == 1 and calls[0] is not None
    D = dy.double()
    pairs = [(x.grad, D @ w.detach().double()), (w.grad, D.t() @ x.detach().double())] + ([(b.grad, D.sum(0))] if bias else [])
    for got, ref in pairs:  # bf16 of fp32 sums: 2^-9 an entry at most, 0.0017 of the norm
        assert float((got.double() - ref).norm() / ref.norm()) < 2.0**-9


def test_the_one_launch_is_taken_where_it_is_faster():
    """The rule against the times that its figures are from."""
    import re
    from pathlib import Path

    from llmctl.ops._lib import native

    picks = []
    for line in (Path(__file__).resolve().parents[2] / "profiles" / "backward_pairs.txt").read_text().splitlines():
        if m := re.match(r"(\d+) (\d+) (\d+) (\d) \| ([\d.]+) \| (.*)$", line):
            T, O, I, bias = map(int, m.groups()[:4])
            one = {int(s): float(t) for s, t in re.findall(r"(\d+):([\d.]+)", m[6])}
            ranges = native().gemm64_back_splits(T, O, I, bool(bias))
            if ranges in one:
                picks.append((float(m[5]), one[ranges]))
    assert len(picks) >= 250 and all(one <= 1.02 * two for two, one in picks)
    assert sum(one for _, one in picks) < 0.8 * sum(two for two, _ in picks)

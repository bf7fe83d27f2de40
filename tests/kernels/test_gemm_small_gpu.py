"""Products of few entries (csrc/gemm_small.hip) against 64 bits, and the training linear on them."""

import importlib

import pytest
import torch

from llmctl.ops._lib import native

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]
L = importlib.import_module("llmctl.exec.linear")


def _rows(R, C, pad, dtype=torch.bfloat16):
    """[R, C] inside a larger tensor that is NaN around it."""
    t = torch.full((R + 1, C + pad), float("nan"), device="cuda", dtype=dtype)
    t[:R, :C] = torch.randn(R, C, device="cuda").to(dtype)
    return t[:R, :C]


def _check(got, want, mag, K):
    # the output's rounding, and K + 8 fp32 additions of products that are exact
    half = 2.0 ** -8 if got.dtype == torch.bfloat16 else 2.0 ** -23
    assert ((got.double() - want).abs() <= half * want.abs() + (K + 16) * 2.0 ** -24 * mag + 1e-30).all()


@pytest.mark.parametrize("layout, M, N, K", [
    ("fwd", 1, 8, 8), ("fwd", 33, 40, 72), ("fwd", 64, 64, 256), ("fwd", 100, 712, 704), ("fwd", 31, 32, 1024),
    ("dgrad", 1, 8, 8), ("dgrad", 33, 40, 72), ("dgrad", 65, 256, 1408), ("dgrad", 100, 712, 1016), ("dgrad", 256, 24, 3072),
    ("wgrad", 8, 8, 1), ("wgrad", 40, 72, 33), ("wgrad", 264, 256, 100), ("wgrad", 64, 32, 4096), ("wgrad", 768, 768, 71), ("wgrad", 1032, 568, 129)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_product_against_64_bits(layout, M, N, K, dtype):
    torch.manual_seed(M + N + K)
    at, bt = layout == "wgrad", layout != "fwd"
    a = _rows(*((K, M) if at else (M, K)), 8)
    b = _rows(*((K, N) if bt else (N, K)), 16)
    ad, bd = (a.t() if at else a).double(), (b if bt else b.t()).double()
    want, mag = ad @ bd, ad.abs() @ bd.abs()
    out = _rows(M, N, 8, dtype)
    keep = out.double()
    native().gemm_small(a, b, out, at, bt, False)
    _check(out, want, mag, K)
    out.copy_(keep)
    if at:
        sums = torch.randn(M, device="cuda").to(dtype)
        before = sums.double()
        native().gemm_small(a, b, out, True, True, True, None, sums, True)
        _check(sums, before + ad.sum(1), before.abs() + ad.abs().sum(1), K)
        native().gemm_small(a, b, out, True, True, False, None, sums, False)
        _check(sums, ad.sum(1), ad.abs().sum(1), K)
    else:
        bias = torch.randn(N, device="cuda").bfloat16()
        native().gemm_small(a, b, out, at, bt, True, bias)
        _check(out, want + keep + bias.double(), mag + keep.abs() + bias.double().abs(), K)


@pytest.mark.parametrize("T, O, I, bias", [(96, 256, 704, False), (256, 768, 256, True), (130, 2304, 768, True), (200, 64, 64, True)])
def test_training_linear(T, O, I, bias, monkeypatch):
    """Sinked gradients, stored and added to, and ordinary ones: as 64 bits give them, on ``gemm_small``."""
    torch.manual_seed(T)
    x = torch.randn(2, T // 2, I, device="cuda").bfloat16().requires_grad_()
    w = torch.nn.Parameter((torch.randn(O, I, device="cuda") * I ** -0.5).bfloat16())
    b = torch.nn.Parameter(torch.randn(O, device="cuda").bfloat16()) if bias else None
    dy = torch.randn(2, T // 2, O, device="cuda").bfloat16()
    assert L.small_pays("wgrad", O, I, T, bias)
    xd, wd, dyd = (t.detach().double() for t in (x, w, dy))
    y = L.linear(x, w, b)
    want = xd @ wd.t() + (b.detach().double() if bias else 0)
    _check(y, want, xd.abs() @ wd.abs().t() + 4, I)
    y.backward(dy)
    _check(x.grad, dyd @ wd, dyd.abs() @ wd.abs(), O)
    d2, x2 = dyd.flatten(0, 1), xd.flatten(0, 1)
    _check(w.grad, d2.t() @ x2, d2.abs().t() @ x2.abs(), T)
    sink = L.GradSink()
    for p in (w, b):
        if p is not None:
            p.grad = torch.full_like(p, float("nan"))  # the first write stores
            sink.attach(p)
    calls, back = [], L.small_back
    monkeypatch.setattr(L, "small_back", lambda *a: calls.append(back(*a)) or calls[-1])
    for n in (1, 2):
        x.grad = None
        L.linear(x, w, b).backward(dy)
        assert (calls[-1] is not None) == (O * I < 1024 * 513)  # both products in one launch
        _check(x.grad, dyd @ wd, dyd.abs() @ wd.abs(), O)
        want, mag = n * (d2.t() @ x2), 3 * n * (d2.abs().t() @ x2.abs())
        assert ((w.grad.double() - want).abs() <= n * 2.0 ** -8 * want.abs() + 2.0 ** -8 * (n - 1) * want.abs() + (T + 16) * 2.0 ** -24 * mag).all()
        if bias:
            want, mag = n * d2.sum(0), 3 * n * d2.abs().sum(0)
            assert ((b.grad.double() - want).abs() <= 2 * n * 2.0 ** -8 * want.abs() + (T + 16) * 2.0 ** -24 * mag).all()


def test_second_gradients_and_autocast_stay_with_the_library():
    x = torch.randn(64, 64, device="cuda").bfloat16().requires_grad_()
    w = torch.randn(64, 64, device="cuda").bfloat16()
    y = L.linear(x, w)
    dy = torch.randn_like(y).requires_grad_()
    (dx,) = torch.autograd.grad(y, x, dy, create_graph=True)
    (back,) = torch.autograd.grad(dx.float().sum(), dy)
    assert torch.allclose(back.float(), w.float().sum(1).expand_as(back), atol=0.5)
    with torch.autocast("cuda", dtype=torch.float16):
        assert L.linear(x.detach(), w).dtype == torch.float16


@pytest.mark.parametrize("bad", ["odd columns", "rows that are not aligned", "shapes", "type"])
def test_refused_on_the_host(bad):
    a, b = torch.randn(16, 64, device="cuda").bfloat16(), torch.randn(32, 64, device="cuda").bfloat16()
    out = torch.empty(16, 32, device="cuda").bfloat16()
    if bad == "odd columns":
        b, out = b[:30], out[:, :30]
    elif bad == "rows that are not aligned":
        a = torch.randn(16, 68, device="cuda").bfloat16()[:, 4:]
    elif bad == "shapes":
        out = out[:8]
    else:
        a = a.float()
    with pytest.raises(RuntimeError, match="gemm_small"):
        native().gemm_small(a, b, out, False, False, False)


@pytest.mark.parametrize("M, N, K, act", [(33, 40, 72, None), (100, 2304, 768, None), (100, 3072, 768, "gelu"), (640, 2304, 768, "gelu"), (700, 712, 256, None)])
def test_a_prompts_products(M, N, K, act, monkeypatch):
    """Serving's products of more rows than a decode step's: one launch, activation included, against 64 bits."""
    from llmctl import ops

    torch.manual_seed(M)
    x, w = torch.randn(M, K, device="cuda").bfloat16(), (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    b = torch.randn(N, device="cuda").bfloat16()
    assert L.small_pays("eager", M, N, K)
    calls, small = [], L.small_linear
    monkeypatch.setattr(L, "small_linear", lambda *a: calls.append(small(*a)) or calls[-1])
    with torch.inference_mode():
        got = ops.decode_linear(x, w, b, act=act)
    assert calls and calls[0] is got
    want = x.double() @ w.double().t() + b.double()
    mag = x.double().abs() @ w.double().abs().t() + b.double().abs()
    if act is None:
        _check(got, want, mag, K)
        return
    want = 0.5 * want * (1 + torch.tanh(0.7978845608028654 * (want + 0.044715 * want ** 3)))
    # a gelu's slope is at most 1.13; its own fp32 steps: a few roundings of values up to |x| (1 + tanh)
    assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1.13 * (K + 16) * 2.0 ** -24 * mag + 2.0 ** -20 * mag).all()


def test_a_transformed_bias_stays_with_the_library():
    """A bias that vmap runs over, old or new, or of a class of its own: as the library takes them."""
    x, w, b = (torch.randn(*s, device="cuda").bfloat16() for s in ((64, 256), (256, 256), (3, 256)))

    class Own(torch.Tensor):
        pass

    with torch.no_grad():
        assert L.small_linear(x, w, b[0], "eager") is not None
        for over in (torch.vmap, torch._vmap_internals._vmap):
            assert torch.equal(over(lambda r: L.forward_linear(x, w, r))(b), over(lambda r: torch.nn.functional.linear(x, w, r))(b))
        got = L.forward_linear(x, w, b[0].as_subclass(Own))
        assert type(got) is Own and torch.equal(got.as_subclass(torch.Tensor), torch.nn.functional.linear(x, w, b[0]))


def test_traced_and_counted_products_stay_with_the_library():
    """Modes that see the library's calls, and traces, which are run with other sizes, see the products as they ever did, forward and backward."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.utils.flop_counter import FlopCounterMode

    x, w, b = (torch.randn(*s, device="cuda").bfloat16() for s in ((65, 256), (256, 256), (256,)))  # (of 65 tokens the library had all three products)
    longer = torch.randn(101, 256, device="cuda").bfloat16()
    assert L.small_linear(x, w, b, "eager") is not None

    def step(x):
        x, v = x.detach().requires_grad_(), w.detach().requires_grad_()
        return torch.autograd.grad(L.linear(x, v, b), (x, v), torch.ones(x.shape[0], 256, device="cuda", dtype=x.dtype))

    with torch.no_grad():
        for traced in (make_fx(lambda x: L.forward_linear(x, w, b), tracing_mode="symbolic", _allow_non_fake_inputs=True)(x),
                       make_fx(lambda x: L.forward_linear(x, w, b))(x), torch.jit.trace(lambda x: L.forward_linear(x, w, b), x, check_trace=False)):
            assert torch.equal(traced(longer), torch.nn.functional.linear(longer, w, b))

    def back(x):
        x = x.detach().requires_grad_()
        return torch.autograd.grad(L.linear(x, w, b).sum(), x)[0]

    traced = make_fx(back, tracing_mode="symbolic", _allow_non_fake_inputs=True)(x)
    got, want = traced(longer).float(), back(longer).float()
    assert float((got - want).norm()) <= 2.0 ** -7 * float(want.norm())  # each rounds its sums to bf16 once
    with FlopCounterMode(display=False) as count:
        step(x)
    assert count.get_total_flops() == 3 * 2 * 65 * 256 * 256


def test_a_traced_loss_takes_other_lengths():
    from llmctl import ops

    short, long = (torch.randn(T, 64, device="cuda").bfloat16() for T in (32, 32769))
    traced = torch.jit.trace(lambda x, y: ops.cross_entropy(x, y, reduction_denom=16.0), (short, torch.zeros(32, dtype=torch.int64, device="cuda")), check_trace=False)
    y = torch.zeros(32769, dtype=torch.int64, device="cuda")
    want = float(torch.nn.functional.cross_entropy(long.double(), y, reduction="sum")) / 16
    assert abs(float(traced(long, y)) - want) <= 64 * 2.0 ** -24 * want


@pytest.mark.parametrize("shape", [(64, 64), (2, 40, 64)])
def test_no_outputs(shape):
    """A weight without rows: an empty result, as from the library."""
    from llmctl import ops

    x, w, b = (torch.randn(*s, device="cuda").bfloat16() for s in (shape, (0, 64), (0,)))
    with torch.no_grad():
        assert L.forward_linear(x, w, b).shape == (*shape[:-1], 0)
        assert ops.decode_linear(x, w, b).shape == (*shape[:-1], 0)


@pytest.mark.parametrize("M,N,K,own", [(33, 8, 8, True), (200, 1024, 64, True), (2048, 1024, 72, True), (2049, 1024, 64, False), (40, 32000, 64, True), (64, 512, 68, False), (64, 8192, 2048, False)])
def test_prompts_with_fp32_results(M, N, K, own):
    """Rows cut from wider ones; sums of K exact products in fp32, in any order."""
    from llmctl.exec.linear import small_linear_f32
    from llmctl.ops import hybrid as hops

    g = torch.Generator(device="cuda").manual_seed(M + N)
    x, w = torch.randn(M, K + 24, generator=g, device="cuda").bfloat16()[:, 8:8 + K], torch.randn(N, K, generator=g, device="cuda").bfloat16()
    X, W = x.double(), w.double()
    y = small_linear_f32(x, w)
    assert (y is not None) == (own and K % 8 == 0)
    for got in (y, hops.linear_f32(x, w)):
        assert got is None or (got.dtype == torch.float32 and bool(((got.double() - X @ W.t()).abs() <= K * 2.0**-23 * (X.abs() @ W.abs().t())).all()))
    p = w.clone().requires_grad_()
    assert small_linear_f32(x, p) is None and small_linear_f32(x.float(), w.float()) is None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert small_linear_f32(x, w) is None

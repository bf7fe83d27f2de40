"""An embedding's gradient: runs of one id within and across the chunks, token counts around them and past one fill of LDS, and the sink that it goes to."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ids(kind, T, V, g):
    if kind == "same":
        return torch.full((T,), V - 1, dtype=torch.int64, device="cuda")
    if kind == "distinct":
        return torch.randperm(max(T, V), generator=g, device="cuda")[:T] % V
    if kind == "skewed":  # as words are: a few ids take most of the places
        return (torch.rand(T, generator=g, device="cuda") ** 4 * V).long().clamp_(0, V - 1)
    return torch.randint(0, V, (T,), generator=g, device="cuda")


@pytest.mark.parametrize("T,H,V", [(1, 8, 3), (15, 8, 40), (16, 512, 5), (17, 520, 5), (33, 768, 64), (300, 64, 7), (8, 8, 3), (9, 512, 4), (2048, 768, 1000), (16385, 16, 300)])
@pytest.mark.parametrize("kind", ["same", "distinct", "skewed", "any"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("add", [False, True])
def test_sums(T, H, V, kind, dtype, add):
    from llmctl import ops

    g = torch.Generator(device="cuda").manual_seed(T * H + V)
    ids = _ids(kind, T, V, g)
    dy = torch.randn(T, H + 8, generator=g, device="cuda").bfloat16()[:, :H]
    out = torch.randn(V, H, generator=g, device="cuda").to(dtype)
    ref = out.double() if add else torch.zeros(V, H, device="cuda", dtype=torch.float64)
    mag = ref.abs()
    ref.index_add_(0, ids, dy.double())
    mag.index_add_(0, ids, dy.double().abs())
    n = torch.bincount(ids, minlength=V).max().item()
    assert ops.embed_grad_ok(ids, dy, out)
    again = out.clone()
    ops.embed_grad_(ids, dy, out, add)
    ops.embed_grad_(ids, dy, again, add)
    assert torch.equal(out, again)
    bound = (n + 1) * 2.0**-24 * mag  # fp32 sums of n rows and the old value, in any order
    if dtype == torch.bfloat16:
        bound = bound + 2.0**-8 * (ref.abs() + bound)
    assert bool(((out.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("tied", [False, True])
def test_sink(tied):
    """Two backwards into one flat gradient: zeros where no token was, callbacks once a backward, tied weights after both writes."""
    from llmctl.exec.linear import GradSink, embedding, linear

    torch.manual_seed(0)
    V, H, T = 384, 256, 256
    w = torch.nn.Parameter(torch.randn(V, H, device="cuda").bfloat16())
    flat = torch.full((V, H), float("nan"), device="cuda", dtype=torch.bfloat16)
    sink, told = GradSink(), []
    sink.callbacks.append(lambda p: told.append(p))
    sink.attach(w, 2 if tied else 1)
    w.grad = flat
    ref = torch.zeros(V, H, device="cuda", dtype=torch.float64)
    for step in range(2):
        ids = torch.randint(0, V, (T,), device="cuda")
        x = embedding(ids, w)
        y = linear(x, w) if tied else x
        dy = torch.randn_like(y)
        y.backward(dy)
        assert len(told) == step + 1
        wd = w.detach().double().requires_grad_(True)
        xd = wd[ids]
        (xd @ wd.t() if tied else xd).backward(dy.double())
        ref += wd.grad
    assert w.grad is flat
    # tied: x's gradient is rounded to bf16 once before the rows are summed; each write rounds the flat gradient once more
    assert (flat.double() - ref).abs().max() <= 6 * 2.0**-8 * ref.abs().max()


@pytest.mark.parametrize("T,H,V", [(20000, 8, 256), (24576, 64, 300)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tokens", ["few", "all"])
def test_many_tokens_of_narrow_rows(T, H, V, dtype, tokens, monkeypatch):
    """The library's sums past the rule's line: two backwards, held in fp32 up to the flat gradient as the kernel holds them."""
    from llmctl import ops
    from llmctl.exec.linear import GradSink, embedding

    assert not ops.embed_grad_pays(T, H, V) or T == 20000
    monkeypatch.setattr(ops, "embed_grad_pays", lambda *a: False)
    g = torch.Generator(device="cuda").manual_seed(T)
    w = torch.nn.Parameter(torch.randn(V, H, generator=g, device="cuda").bfloat16())
    flat = torch.full((V, H), float("nan"), device="cuda", dtype=dtype)
    sink = GradSink()
    sink.attach(w)
    if dtype == torch.float32:
        w.main_grad = flat
    else:
        w.grad = flat
    ref, mag, err = torch.zeros(V, H, device="cuda", dtype=torch.float64), torch.zeros(V, H, device="cuda", dtype=torch.float64), 0.0
    for _ in range(2):
        ids = torch.randint(0, V if tokens == "all" else 3, (T,), generator=g, device="cuda")
        dy = torch.randn(T, H, generator=g, device="cuda").bfloat16()
        embedding(ids, w).backward(dy)
        ref.index_add_(0, ids, dy.double())
        mag.index_add_(0, ids, dy.double().abs())
        # fp32 sums, and for a bf16 gradient the rounding of each write of it
        err = err + (T + 1) * 2.0**-24 * mag + (2.0**-8 * ref.abs() if dtype == torch.bfloat16 else 0.0)
    assert bool(((flat.double() - ref).abs() <= err * (1 + 2.0**-7) + 1e-30).all())


@pytest.mark.parametrize("T", [2, 63, 64, 65, 255, 257, 384, 385])
@pytest.mark.parametrize("kind", ["same", "distinct", "skewed"])
@pytest.mark.parametrize("H", [8, 520])
def test_few_tokens(T, kind, H):
    """The one launch of few tokens and the three of more: places at the edges of a wave's 64 and of the line between them."""
    from llmctl import ops

    V = 700
    g = torch.Generator(device="cuda").manual_seed(T + H)
    ids = _ids(kind, T, V, g)
    dy = torch.randn(T, H, generator=g, device="cuda").bfloat16()
    out = torch.randn(V, H, generator=g, device="cuda")
    ref = out.double()
    mag = ref.abs()
    ref.index_add_(0, ids, dy.double())
    mag.index_add_(0, ids, dy.double().abs())
    ops.embed_grad_(ids, dy, out, True)
    n = torch.bincount(ids, minlength=V).max().item()
    assert bool(((out.double() - ref).abs() <= (n + 1) * 2.0 ** -24 * mag).all())

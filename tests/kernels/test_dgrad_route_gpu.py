"""The data gradient's routes (knob ``dgrad64`` = auto): the in-house kernel where the shape fits up to 16384 rows, for its whole tiles
where a large weight's rows do not, else W as it is, or W^T copies for large weights and many rows; each against fp32 on the same
operands."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,inn,out,route", [
    (256, 256, 128, "gemm64"), (300, 256, 128, "plain"), (256, 264, 128, "plain"), (16384, 256, 128, "gemm64"), (16640, 256, 128, "plain"),
    (8192, 4096, 4096, "gemm64"), (257, 4096, 4096, "plain"), (1535, 4096, 4096, "plain"), (1537, 4096, 4096, "split"), (8200, 4096, 4096, "split"), (16400, 4096, 4096, "split"),
    (16640, 4096, 4096, "copy"), (8200, 4096, 4104, "copy"), (8184, 4096, 4104, "plain"), (8200, 4096, 4088, "plain")])
def test_data_gradient_routes(T, inn, out, route):
    from llmctl.config.knobs import override
    from llmctl.exec.linear import GradSink, dgrad64_ok, dgrad64_part, linear

    g = torch.Generator(device="cuda").manual_seed(T)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    with override(dgrad64="auto"):
        x, w, dy = r(T, inn).requires_grad_(), torch.nn.Parameter(r(out, inn)), r(T, out)
        w.grad = torch.zeros_like(w)
        GradSink().attach(w)
        linear(x, w).backward(dy)
        assert dgrad64_ok(dy, w) == (route == "gemm64") and bool(dgrad64_part(dy, w)) == (route == "split")
        assert (getattr(w, "_llmctl_wt", None) is not None) == (route == "copy")
    want = dy.float() @ w.detach().float()
    # one rounding to bf16 over fp32 sums of ``out`` terms
    assert ((x.grad.float() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -14 * out ** 0.5).all()


@pytest.mark.parametrize("T,inn,out,gemm64", [(16384, 256, 128, True), (16640, 256, 128, True), (16640, 4096, 4096, True), (16700, 4096, 4096, False), (16640, 4096, 4104, False)])
def test_a_tied_weight_keeps_no_copy(T, inn, out, gemm64, monkeypatch):
    """The embedding that is the output projection too: gemm64 beyond 16384 rows as well, else W as it is."""
    import importlib

    from llmctl.config.knobs import override

    L = importlib.import_module("llmctl.exec.linear")
    rows, whole = [], L.dgrad64
    monkeypatch.setattr(L, "dgrad64", lambda dy, w, r=None: rows.append(r) or whole(dy, w, r))
    g = torch.Generator(device="cuda").manual_seed(T)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    with override(dgrad64="auto"):
        x, w, dy = r(T, inn).requires_grad_(), torch.nn.Parameter(r(out, inn)), r(T, out)
        w.grad = torch.zeros_like(w)
        L.GradSink().attach(w, 2)
        L.linear(x, w).backward(dy)
    assert getattr(w, "_llmctl_wt", None) is None and rows == ([None] if gemm64 else [])
    want = dy.float() @ w.detach().float()
    assert ((x.grad.float() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -14 * out ** 0.5).all()

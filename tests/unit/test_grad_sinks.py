"""Gradients of norm vectors and biases that go through a sink (``llmctl.exec.linear.GradSink``) while others are frozen."""

import dataclasses

import pytest
import torch

from llmctl import ops
from llmctl.exec.linear import GradSink, linear
from llmctl.models import get_model_config
from llmctl.runtime.engine import TrainingConfig, TrainingEngine
from llmctl.comms.overlap import GradSyncEngine  # (after the engine, which imports it)
from llmctl.runtime.flat import FlatParameters, grad_view


def frozen_vector_gradients(device: str, kind: str, frozen: str, before: bool, grad_dtype: torch.dtype):
    """Two steps of two micro-steps of one norm (``kind``) with the vectors named in ``frozen`` frozen, before or after the flat
    buffers are made: ([gradient of w, of b] through sinks, the same by autograd without any), fp32, None where frozen."""
    H, g = 64, torch.Generator().manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g).bfloat16().to(device)
    xs, rs, dys = ([r(7, H) for _ in range(2)] for _ in range(3))
    vecs = [r(H), r(H)]
    ln = "layernorm" in kind

    def backward(w, b, i):
        x, args = xs[i].clone().requires_grad_(), (w, b) if ln else (w,)
        if kind.startswith("add_"):
            y, res = getattr(ops, kind)(x, rs[i], *args)
            ((y.float() * dys[i].float()).sum() + (res.float() * dys[1 - i].float()).sum()).backward()
        else:
            (getattr(ops, kind)(x, *args).float() * dys[i].float()).sum().backward()

    def freeze(w, b):
        for n, p in (("w", w), ("b", b)):
            if n in frozen:
                p.requires_grad_(False)

    w, b = (torch.nn.Parameter(v.clone()) for v in vecs)
    other = torch.nn.Parameter(torch.zeros(8, dtype=torch.bfloat16, device=device))  # (there is always something to train)
    if before:
        freeze(w, b)
    flat = FlatParameters([("w", w), ("b", b), ("other", other)], bucket_numel=1 << 20, grad_dtype=grad_dtype)
    flat.install_sinks(GradSink(), lambda n, p: n != "other")
    if not before:
        flat.zero_grad()
        backward(w, b, 0)  # a step with everything trainable, whose gradients must not show later
        freeze(w, b)
    for _ in range(2):
        flat.zero_grad()
        for i in range(2):
            backward(w, b, i)
        flat.settle_grads()
    got = [grad_view(p).float() if p.requires_grad and (ln or n == "w") else None for n, p in (("w", w), ("b", b))]
    pw, pb = (torch.nn.Parameter(v.clone()) for v in vecs)
    freeze(pw, pb)
    want = [None, None]
    for i in range(2):
        pw.grad = pb.grad = None
        backward(pw, pb, i)
        for k, p in enumerate((pw, pb)):
            if p.grad is not None:
                want[k] = p.grad.float() + (0 if want[k] is None else want[k])
    return got, want


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("frozen", ["w", "b", "wb"])
@pytest.mark.parametrize("before", [True, False])
@pytest.mark.parametrize("kind", ["layernorm", "add_layernorm", "rmsnorm", "add_rmsnorm"])
@pytest.mark.parametrize("grad_dtype", [torch.bfloat16, torch.float32])
def test_a_frozen_vector_leaves_the_other_gradient_right(kind, frozen, before, grad_dtype, device):
    got, want = frozen_vector_gradients(device, kind, frozen, before, grad_dtype)
    for g, w in zip(got, want):
        assert (g is None) == (w is None)
        # the same sums; bf16 gradients are rounded per micro-step, twice in two steps of two
        assert g is None or (g - w).abs().max() <= 2.0 ** -6 * w.abs().max()


def _engine():
    cfg = TrainingConfig(model_name_or_path="gpt2-125m", batch_size=1, seq_len=16, device="cpu", log_level="warning", learning_rate=0.0,
                         weight_decay=0.0, max_steps=10, mixed_precision="fp32")
    mc = dataclasses.replace(get_model_config("gpt2-125m"), layers=1, hidden=64, heads=4, kv_heads=4, ffn=128, vocab_size=64)
    return TrainingEngine(cfg, mc)


@pytest.mark.parametrize("name", ["attn_norm_b", "attn_norm_w", "bo"])
def test_gradients_do_not_grow_over_steps_of_the_engine(name):
    torch.manual_seed(0)
    eng = _engine()
    getattr(eng.model.layers[0], name).requires_grad_(False)
    ids = torch.randint(0, 64, (1, 17))
    seen = []
    for _ in range(3):  # learning rate 0, one batch: the same gradients every step
        eng.train_step([(ids[:, :-1].contiguous(), ids[:, 1:].contiguous())])
        seen.append({eng.flat.names[id(p)]: grad_view(p).clone() for p in eng.flat.params})
    assert any("norm" in n and g.abs().max() > 0 for n, g in seen[0].items())
    for later in seen[1:]:
        for n, g in later.items():
            assert torch.equal(g, seen[0][n]), n
    assert seen[0]["layers.0." + name].abs().max() == 0


def test_a_vector_left_out_of_a_step_has_no_old_gradient():
    w, b = (torch.nn.Parameter(torch.ones(8)) for _ in range(2))
    flat = FlatParameters([("w", w), ("b", b)], bucket_numel=1 << 20)
    flat.install_sinks(GradSink(), lambda n, p: True)
    sync = GradSyncEngine(flat)
    x = torch.randn(4, 8)
    flat.zero_grad()
    ops.layernorm(x, w, b).sum().backward()
    sync.finish()
    assert b.grad.abs().max() > 0
    flat.zero_grad()
    b.requires_grad_(False)  # after zero_grad: nothing writes it this time
    ops.layernorm(x, w, b).sum().backward()
    sync.finish()
    assert b.grad.abs().max() == 0
    flat.zero_grad()
    b.requires_grad_(True)
    ops.layernorm(x, w, b).sum().backward()
    assert torch.equal(b.grad, torch.full((8,), 4.0))


@pytest.mark.parametrize("frozen", [0, 1])
def test_buckets_are_issued_during_backward(frozen):
    """A frozen vector outside the flat buffers does not hold back the bucket of its partner."""
    w, b = (torch.nn.Parameter(torch.ones(8)) for _ in range(2))
    (w, b)[frozen].requires_grad_(False)
    m = torch.nn.Parameter(torch.randn(8, 8))
    flat = FlatParameters([("w", w), ("b", b), ("m", m)], bucket_numel=1)
    flat.install_sinks(GradSink(), lambda n, p: True)
    sync, issued = GradSyncEngine(flat), []
    sync._launch = lambda bucket: issued.append([flat.names[id(p)] for p in bucket.params])
    flat.zero_grad()
    linear(ops.layernorm(torch.randn(4, 8), w, b), m).sum().backward()
    assert sorted(sum(issued, [])) == sorted(["m", "wb"[1 - frozen]])
    n = len(issued)
    sync.finish()
    assert len(issued) == n


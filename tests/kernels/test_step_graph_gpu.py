"""Replayed training steps (``llmctl.runtime.step_graph``) against eager ones, and the steps that must not be replayed."""

import ctypes
import dataclasses
import gc
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def engine(model="tiny", layers=2, knob=True, tokens=(2, 128), heads=None, cls=None, **kw):
    from llmctl.models import get_model_config
    from llmctl.runtime.engine import TrainingConfig, TrainingEngine

    cfg = dataclasses.replace(get_model_config(model), layers=layers, **({} if heads is None else dict(heads=heads, kv_heads=heads)))
    return (cls or TrainingEngine)(TrainingConfig(model_name_or_path=model, batch_size=tokens[0], seq_len=tokens[1], device="cuda", log_level="warning",
                                         learning_rate=1e-3, max_steps=50, seed=3, perf_knobs={"step_graph": knob}, **kw), cfg)


def batch(eng, g, b, s):
    t = torch.randint(0, eng.model_config.vocab_size, (b, s + 1), generator=g).to("cuda")
    return t[:, :-1], t[:, 1:]  # (rows of another tensor, as a loader's are)


# (the last three: heads of 128, whose dK/dV kernel clears its counters with a launch of its own; a loss over 16384 tokens, one launch too; and one over more than 32768,
# which the library sums with a memset, so that its steps stay eager)
@pytest.mark.parametrize("model,layers,sizes,heads,recorded", [
    ("tiny", 2, [(2, 128)], None, 1), ("tiny", 2, [(1, 65), (3, 100), (8, 512)], None, 3), ("gpt2-125m", 2, [(2, 64), (1, 333)], None, 2),
    ("tiny", 2, [(2, 128), (5, 256)], 2, 2), ("tiny", 1, [(32, 512)], None, 1), ("tiny", 1, [(65, 512)], None, 0)])
def test_replayed_steps_match_eager_ones(native_lib, model, layers, sizes, heads, recorded):
    """Losses, norms, gradients and states over many steps of alternating shapes, other work on the device between them.  Both sides run the same
    kernels; what differs from run to run is the order of the clip norm's atomics (and a library product's partial sums), which moves the weights by
    rounding: the bound is four times the spread of two eager runs, or rounding of bf16 weights (2^-9) where they happen to agree."""
    from llmctl.runtime.step_graph import pays

    def run(knob):
        eng, g, out = engine(model, layers, knob, heads=heads), torch.Generator().manual_seed(1), []
        for step in range(5):
            for b, s in sizes:
                r = eng.train_step([batch(eng, g, b, s)])
                keep = torch.full((1 << 20,), float(step), device="cuda")  # memory that a stale pointer would hit
                out += [r["loss"], r["grad_norm"], keep.sum() * 0]
        torch.cuda.synchronize()
        assert len(eng.step_graphs.table) == (recorded if knob else 0)
        assert all(pays(eng.flat.numel, b * s, layers) for b, s in sizes)  # (none is left eager for its length)
        return torch.stack([o.float().reshape(()) for o in out]), eng.flat.grad.float(), eng.optimizer.master, eng.optimizer.exp_avg

    a, b, c = run(True), run(False), run(False)
    for x, y, z in zip(a, b, c):
        assert torch.isfinite(x).all()
        assert (x - y).norm() <= max(4 * (y - z).norm().item(), 2.0 ** -9 * y.norm().item())


def test_recorded_beside_a_serving_graph(native_lib):
    """A graph recorded in inference mode that is still there owns the generator's tensors: they are not written outside that mode."""
    served = torch.cuda.CUDAGraph()
    t = torch.zeros(8, device="cuda")
    with torch.inference_mode():
        t.add_(1)
        with torch.cuda.graph(served):
            t.add_(1)
    eng, g = engine(), torch.Generator().manual_seed(4)
    for _ in range(5):
        assert torch.isfinite(eng.train_step([batch(eng, g, 2, 128)])["loss"])
        served.replay()
    assert len(eng.step_graphs.table) == 1


def test_other_threads_draw_while_a_step_is_recorded(native_lib, monkeypatch):
    """A step draws no random numbers: a thread that does, on its own stream, is not kept from it by a recording, and its numbers are those of the seed."""
    from llmctl.runtime.flat import FlatParameters

    zero_grad, drawn, failed = FlatParameters.zero_grad, [], []

    def draw():
        try:
            drawn.append(torch.randn(64, device="cuda"))
        except RuntimeError as e:
            failed.append(e)

    def beside(self):
        if torch.cuda.is_current_stream_capturing():
            t = threading.Thread(target=draw)
            t.start(), t.join()
        return zero_grad(self)

    monkeypatch.setattr(FlatParameters, "zero_grad", beside)
    eng, g = engine(), torch.Generator().manual_seed(7)
    torch.cuda.manual_seed(11)
    want = [torch.randn(64, device="cuda") for _ in range(2)]
    torch.cuda.manual_seed(11)
    for _ in range(5):
        eng.train_step([batch(eng, g, 2, 128)])
    assert len(eng.step_graphs.table) == 1 and not failed and len(drawn) == 1
    draw()
    assert all(torch.equal(x, y) for x, y in zip(want, drawn))


def test_a_recording_that_fails(native_lib, monkeypatch):
    """Its steps stay eager; other shapes are recorded, and given back with the engine."""
    from llmctl.runtime.flat import FlatParameters

    zero_grad, fail = FlatParameters.zero_grad, [True]

    def broken(self):
        zero_grad(self)
        if fail and torch.cuda.is_current_stream_capturing():
            fail.clear()
            raise RuntimeError("no")

    monkeypatch.setattr(FlatParameters, "zero_grad", broken)
    eng, g = engine(), torch.Generator().manual_seed(8)
    for b in (2, 3):
        for _ in range(4):
            assert torch.isfinite(eng.train_step([batch(eng, g, b, 128)])["loss"])
        assert len(eng.step_graphs.table) == b - 2
    eng.step_graphs.table.clear()
    for _ in range(4):
        assert torch.isfinite(eng.train_step([batch(eng, g, 2, 128)])["loss"])
    assert len(eng.step_graphs.table) == 1


def test_streams_of_engines_that_are_gone_are_used_again(native_lib):
    """Engines that live side by side record on streams of their own (the library's workspaces go by stream); the next one takes that of one that is gone."""
    def recorded():
        eng, g = engine(), torch.Generator().manual_seed(9)
        for _ in range(4):
            eng.train_step([batch(eng, g, 2, 128)])
        assert len(eng.step_graphs.table) == 1
        return eng, eng.step_graphs.stream.cuda_stream

    gc.collect()
    a, on_a = recorded()
    b, on_b = recorded()
    assert on_a != on_b
    del a
    gc.collect()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    c, on_c = recorded()
    assert on_c == on_a
    assert torch.cuda.memory_allocated() - before < 64 << 20  # an engine of this model, and no further workspaces


def test_what_listens_is_heard(native_lib):
    """Hooks, modes and faults see every step; parameters that change storage or stop training are not replayed into."""
    eng, g = engine(), torch.Generator().manual_seed(2)
    step = lambda: eng.train_step([batch(eng, g, 2, 128)])  # noqa: E731
    for _ in range(4):  # (the first one builds the rotary tables)
        step()
    assert len(eng.step_graphs.table) == 1
    seen = []
    h = eng.model.layers[0].register_forward_hook(lambda *a: seen.append(1))
    step(), step()
    assert len(seen) == 2
    h.remove()
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t, lambda t: t):
        step()
    assert packed
    p = eng.model.layers[0].wo
    p.requires_grad_(False)
    for _ in range(4):
        step()
    assert float(p.grad.abs().max()) == 0  # not trained, whatever was recorded before
    p.requires_grad_(True)
    w = eng.model.layers[1].attn_norm_w
    before = eng.flat.grad.clone()
    with torch.no_grad():
        w.data = torch.zeros_like(w)  # another storage: the model reads this one
    for _ in range(4):
        step()
    wq = eng.model.layers[1].wqkv
    assert float(wq.grad.abs().max()) == 0 and not torch.equal(before, eng.flat.grad)
    p.grad = None
    step()
    assert p.grad is not None and p.grad.data_ptr() == eng.flat.grad.data_ptr() + 2 * eng.flat.offsets[id(p)]


def test_gradient_hooks_are_heard(native_lib):
    """Post-accumulate hooks: a user's that is there from the first step on (on a weight whose gradient a product writes, on a vector), and one in the place of the engine's own."""
    eng, g, seen = engine(), torch.Generator().manual_seed(5), []
    l = eng.model.layers[0]
    hooks = [p.register_post_accumulate_grad_hook(lambda p: seen.append(1)) for p in (l.wo, l.attn_norm_w)]
    step = lambda: eng.train_step([batch(eng, g, 2, 128)])  # noqa: E731
    for n in range(1, 6):
        step()
        assert len(seen) == 2 * n
    assert len(eng.step_graphs.table) == 0
    for h in hooks:
        h.remove()
    for _ in range(4):
        step()
    assert len(eng.step_graphs.table) == 1 and len(seen) == 10
    eng, seen = engine("gpt2-125m", 2), []
    for _ in range(4):
        step()
    assert len(eng.step_graphs.table) == 1
    p = next(p for p in eng.flat.params if p._post_accumulate_grad_hooks)
    p._post_accumulate_grad_hooks.clear()
    p.register_post_accumulate_grad_hook(lambda p: (seen.append(1), eng.sync._on_grad(p)) and None)
    step(), step()
    assert len(seen) == 2


def test_steps_of_a_subclass_run_its_own_code(native_lib):
    """What an engine of another class, or its configuration, changes from step to step is not frozen in a recording."""
    from llmctl.runtime.engine import TrainingEngine
    from llmctl.runtime.step_graph import fingerprint, same

    class Weighted(TrainingEngine):
        calls = 0

        def _forward_backward(self, *a, **kw):
            self.calls += 1
            return super()._forward_backward(*a, **kw)

    class Named(TrainingEngine):  # overrides nothing that a step runs
        def evaluate(self, batches):
            return 0.0

    for cls, calls, recorded in ((Weighted, 5, 0), (Named, None, 1)):
        eng, g = engine(cls=cls), torch.Generator().manual_seed(6)
        for _ in range(5):
            eng.train_step([batch(eng, g, 2, 128)])
        assert len(eng.step_graphs.table) == recorded and getattr(eng, "calls", None) == calls
    before = fingerprint(eng)
    assert same(before, fingerprint(eng))
    for d, k in ((eng.model.cfg.rope, "base"), (eng.model.cfg.attention, "scale")):
        old = dict(d)
        d[k] = 123.0
        assert not same(before, fingerprint(eng))
        d.clear(), d.update(old)
    assert same(before, fingerprint(eng))


class _Memset(ctypes.Structure):  # hipMemsetParams
    _fields_ = [("dst", ctypes.c_void_p), ("elementSize", ctypes.c_uint), ("height", ctypes.c_size_t), ("pitch", ctypes.c_size_t), ("value", ctypes.c_uint),
                ("width", ctypes.c_size_t)]


@pytest.mark.parametrize("memsets", [0, 1, 3])
def test_memsets_of_a_graph_are_counted(native_lib, memsets):
    """In a graph that was put together by hand and is never run, and in a recording that has none."""
    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
    x, graph, node = torch.ones(256, device="cuda"), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipGraphCreate(ctypes.byref(graph), 0) == 0
    for _ in range(memsets):
        assert hip.hipGraphAddMemsetNode(ctypes.byref(node), graph, None, ctypes.c_size_t(0), ctypes.byref(_Memset(x.data_ptr(), 4, 1, 4 * x.numel(), 0, x.numel()))) == 0
    assert hip.hipGraphAddEmptyNode(ctypes.byref(node), graph, None, ctypes.c_size_t(0)) == 0
    assert native_lib.graph_memsets(graph.value) == memsets
    assert hip.hipGraphDestroy(graph) == 0
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g):
        x.mul_(1.0)
    assert native_lib.graph_memsets(g.raw_cuda_graph()) == 0
    g.reset()


def test_long_steps_stay_eager(native_lib):
    from llmctl.runtime.step_graph import pays

    assert pays(3_000_000, 256, 2) and pays(124_000_000, 1024, 12) and not pays(124_000_000, 8192, 12) and not pays(6_700_000_000, 64, 32)
    eng, g = engine("gpt2-125m", 1), torch.Generator().manual_seed(3)
    for _ in range(4):
        eng.train_step([batch(eng, g, 8, 1024)])
    assert len(eng.step_graphs.table) == 0

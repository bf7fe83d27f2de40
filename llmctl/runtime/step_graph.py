"""Small training steps from one HIP graph: forward, backward and the flat gradients of a batch, recorded once per shape and replayed.

A step of a small model is bound by the host: every launch passes through an autograd function, its checks and the
dispatcher, 15 to 20 us each, while the kernels take 3 to 10.  The recording holds ``zero_grad``, the model's forward and backward
and ``settle_grads``; the clip norm and AdamW, whose step count and learning rate are launch arguments, stay outside and run as
ever.  Whole steps, one MI355X, us, eager / replayed: tiny (2 layers) 256 tokens 940 / 262, 4096 tokens 1335 / 627; gpt2-125m (12
layers) 128 tokens 5852 / 3210, 1024 5888 / 4699, 2048 7594 / 5745 (eager steps are the host's and differ from one to another: 1333, 1742, 7925, 7944, 8088).

A replay runs no Python, so whatever a step's Python could see or change is compared with what was recorded before every
replay (:func:`fingerprint`), and a step that anything listens to (hooks, dispatch modes, anomaly mode, faults to inject) runs eagerly."""

from __future__ import annotations

import weakref
from typing import Dict, List, Optional, Tuple

import torch

from llmctl.serve.decode_graph import GraphTable
from llmctl.utils.env import graph_capture_gc_guard

# What a recording is worth, from the sizes: host seconds of an eager step against seconds of its kernels (the products, and weights, gradients and
# optimizer states through HBM).  Where the kernels take longer than the host a replay gains nothing and would keep its activations for
# itself: gpt2-125m eager / replayed, us, 4096 tokens 8180 / 8188, 8192 11399 / 11395; one GPT-7B layer 64 tokens 4017 / 3991.
HOST_STEP, HOST_LAYER = 0.5e-3, 0.55e-3
PRODUCT_RATE, BYTES_PER_PARAMETER, COPY_RATE = 0.45e15, 40, 4.5e12


def pays(parameters: int, tokens: int, layers: int) -> bool:
    kernels = 6.0 * parameters * tokens / PRODUCT_RATE + BYTES_PER_PARAMETER * parameters / COPY_RATE
    return kernels < HOST_STEP + HOST_LAYER * layers


def _watched() -> bool:
    """Something in this thread sees or changes the calls of a step as they are made."""
    C = torch._C
    return (not torch.is_grad_enabled() or torch.is_inference_mode_enabled() or torch.is_autocast_enabled("cuda") or torch.is_anomaly_enabled()
            or C._len_torch_function_stack() > 0 or C._len_torch_dispatch_stack() > 0 or C._functorch.peek_interpreter_stack() is not None
            or C._autograd._top_saved_tensors_default_hooks(True) is not None or C._autograd._profiler_enabled()
            or not C._autograd._saved_tensors_hooks_is_enabled() or torch.cuda.is_current_stream_capturing())


_STEP = ("_gradients", "_forward_backward", "_packing")  # the engine's methods in a recording


def _own_code(engine) -> bool:
    """Nobody has put code of their own, by a subclass or on an object, in the place of what a recording runs once."""
    from llmctl.comms.overlap import GradSyncEngine
    from llmctl.exec.linear import GradSink
    from llmctl.runtime.engine import TrainingEngine
    from llmctl.runtime.flat import FlatParameters

    return (all(getattr(type(engine), n) is getattr(TrainingEngine, n) and n not in vars(engine) for n in _STEP)
            and all(type(o) is t and not any(map(callable, vars(o).values()))
                    for o, t in ((engine.sync, GradSyncEngine), (engine.flat, FlatParameters), (engine.grad_sink, GradSink))))


def _values(v):
    """A copy of a configuration's values that later changes inside it do not reach."""
    if isinstance(v, dict):
        return {k: _values(x) for k, x in v.items()}
    return [_values(x) for x in v] if isinstance(v, (list, tuple)) else v


def fingerprint(engine) -> Optional[Tuple]:
    """What the recorded calls of a step depend on besides its batch; None: this step must run eagerly."""
    from torch.nn.modules import module as nnm

    from llmctl.exec.linear import GEMM64_CONFIGS, GEMM64_SHAPE_CONFIGS
    from llmctl.models.transformer import DecoderLayer, DecoderLM
    from llmctl.ops._lib import use_native

    c, m, opt, sync, flat = engine.config, engine.model, engine.optimizer, engine.sync, engine.flat
    if (engine.env.world_size > 1 or engine.eflat is not None or engine.pipeline is not None or engine.faults
            or c.pack_sequences or opt.overlap_update or opt._pending or flat.main_grads or sync is None or not sync.enabled
            or type(m) is not DecoderLM or m.cfg.is_moe or m.pc.activation_checkpoint != "none"
            or not _own_code(engine) or not use_native(flat.data)
            or torch.cuda.current_device() != engine.device.index
            or nnm._global_forward_hooks or nnm._global_forward_pre_hooks or nnm._global_backward_hooks or nnm._global_backward_pre_hooks or _watched()):
        return None
    sink = engine.grad_sink
    if sink is None or sink.callbacks != [sync._on_grad] or sink.always_transpose:
        return None
    mods = list(m.modules())
    if any(d._forward_hooks or d._forward_pre_hooks or d._backward_hooks or d._backward_pre_hooks or d._buffers
           or any(map(callable, vars(d).values())) for d in mods):
        return None
    if any(type(d) is not DecoderLayer or d.cfg is not m.cfg or d.pc is not m.pc for d in m.layers):
        return None
    ps = [p for d in mods for p in d._parameters.values() if p is not None]
    if any(p._backward_hooks for p in ps):
        return None
    sinked = [getattr(p, "_llmctl_grad_sink", None) is sink for p in ps]
    for p, written in zip(ps, sinked):  # the engine's own hook and no other
        if [*(p._post_accumulate_grad_hooks or {}).values()] != ([] if written else [sync._on_grad]):
            return None
    at, size, grads = flat.grad.data_ptr(), flat.grad.element_size(), [p.grad for p in flat.params]
    if any(g is None or g.data_ptr() != at + size * flat.offsets[id(p)] for p, g in zip(flat.params, grads)):
        return None  # (``zero_grad`` puts the views back)
    ropes = [t for v in m._rope_cache.values() for t in v]
    return (list(map(id, mods)), list(map(id, ps)), list(map(id, ropes)), list(map(torch.Tensor.data_ptr, ps)),
            [(p.requires_grad, p._llmctl_writes if written else 0) for p, written in zip(ps, sinked)],
            at, _values(vars(m.cfg)), dict(vars(m.pc)), engine.knobs,
            dict(GEMM64_CONFIGS), dict(GEMM64_SHAPE_CONFIGS), torch.are_deterministic_algorithms_enabled(), (mods, ps, ropes))


def same(a: Tuple, b: Tuple) -> bool:
    return a[:-1] == b[:-1]  # (the last entry keeps the objects, so that no identity is given to another one)


class StepGraph:
    """One recorded shape: static inputs, the graph, its loss."""

    def __init__(self, x: torch.Tensor, y: torch.Tensor):
        self.x, self.y = torch.empty_like(x, memory_format=torch.contiguous_format), torch.empty_like(y, memory_format=torch.contiguous_format)
        self.graph = self.loss = None

    def capture(self, engine, denom: float, stream, pool) -> None:
        """Record.  Nothing runs, so a failure (raised) leaves the gradients as they were."""
        from llmctl.ops._lib import native

        lib, g = native(), torch.classes.llmctl.StepCapture(*pool)
        with graph_capture_gc_guard(collect=False), torch.cuda.stream(stream):
            g.begin()
            try:
                loss = engine._gradients(self.x, self.y, denom)
            except BaseException:
                g.release()
                raise
            try:
                g.end()
                if lib.graph_memsets(g.graph()):  # (a library's sum over many blocks clears its counters so)
                    raise RuntimeError("the step records a memset")
                g.instantiate()
            except RuntimeError:
                del loss
                g.release()
                raise
        self.graph, self.loss = g, loss

    def run(self, x: torch.Tensor, y: torch.Tensor) -> torch.Tensor:
        self.x.copy_(x)
        self.y.copy_(y)
        self.graph.replay()
        return self.loss.clone()  # (the next replay writes the graph's own)

    def release(self) -> None:
        self.graph.release()  # (waits for its last replay, on whatever stream)
        self.graph = self.loss = None


# streams of engines that are gone, by device: the library keeps two workspaces for good per stream that its products are recorded on (160 MB), and the graphs
# of engines that live side by side may not share one
_idle: Dict[torch.device, List["torch.cuda.Stream"]] = {}


class StepGraphs:
    """The recorded steps of one engine: a stream and a memory pool of its own (the graphs run one after the other, as the steps do)."""

    def __init__(self):
        self.table, self.seen, self.stream, self.pool = GraphTable(), None, None, None

    def _take_stream(self, device: torch.device) -> None:
        idle = _idle.setdefault(device, [])
        try:
            self.stream = idle.pop()
        except IndexError:
            self.stream = torch.cuda.Stream(device=device)
        weakref.finalize(self, idle.append, self.stream).atexit = False

    def run(self, engine, batches: List[Tuple[torch.Tensor, torch.Tensor]]) -> Optional[torch.Tensor]:
        """The loss of a replayed step, its gradients in the flat buffer; None: run it eagerly."""
        if len(batches) != 1 or engine.device.type != "cuda" or not engine.knobs.step_graph or engine.zero3 is not None:
            return None
        (x, y), m = batches[0], engine.model
        for t in (x, y):
            if type(t) is not torch.Tensor or t.device != engine.device or t.dtype != torch.int64 or t.dim() != 2 or x.shape != y.shape:
                return None
        if not pays(engine.flat.numel, x.numel(), len(m.layers)):
            return None
        shape = tuple(x.shape)
        now = fingerprint(engine) if self.table.due(shape) else self.seen  # (a shape's first steps are not replayed: nothing to compare)
        if now is None and self.table.due(shape):
            return None
        if self.seen is not None and not same(now, self.seen):
            self.table.clear()
        self.seen = now
        g = self.table.step(shape, lambda shape: self._record(engine, x, y, float(y.numel())))
        return None if g is None else g.run(x, y)

    def _record(self, engine, x, y, denom) -> Optional[StepGraph]:
        from llmctl.exec.linear import weight_t_ok
        from llmctl.runtime.engine import log

        if any(p.dim() == 2 and weight_t_ok(x.numel(), p) for p in engine.flat.params):
            return None  # (a transposed copy is refreshed once a step by its epoch, on the host)
        if not len(self.table):  # (a pool ends with its last graph)
            self.pool = torch.cuda.graph_pool_handle()
        if self.stream is None:
            self._take_stream(engine.device)
        try:
            g = StepGraph(x, y)
            g.capture(engine, denom, self.stream, self.pool)
            return g
        except RuntimeError as e:  # (no memory left, too)
            log.warning("training steps of %s tokens stay eager: %s", tuple(x.shape), e)
            with engine.sync.no_sync():  # (forgets what the recording counted)
                pass
            return None

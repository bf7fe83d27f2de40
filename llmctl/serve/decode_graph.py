"""A captured decode step of a hybrid-mixer model: static device inputs behind one staged copy, the model's step over
``n`` rows and its logits as one HIP graph.

Recurrent states live in the step itself, so nothing may run twice: there are no warm-up passes, and the pools have no scratch
slot that a padded row could write.  The
engine runs the first steps of a shape eagerly (:data:`WARM_STEPS`: they load the kernels and build what the modules
derive from their weights once), then records the same calls and replays them.  A shape is the number of rows and the
power of two that holds the longest context, which sizes the split of the keys over workgroups; the kernels read every
sequence's own length from device memory, so any context runs through any split.

Batches change shape all the time, so a recording must be cheap: it takes the host's time for the step's launches, without the
synchronisation, the collection of garbage and the emptied allocator that ``torch.cuda.graph`` starts with.  The step that records and its
first replay, one MI355X, 9 to 15 rows, with / without those three: Malinex (3 layers) 26.4 / 1.1 ms, Lenitar (4) 29 / 1.7, Dumazen (6) 28 / 1.6; their
eager steps take 0.7, 0.9 and 1.0.  Sixteen row counts in turn, 12 rounds: Malinex 1405 / 346 us a step, Lenitar 1515 / 486.
What does not record (no memory left, a module that waits for the device) runs eagerly, as the first steps do."""

from __future__ import annotations

import threading
from typing import Callable, Dict, List, Optional, Sequence, Tuple

import numpy as np
import torch

from llmctl.exec.linear import recorded_step
from llmctl.utils.env import graph_capture_gc_guard

WARM_STEPS = 2  # eager steps of a shape before it is captured
CROWDED_STEPS = 16  # the same once another shape's graph has to go for it: what a recording costs is then a small part of these steps
MAX_GRAPHS = 64  # shapes kept per engine; the least recently used one goes first
STAGES = 4  # pinned input sets: the host runs at most this many steps ahead of the copies


def packed_layout(arrays: Sequence[np.ndarray]) -> Tuple[List[int], int]:
    """Byte offset of every array in one buffer (16-byte aligned) and the buffer's size."""
    offs, at = [], 0
    for a in arrays:
        offs.append(at)
        at += (a.nbytes + 15) // 16 * 16
    return offs, max(at, 16)


def packed_views(buf: torch.Tensor, offs: Sequence[int], arrays: Sequence[np.ndarray]) -> List[torch.Tensor]:
    """Typed views of the packed buffer, one per array."""
    kinds = {np.dtype(np.int64): torch.int64, np.dtype(np.int32): torch.int32}
    return [buf[o:o + a.nbytes].view(kinds[a.dtype]).view(a.shape) for o, a in zip(offs, arrays)]


def upload_packed(arrays: Sequence[np.ndarray], device) -> List[torch.Tensor]:
    """The arrays on ``device`` through ONE host-to-device copy, for a GPU from pinned memory, which its allocator keeps until the copy is over: the
    host does not wait for the steps before (a Dumazen prompt of 700 tokens among others 1525 us with the wait, 1430 without)."""
    offs, size = packed_layout(arrays)
    host = torch.empty(size, dtype=torch.uint8, pin_memory=torch.device(device).type == "cuda")
    flat = host.numpy()
    for o, a in zip(offs, arrays):
        flat[o:o + a.nbytes] = np.ascontiguousarray(a).view(np.uint8).reshape(-1)
    return packed_views(host.to(device, non_blocking=True), offs, arrays)


class DecodeGraph:
    FIELDS = ("ids", "slots", "pos", "ctx", "start", "state", "bt")

    def __init__(self, n: int, max_blocks: int, max_ctx: int, device):
        from llmctl.models.mixers import StepBatch

        i64, i32 = np.zeros(n, np.int64), np.zeros(n, np.int32)
        self.arrays = [i64, i64, i32, i32, i32, i32, np.zeros((n, max_blocks), np.int32)]
        self.offs, size = packed_layout(self.arrays)
        self.buf = torch.zeros(size, dtype=torch.uint8, device=device)
        v = dict(zip(self.FIELDS, packed_views(self.buf, self.offs, self.arrays)))
        self.ids = v["ids"]
        self.ids_end = self.offs[1]
        cu = torch.arange(n + 1, dtype=torch.int32, device=device)
        self.batch = StepBatch(ids=v["ids"], pos=v["pos"], slots=v["slots"], Tp=0, p_cu=None, p_ctx=None, p_bt=None,
                               d_ctx=v["ctx"], d_bt=v["bt"], cu=cu, start=v["start"], state=v["state"], max_q=0,
                               cu_host=list(range(n + 1)), seq_of=cu[:n], d_max_ctx=max_ctx, carried=False, fresh=False)
        # one pinned block for all input sets (each pinned allocation is a call into the driver)
        hosts = torch.zeros(STAGES, size, dtype=torch.uint8, pin_memory=True)
        self.stages = [(h, h.numpy(), torch.cuda.Event()) for h in hosts]
        self.turn = 0
        self.graph = self.logits = None

    def capture(self, model, cache, pool) -> None:
        """Record the step.  Nothing runs, so a failure (raised) leaves caches and states as they were."""
        g = torch.cuda.CUDAGraph()
        with _capturing, recorded_step(), graph_capture_gc_guard(collect=False), torch.cuda.stream(_capture_stream(self.buf.device)):
            # other threads go on working meanwhile: only this thread's calls are held to what a capture allows
            g.capture_begin(pool=pool, capture_error_mode="thread_local")
            try:
                self.batch.scratch.clear()
                logits = model.logits(model.step(self.batch, cache, **({"final": True} if getattr(model, "normed_step", False) else {})))
            except BaseException:
                try:
                    g.capture_end()
                except RuntimeError:
                    pass  # (the first error is the one to tell)
                self.batch.scratch.clear()
                g.reset()
                raise
            g.capture_end()
        self.graph, self.logits = g, logits

    def release(self) -> None:
        torch.cuda.synchronize(self.buf.device)  # its last replay, on whatever stream
        self.graph.reset()
        self.graph = self.logits = None

    def run(self, values: Dict[str, np.ndarray], ids_on_device=None) -> torch.Tensor:
        """Stage the step's inputs, copy them over, replay.  ``ids_on_device``: the input tokens, already sampled there.
        Returns a fresh tensor of logits (the next replay overwrites the graph's own)."""
        host, flat, ev = self.stages[self.turn]
        self.turn = (self.turn + 1) % STAGES
        ev.synchronize()  # the copy that last read this set
        for name, o, a in zip(self.FIELDS, self.offs, self.arrays):
            if name == "ids" and ids_on_device is not None:
                continue
            flat[o:o + a.nbytes].view(a.dtype).reshape(a.shape)[...] = values[name]
        if ids_on_device is None:
            self.buf.copy_(host, non_blocking=True)
        else:
            self.buf[self.ids_end:].copy_(host[self.ids_end:], non_blocking=True)
            self.ids.copy_(ids_on_device)
        ev.record()
        self.graph.replay()
        return self.logits.clone()


_capturing = threading.Lock()  # one recording at a time: they share a stream
_capture_streams: Dict[torch.device, "torch.cuda.Stream"] = {}


def _capture_stream(device: torch.device) -> "torch.cuda.Stream":
    s = _capture_streams.get(device)
    if s is None:
        s = _capture_streams[device] = torch.cuda.Stream(device=device)
    return s


class GraphTable:
    """The shapes of an engine's decode steps: how many eager steps each has had, or its graph, or that it does not record."""

    def __init__(self):
        self._shapes: Dict[Tuple[int, int], object] = {}  # least recently used first
        self._graphs = 0

    def __len__(self) -> int:
        return self._graphs

    def due(self, shape: Tuple[int, int]) -> bool:
        """Whether the next step of ``shape`` may be replayed or recorded."""
        e = self._shapes.get(shape, 0)
        return e is not None and (not isinstance(e, int) or e >= WARM_STEPS)

    def warming(self, shape: Tuple[int, int]) -> bool:
        """Whether ``shape`` is to be recorded after some more eager steps."""
        return isinstance(self._shapes.get(shape), int)

    def step(self, shape: Tuple[int, int], record: Callable[[Tuple[int, int]], Optional[DecodeGraph]]) -> Optional[DecodeGraph]:
        """The graph that runs the next step of ``shape``; None: it runs eagerly.  ``record(shape)``: its graph, or None where it
        cannot be recorded."""
        e = self._shapes.pop(shape, 0)
        if isinstance(e, int):
            if e >= (WARM_STEPS if self._graphs < MAX_GRAPHS else CROWDED_STEPS):
                if self._graphs >= MAX_GRAPHS:
                    old = next(k for k, v in self._shapes.items() if v is not None and not isinstance(v, int))
                    self._shapes.pop(old).release()
                    self._graphs -= 1
                e = record(shape)
                self._graphs += e is not None
            else:
                e += 1
        self._shapes[shape] = e
        return None if isinstance(e, int) else e

    def clear(self) -> None:
        for e in self._shapes.values():
            if e is not None and not isinstance(e, int):
                e.release()
        self._shapes.clear()
        self._graphs = 0

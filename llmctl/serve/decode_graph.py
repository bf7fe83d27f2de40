"""A captured decode step of a hybrid-mixer model: static device inputs behind one staged copy, the model's step over
``n`` rows and its logits as one HIP graph.

Recurrent states live in the step itself, so nothing may run twice: there are no warm-up passes and no padded rows.  The
engine runs the first steps of a shape eagerly (:data:`WARM_STEPS`: they load the kernels and build what the modules
derive from their weights once), then records the same calls and replays them.  A shape is the number of rows and the
power of two that holds the longest context, which sizes the split of the keys over workgroups; the kernels read every
sequence's own length from device memory, so any context runs through any split."""

from __future__ import annotations

from typing import Dict, List, Sequence, Tuple

import numpy as np
import torch

from llmctl.utils.env import graph_capture_gc_guard

WARM_STEPS = 2  # eager steps of a shape before it is captured
MAX_GRAPHS = 32  # shapes kept per engine; the least recently used one goes first
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
    """The arrays on ``device`` through ONE host-to-device copy."""
    offs, size = packed_layout(arrays)
    host = np.empty(size, dtype=np.uint8)
    for o, a in zip(offs, arrays):
        host[o:o + a.nbytes] = np.ascontiguousarray(a).view(np.uint8).reshape(-1)
    return packed_views(torch.from_numpy(host).to(device), offs, arrays)


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
        self.stages = []
        for _ in range(STAGES):
            host = torch.zeros(size, dtype=torch.uint8, pin_memory=True)
            ev = torch.cuda.Event()
            self.stages.append((host, host.numpy(), ev))
        self.turn = 0
        self.graph = self.logits = None

    def capture(self, model, cache, pool) -> None:
        g = torch.cuda.CUDAGraph()
        with graph_capture_gc_guard(), torch.cuda.graph(g, pool=pool):
            self.batch.scratch.clear()
            self.logits = model.logits(model.step(self.batch, cache))
        self.graph = g

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

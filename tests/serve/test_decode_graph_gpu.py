"""Captured decode steps of the hybrid families against the eager ones: the same sequences through an engine with graphs and
one without, over several replays with eager work in between, sequences that come and go (other row counts, reused state
slots and pages), a context that passes a power of two, tokens fed back on the device, weights changed in place or exchanged, shapes
that are given up or do not record, and other threads at work during a recording."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

MODELS = ["lenitar-w128-l4", "dumalix-w128-l4-h4-g2", "malinex-w128-l4-h4-g2-e4-s1", "malinex-w128-l3-h4-g2",
          "pamazen-w128-l4-h4-g2-e4", "dapipel-w128-l4-h4-g2-e4", "dumazen-w128-l4-h4-g2"]


def _engine(name, graphs, dtype):
    from llmctl.serve.engine import InferenceEngine

    return InferenceEngine(name, device="cuda", max_batch_size=4, num_kv_blocks=64, block_size=16, max_model_len=256, dtype=dtype,
                           use_graphs=graphs, prefix_caching=False, seed=3)


def _close(a, b, dtype):
    # the eager step splits the keys by the longest context itself, the captured one by the power of two above it: the
    # same sums in another order (bf16: an output may round the other way in every layer; fp32: sums of some hundred terms)
    tol = 2e-2 if dtype == torch.bfloat16 else 1e-4
    assert (a.float() - b.float()).norm() <= tol * b.float().norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("name", MODELS)
def test_captured_steps_match_eager_ones(name, dtype):
    from llmctl.serve.scheduler import PrefillChunk

    es = [_engine(name, g, dtype) for g in (True, False)]
    gen = torch.Generator().manual_seed(0)
    toks = lambda n: torch.randint(0, 500, (n,), generator=gen).tolist()

    def admit(ids):
        out = []
        for e in es:
            s = e.open_sequence(ids)
            e.prefill([PrefillChunk(s, 0, len(ids))])
            e.scheduler.computed(s, len(ids))
            out.append(s)
        return out

    def step(pairs):
        new, got = [toks(1)[0] for _ in pairs], []
        for k, e in enumerate(es):
            for p, t in zip(pairs, new):
                e.scheduler.extend(p[k], [t])
                p[k]._decode_slot = int(e.kv.slots(p[k].seq_id, p[k].num_tokens - 1, 1)[0])
            got.append(e.decode([p[k] for p in pairs]))
            for p in pairs:
                e.scheduler.computed(p[k], 1)
        _close(got[0], got[1], dtype)
        return got[0]

    live = [admit(toks(n)) for n in (60, 5, 17)]
    first = None
    for i in range(9):  # the longest context passes 64; three replays and more on each side of it
        out = step(live)
        if i == 4:
            first = (out, out.clone())
    assert torch.equal(*first)  # a later replay does not write into logits that were handed out
    for k, e in enumerate(es):
        e.scheduler.finish(live[1][k], "stop")
    del live[1]
    for _ in range(4):
        step(live)
    live.append(admit(toks(40)))  # the freed slot and pages, beside eager prefills
    for _ in range(5):
        step(live)
    for e in es:  # weights changed in place: neither the graph nor what modules derive from them may stay
        with torch.no_grad():
            for p in e.model.parameters():
                p.mul_(0.9)
    for _ in range(4):
        step(live)
    replays = es[0].stats["graph_replays"]
    moe_fp32 = dtype == torch.float32 and name.startswith("lenitar")  # its experts count rows on the host in fp32
    assert replays == 0 if moe_fp32 else replays >= 8
    assert es[1].stats["graph_replays"] == 0
    for e in es:
        e.close()


class _Pair:
    """The same sequences in an engine with graphs and one without."""

    def __init__(self, name, dtype=torch.bfloat16):
        self.es, self.dtype = [_engine(name, g, dtype) for g in (True, False)], dtype
        self.gen = torch.Generator().manual_seed(1)
        self.live = []

    def admit(self, n):
        from llmctl.serve.scheduler import PrefillChunk

        ids, out = torch.randint(0, 500, (n,), generator=self.gen).tolist(), []
        for e in self.es:
            s = e.open_sequence(ids)
            e.prefill([PrefillChunk(s, 0, n)])
            e.scheduler.computed(s, n)
            out.append(s)
        self.live.append(out)

    def step(self, rows):
        new, got = torch.randint(0, 500, (rows,), generator=self.gen).tolist(), []
        for k, e in enumerate(self.es):
            seqs = [p[k] for p in self.live[:rows]]
            for s, t in zip(seqs, new):
                e.scheduler.extend(s, [t])
                s._decode_slot = int(e.kv.slots(s.seq_id, s.num_tokens - 1, 1)[0])
            got.append(e.decode(seqs))
            for s in seqs:
                e.scheduler.computed(s, 1)
        _close(got[0], got[1], self.dtype)

    def check_caches(self):
        """Rows and states of the live sequences."""
        for i in range(len(self.es[0].kv_cache._layers)):
            flat = lambda v: [t for w in (v if isinstance(v, tuple) else (v,)) for t in (w if isinstance(w, tuple) else (w,))]
            for a, b in zip(*(flat(e.kv_cache.layer(i)) for e in self.es)):
                if b.float().norm() > 0:
                    _close(a, b, self.dtype)

    def replays(self):
        return self.es[0].stats["graph_replays"]

    def close(self):
        for e in self.es:
            e.close()


def test_shapes_come_and_go(monkeypatch):
    from llmctl.serve import decode_graph as dg

    monkeypatch.setattr(dg, "MAX_GRAPHS", 2)
    monkeypatch.setattr(dg, "CROWDED_STEPS", 3)
    p = _Pair("dumazen-w128-l4-h4-g2")
    for n in (40, 41, 36, 38):
        p.admit(n)
    for rows in (4, 4, 4, 3, 3, 3, 2, 2, 2, 2, 4, 4, 4, 4, 3, 1, 1, 2, 1, 1, 4, 4):
        p.step(rows)
    p.check_caches()
    assert p.replays() == 6 and len(p.es[0]._decode_graphs) == 2  # recorded: 4, 3, 2 (4 goes), 4 (3 goes), 1 (4 goes); one more of 2
    p.close()


@pytest.mark.parametrize("width", [5, 20])
def test_plans_with_block_tables_of_another_width(width):
    """A caller's own plan may hold just the blocks that are in use, or more columns than the engine's."""
    p = _Pair("malinex-w128-l4-h4-g2-e4-s1")
    for n in (40, 45):  # (no context passes a power of two)
        p.admit(n)
    for _ in range(4):
        p.step(2)
    assert p.replays() == 2
    got = []
    for k, e in enumerate(p.es):
        seqs = [s[k] for s in p.live]
        for s in seqs:
            e.scheduler.extend(s, [7])
            s._decode_slot = int(e.kv.slots(s.seq_id, s.num_tokens - 1, 1)[0])
        plan = e.decode_plan(seqs)
        assert plan["bt"].shape[1] == 16 and all(c <= 5 * 16 for c in plan["ctx"])
        plan["bt"] = np.pad(plan["bt"], ((0, 0), (0, 4)))[:, :width].copy()
        got.append(e.decode_exec(plan))
        for s in seqs:
            e.scheduler.computed(s, 1)
    _close(got[0], got[1], p.dtype)
    p.step(2)
    p.check_caches()
    assert p.replays() == 3
    p.close()


@pytest.mark.parametrize("error,stays", [(RuntimeError, 0), (torch.OutOfMemoryError, 3)])
def test_a_step_that_does_not_record_runs_eagerly(monkeypatch, error, stays):
    """A failure inside the recording (memory: once) leaves caches, states and later recordings as they should be."""
    p = _Pair("malinex-w128-l4-h4-g2-e4-s1")
    for n in (20, 7, 40):
        p.admit(n)
    model, failures = p.es[0].model, []
    logits = type(model).logits

    def fail(self, x):
        if torch.cuda.is_current_stream_capturing() and x.shape[0] == 3 and not (stays and failures):
            failures.append(1)
            raise error("no room")
        return logits(self, x)

    monkeypatch.setattr(type(model), "logits", fail)
    for _ in range(5):
        p.step(3)
    assert len(failures) == 1 and p.replays() == stays
    for _ in range(5):
        p.step(2)
    p.check_caches()
    assert p.replays() == stays + 3
    p.close()


def test_exchanged_weights_are_used():
    """Two parameters that change places, one that is another object (a checkpoint assigned), a module that is another one."""
    p = _Pair("dumazen-w128-l4-h4-g2")
    p.admit(20)
    p.admit(9)
    models = [e.model for e in p.es]

    def change_places(m):
        a, b = (m.layers[i].ff.w_down for i in (0, 1))
        a.data, b.data = b.data, a.data

    def assign(m):
        m.load_state_dict({k: v * 0.9 if v.is_floating_point() else v for k, v in m.state_dict().items()}, assign=True)

    def exchange(m):
        m.layers[0].ff, m.layers[1].ff = m.layers[1].ff, m.layers[0].ff

    for change in (None, change_places, assign, exchange):
        before = p.replays()
        if change is not None:
            for m in models:
                change(m)
        for _ in range(4):
            p.step(2)
        assert p.replays() == before + 2
    p.close()


def test_other_threads_work_during_recordings():
    import threading

    stop, errors = threading.Event(), []

    def work():
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                k = 0
                while not stop.is_set():
                    k = k % 64 + 1
                    t = torch.full((k << 14,), float(k), device="cuda")
                    assert float(t.sum().cpu()) == k * (k << 14)
                    torch.from_numpy(t[:8].cpu().numpy()).cuda()
                    s.synchronize()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    th = threading.Thread(target=work)
    th.start()
    try:
        p = _Pair("dumazen-w128-l4-h4-g2")
        for n in (36, 37, 38, 39):
            p.admit(n)
        for rows in (4, 3, 2, 1):
            for _ in range(4):
                p.step(rows)
        assert p.replays() == 8
    finally:
        stop.set()
        th.join()
    assert not errors, errors
    p.close()


def test_the_position_limit_holds_for_replays(monkeypatch):
    p = _Pair("malinex-w128-l4-h4-g2-e4-s1")
    p.admit(20)
    for _ in range(4):
        p.step(1)
    assert p.replays() == 2
    monkeypatch.setattr(type(p.es[0].model), "position_limit", 24)
    for e in p.es:
        with pytest.raises(ValueError, match="beyond the model's 24"):
            s = p.live[0][p.es.index(e)]
            e.scheduler.extend(s, [1])
            s._decode_slot = int(e.kv.slots(s.seq_id, s.num_tokens - 1, 1)[0])
            e.decode([s])
    p.close()


@pytest.mark.parametrize("name", ["malinex-w128-l4-h4-g2-e4-s1", "dumazen-w128-l4-h4-g2"])
def test_generated_tokens_are_the_same(name):
    """Greedy generation, where a continued step takes its input tokens from the device."""
    from llmctl.serve.scheduler import SamplingParams

    outs = []
    for graphs in (True, False):
        e = _engine(name, graphs, torch.float32)
        seqs = e.generate([[1, 2, 3, 4, 5], [7, 8], [9] * 30], SamplingParams(max_tokens=24, temperature=0.0, ignore_eos=True))
        outs.append([s.output_ids for s in seqs])
        assert (e.stats["graph_replays"] > 0) == graphs
        e.close()
    assert outs[0] == outs[1]


def test_the_upload_of_a_step_does_not_wait():
    """The index arrays are on their way while earlier kernels still run, and arrive as they were when the call was made."""
    from llmctl.serve.decode_graph import upload_packed

    arrays = [np.arange(700, dtype=np.int64), np.zeros(0, np.int32), np.arange(300, dtype=np.int32).reshape(3, 100)]
    upload_packed(arrays, torch.device("cuda"))  # (the first pinned block of this size is an allocation)
    a = torch.randn(8192, 8192, device="cuda").bfloat16()
    torch.cuda.synchronize()
    for _ in range(40):  # some 30 ms
        b = a @ a
    done = torch.cuda.Event()
    done.record()
    got = upload_packed(arrays, torch.device("cuda"))
    want = [x.copy() for x in arrays]
    for x in arrays:
        x[...] = -1
    assert not done.query()
    for g, w in zip(got, want):
        assert g.shape == w.shape and torch.equal(g.cpu(), torch.from_numpy(w))


def _cache_tensors(e):
    out = []
    for i in range(len(e.kv_cache._layers)):
        v = e.kv_cache.layer(i)
        for w in v if isinstance(v, tuple) else (v,):
            out += list(w) if isinstance(w, tuple) else [w]
    return out


@pytest.mark.parametrize("name,cut", [("lenitar-w128-l4", None), ("malinex-w128-l4-h4-g2-e4-s1", None), ("malinex-w128-l3-h4-g2", None), ("dumazen-w128-l4-h4-g2", None),
                                      ("malinex-w2048-l3-h16-g4", None), ("dumazen-w2048-l3-h16-g4", None), ("dumazen-w128-l4-h4-g2", "ff"), ("dumazen-w128-l4-h4-g2", "layers"), ("malinex-w128-l3-h4-g2", "layers")])
def test_a_step_gives_the_same_bits_captured_or_not(name, cut):
    """One decode step from the same caches, eager, captured, and eager with the final norm as a pass of its own; a last layer without a feed-forward part, and
    no layers at all."""
    from llmctl.serve.decode_graph import DecodeGraph
    from llmctl.serve.scheduler import PrefillChunk

    e = _engine(name, False, torch.bfloat16)
    if cut == "ff":
        e.model.layers[-1].ff = None
    elif cut == "layers":
        if hasattr(e.model, "order"):
            e.model.order = []
        else:
            e.model.layers = torch.nn.ModuleList()
    gen = torch.Generator().manual_seed(2)
    seqs = []
    for n in (63, 40, 17):  # the longest context becomes 64, which the captured step's bound is too
        ids = torch.randint(0, 500, (n,), generator=gen).tolist()
        s = e.open_sequence(ids)
        e.prefill([PrefillChunk(s, 0, n)])
        e.scheduler.computed(s, n)
        e.scheduler.extend(s, [n])
        s._decode_slot = int(e.kv.slots(s.seq_id, s.num_tokens - 1, 1)[0])
        seqs.append(s)
    plan = e.decode_plan(seqs)
    assert max(plan["ctx"]) == 64
    live = _cache_tensors(e)
    saved = [t.clone() for t in live]

    def restore():
        with torch.inference_mode():
            for t, v in zip(live, saved):
                t.copy_(v)

    with torch.inference_mode():
        eager = e.decode_exec(plan).clone()
        restore()
        g = DecodeGraph(3, e.max_blocks_per_seq, 64, e.device)
        g.capture(e.model, e.kv_cache, torch.cuda.graph_pool_handle())
        run = lambda: g.run({"ids": plan["ids"], "slots": plan["slots"], "pos": plan["positions"], "ctx": plan["ctx"], "start": plan["positions"], "state": plan["state"],
                             "bt": plan["bt"]})
        captured = run()
        for _ in range(2):  # (a replay after others, from the same caches)
            restore()
            assert torch.equal(run(), captured)
        restore()
        e.model.normed_step = False  # the final norm of its own, in the form that prompts take
        apart = e.decode_exec(plan)
        assert torch.equal(eager, captured)
        # the same norm in another order of its sum: its bf16 results may round the other way
        a, b = eager.float(), apart.float()
        assert ((a - b).norm(dim=1) <= 2.0**-7 * b.norm(dim=1)).all()
    g.release()
    e.close()


@pytest.mark.parametrize("name,rows", [("lenitar-w1024-l4", 33), ("malinex-w2048-l3-h16-g4-e4", 64), ("dumazen-w2048-l3-h16-g4", 64), ("gpt2-125m", 33)])
def test_a_recording_calls_no_library_product_first(name, rows, monkeypatch):
    """More than 32 rows, whose products go by size: what the recorded step has the library do, the eager steps ahead of it did (it makes its handle and loads its kernels there)."""
    from llmctl.serve.engine import InferenceEngine
    from llmctl.serve.scheduler import PrefillChunk

    e = InferenceEngine(name, device="cuda", max_batch_size=rows, num_kv_blocks=rows + 1, block_size=16, max_model_len=16, dtype=torch.bfloat16, prefix_caching=False, seed=3)
    a, b = torch.ones(64, 256, device="cuda", dtype=torch.bfloat16), torch.ones(256, 256, device="cuda", dtype=torch.bfloat16)
    torch.nn.functional.linear(a, b), torch.nn.functional.linear(a, b, b[0])  # (its handle, so that this test ends in any case)
    seqs = [e.open_sequence([1 + i, 2, 3, 4, 5]) for i in range(rows)]
    e.prefill([PrefillChunk(s, 0, 5) for s in seqs])
    for s in seqs:
        e.scheduler.computed(s, 5)
    calls, lib = {False: set(), True: set()}, torch.nn.functional.linear

    def linear(x, w, *rest):
        calls[torch.cuda.is_current_stream_capturing()].add((tuple(x.shape), tuple(w.shape)))
        return lib(x, w, *rest)

    monkeypatch.setattr(torch.nn.functional, "linear", linear)
    for t in range(3):  # contexts of 6 to 8: one shape
        for s in seqs:
            e.scheduler.extend(s, [6 + t])
            s._decode_slot = int(e.kv.slots(s.seq_id, s.num_tokens - 1, 1)[0])
        e.decode(seqs)
        for s in seqs:
            e.scheduler.computed(s, 1)
    assert len(e._decode_graphs if e.hybrid else e._graphs) == 1 and calls[True] and calls[True] <= calls[False]

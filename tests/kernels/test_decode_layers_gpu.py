"""A whole decode step in one launch (``csrc/decode_layers.hip``) against plain torch in float64, and against itself with other numbers of workgroups."""

import json
import math

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
V, BLOCK = 64, 16


def make(H, L, ctx, seed=0):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s, k=1.0: (torch.randn(*s, generator=g) * k).to(torch.bfloat16).cuda()  # noqa: E731
    B, mb = len(ctx), max(ctx) // BLOCK + 2
    w = []
    for _ in range(L):
        w += [1 + r(H, k=0.1), r(H, k=0.1), r(3 * H, H, k=0.05), r(3 * H, k=0.1), r(H, H, k=0.03), r(H, k=0.1),
              1 + r(H, k=0.1), r(H, k=0.1), r(4 * H, H, k=0.03), r(4 * H, k=0.1), r(H, 4 * H, k=0.02), r(H, k=0.1)]
    w += [1 + r(H, k=0.1), r(H, k=0.1)]
    blocks = B * mb + 1
    bt = (1 + torch.randperm(B * mb, generator=g)).view(B, mb).int().cuda()
    k, v = r(L, blocks, BLOCK, H // 64, 64), r(L, blocks, BLOCK, H // 64, 64)
    pos = torch.tensor([c - 1 for c in ctx], dtype=torch.int32).cuda()
    slots = torch.tensor([int(bt[b, (c - 1) // BLOCK]) * BLOCK + (c - 1) % BLOCK for b, c in enumerate(ctx)]).cuda()
    return dict(ids=torch.randint(0, V, (B,), generator=g).cuda(), positions=pos, slots=slots, block_tables=bt,
                ctx_lens=torch.tensor(ctx, dtype=torch.int32).cuda(), table=r(V, H), pos_table=r(max(ctx), H), weights=w, k_cache=k, v_cache=v, eps=1e-5)


def plain(a):
    """The same in float64, K and V of the step's tokens rounded as the cache holds them; returns (rows, keys, values)."""
    w, H = [t.double() for t in a["weights"]], a["table"].shape[1]
    L, heads, ks, vs = (len(w) - 2) // 12, a["table"].shape[1] // 64, [], []
    x = a["table"].double()[a["ids"]] + a["pos_table"].double()[a["positions"].long()]
    for l in range(L):
        n1w, n1b, wqkv, bqkv, wo, bo, n2w, n2b, wu, bu, wd, bd = w[12 * l:12 * l + 12]
        q, k, v = (F.layer_norm(x, (H,), n1w, n1b, a["eps"]) @ wqkv.t() + bqkv).view(-1, 3, heads, 64).unbind(1)
        k, v, o = k.bfloat16().double(), v.bfloat16().double(), []
        ks.append(k), vs.append(v)
        for b, c in enumerate(a["ctx_lens"].tolist()):
            rows = (a["block_tables"][b].long()[:, None] * BLOCK + torch.arange(BLOCK, device="cuda")).reshape(-1)[:c - 1]
            kk = torch.cat([a["k_cache"][l].view(-1, heads, 64)[rows].double(), k[b:b + 1]])
            vv = torch.cat([a["v_cache"][l].view(-1, heads, 64)[rows].double(), v[b:b + 1]])
            o.append(torch.einsum("ht,thd->hd", torch.softmax(torch.einsum("hd,thd->ht", q[b], kk) / 8, -1), vv).reshape(-1))
        x = x + torch.stack(o) @ wo.t() + bo
        x = x + F.gelu(F.layer_norm(x, (H,), n2w, n2b, a["eps"]) @ wu.t() + bu, approximate="tanh") @ wd.t() + bd
    return F.layer_norm(x, (H,), w[-2], w[-1], a["eps"]), torch.stack(ks), torch.stack(vs)


def run(a, ws, **kw):
    from llmctl import ops

    b = dict(a, k_cache=a["k_cache"].clone(), v_cache=a["v_cache"].clone())
    out = ops.decode_layers(b["ids"], b["positions"], b["slots"], b["block_tables"], b["ctx_lens"], b["table"], b["pos_table"], b["weights"], b["k_cache"],
                            b["v_cache"], b["eps"], ws, **kw)
    return out, b["k_cache"], b["v_cache"]


# one row without a past, spans of 256 keys and one more, several spans' sums, rows of different lengths in groups of two and three, every width
@pytest.mark.parametrize("H,L,ctx", [(256, 2, [1]), (256, 1, [4001]), (768, 3, [129]), (768, 2, [257]), (768, 2, [258]), (768, 2, [2000, 1]), (512, 2, [17, 600, 1025]),
                                     (1024, 2, [5, 300, 1, 16]), (256, 2, [513, 512, 2, 33])])
def test_step_matches_float64(native_lib, H, L, ctx):
    """Against float64.  What is rounded: K, V, the MLP's activations (bf16, 2^-9 each) and the result (2^-9); every layer's come on top of the former ones'."""
    from llmctl import ops

    a = make(H, L, ctx)
    ws = ops.decode_layers_workspace(H, "cuda")
    want, ks, vs = plain(a)
    first = None
    for step in range(3):  # (the workspace carries its count on)
        out, k, v = run(a, ws)
        torch.cuda.synchronize()
        assert (out.double() - want).norm() <= (1 + L) * 2.0 ** -8 * want.norm()
        rows = a["slots"].long()
        for got, new, old in ((k, ks, a["k_cache"]), (v, vs, a["v_cache"])):
            flat = got.view(L, -1, H // 64, 64)
            assert (flat[:, rows].double() - new).norm() <= L * 2.0 ** -8 * new.norm()
            keep = torch.ones(flat.shape[1], dtype=torch.bool, device="cuda")
            keep[rows] = False
            assert torch.equal(flat[:, keep], old.view(L, -1, H // 64, 64)[:, keep])  # nothing else is written
        first = first if first is not None else (out, k, v)
        assert all(torch.equal(x, y) for x, y in zip(first, (out, k, v)))


@pytest.mark.parametrize("workgroups,gate_us", [(1, 200), (7, 200), (127, 200), (128, 0), (128, 1)])
@pytest.mark.parametrize("ctx", [[300], [40, 1, 700]])
def test_any_number_of_workgroups(native_lib, workgroups, gate_us, ctx):
    """Shares that go round, and a gate that closes before all are there, give the same bits; so does a graph, replayed beside other work."""
    from llmctl import ops

    a = make(256, 2, ctx, seed=1)
    ws = ops.decode_layers_workspace(256, "cuda")
    want = run(a, ws)
    for _ in range(4):
        got = run(a, ws, workgroups=workgroups, gate_us=gate_us)
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(want, got))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        got = run(a, ws, workgroups=workgroups, gate_us=gate_us)
    for _ in range(4):
        got[0].zero_()
        g.replay()
        assert torch.equal(got[0], want[0])
        run(a, ws)


def test_rows_without_a_slot_are_not_cached(native_lib):
    from llmctl import ops

    a = make(256, 1, [20, 1], seed=2)
    a["slots"] = torch.tensor([int(a["slots"][0]), -1], device="cuda")
    _, k, _ = run(a, ops.decode_layers_workspace(256, "cuda"))
    assert int((k != a["k_cache"]).any(-1).any(-1).sum()) == 1


def test_what_it_does_not_take(native_lib):
    from llmctl import ops

    cache = torch.zeros(1, 1, 1, 1, 64, dtype=torch.bfloat16, device="cuda")
    ok = lambda *a, c=cache: ops.decode_layers_ok(*a, c)  # noqa: E731
    assert ok(768, 12, 12, 3072, 12, 4) and not ok(768, 12, 12, 3072, 12, 5) and not ok(768, 12, 4, 3072, 12, 1) and not ok(768, 6, 6, 3072, 12, 1)
    assert not ok(1280, 20, 20, 5120, 12, 1) and not ok(768, 12, 12, 2048, 12, 1) and not ok(768, 12, 12, 3072, 33, 1)
    a = make(256, 1, [3])
    with pytest.raises(RuntimeError):
        run(dict(a, weights=a["weights"][:-1]), ops.decode_layers_workspace(256, "cuda"))
    with pytest.raises(RuntimeError):
        run(a, ops.decode_layers_workspace(512, "cuda"))
    assert math.isfinite(float(run(a, ops.decode_layers_workspace(256, "cuda"))[0].float().sum()))


def _count(ws, base):
    """The layers that a workspace has counted (second word, low half; the high one is zero between steps)."""
    ws[1] = base


def _fits(a, got):
    want, ks, _ = plain(a)
    assert float((got[0].double() - want).norm()) <= (1 + len(ks)) * 2.0 ** -8 * float(want.norm())
    new = run(a, torch.zeros_like(a["ws"]))  # a workspace that has seen no step
    assert all(torch.equal(x, y) for x, y in zip(got, new))


@pytest.mark.parametrize("L", [2, 3, 5])
@pytest.mark.parametrize("bits", [16, 32])
def test_words_that_narrower_steps_left_are_not_taken(native_lib, L, bits):
    """Two rows, then so many steps of one row (counted, not run, but for the last) that the next first layer's count ends in the bits of a word that the second row
    left; then two rows of other tokens."""
    from llmctl import ops

    two, one, other = (make(256, L, ctx, seed=s) for s, ctx in ((1, [40, 30]), (2, [21]), (3, [33, 600])))
    for last in range(1, L + 1):  # whichever layer's word it were
        two["ws"] = one["ws"] = other["ws"] = ws = ops.decode_layers_workspace(256, "cuda")
        run(two, ws)
        _count(ws, ((1 << bits) + last - 1 - L) & 0xffffffff)
        _fits(one, run(one, ws))
        _fits(other, run(other, ws))


@pytest.mark.parametrize("start", [0, 65536 - 14, (1 << 32) - 14])
def test_rows_and_spans_come_and_go_on_one_workspace(native_lib, start):
    """Steps of 4, 1, 2 .. rows, one span of keys and several, the count past 16 and past 32 bits on the way."""
    from llmctl import ops

    ws = ops.decode_layers_workspace(256, "cuda")
    steps = [dict(make(256, 3, ctx, seed=i), ws=ws) for i, ctx in enumerate(([20, 3, 700, 1], [1500], [9, 40], [5], [2000, 300, 7, 64], [11, 800]))]
    for turn in range(2):
        for i, a in enumerate(steps):
            if turn and not i:
                _count(ws, start)
            _fits(a, run(a, ws))


@pytest.mark.parametrize("ctx,bad", [([20], range(19)), ([700, 5], range(0, 8)), ([300], [270])])
def test_keys_that_are_not_numbers_come_through(native_lib, ctx, bad):
    """A key row of NaN makes its head's scores NaN: the row's result shows it, whichever lanes read it, and the other row's does not."""
    from llmctl import ops

    a = make(256, 1, ctx)
    for t in bad:
        a["k_cache"][0, int(a["block_tables"][0, t // BLOCK]), t % BLOCK] = float("nan")
    out = run(a, ops.decode_layers_workspace(256, "cuda"))[0]
    assert bool(torch.isnan(out[0]).all()) and bool(torch.isfinite(out[1:]).all())


def engine(tmp_path, knob=True, graphs=True, **kw):
    from llmctl.serve.engine import InferenceEngine

    f = tmp_path / "model.json"
    f.write_text(json.dumps({"name": "narrow", "arch": "decoder-only", "layers": 3, "hidden": 256, "ffn": 1024, "heads": 4, "vocab_size": 512, "norm": "layernorm",
                             "activation": "gelu", "position": "learned", "max_position_embeddings": 512, **kw}))
    return InferenceEngine(str(f), device="cuda", max_batch_size=4, num_kv_blocks=128, block_size=BLOCK, max_model_len=512, use_graphs=graphs, seed=5,
                           perf_knobs={"decode_layers": knob})


def steps(eng, prompts, n=4, change=None):
    """The logits of a prompt's last token and of n decode steps of fixed tokens, the sequences' caches made by the engine."""
    from llmctl.serve.scheduler import PrefillChunk

    seqs = [eng.open_sequence(p) for p in prompts]
    out = [eng.prefill([PrefillChunk(s, 0, len(s.prompt_ids)) for s in seqs]).float().clone()]
    if change is not None:
        change(eng)
    for i in range(n):
        for s in seqs:
            s.output_ids.append(7 * i + len(s.prompt_ids))
            s._decode_slot = eng.kv.append_token(s.seq_id)
        out.append(eng.decode(seqs).float().clone())
    return out


def off_16_bytes(t):
    u = torch.empty(t.numel() + 4, dtype=t.dtype, device=t.device)[4:].view(t.shape)
    return torch.nn.Parameter(u.copy_(t.detach()), requires_grad=False)


@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("what", ["as it is", "wider heads", "narrower heads", "embedding off 16 bytes", "positions off 16 bytes"])
def test_engine_takes_what_it_took(native_lib, tmp_path, graphs, what):
    """Through the engine's own rule: a model that fits gives the chain's logits to rounding, one that does not (heads that are not hidden / heads wide, tables that the
    kernel cannot read in 16 bytes) runs the chain, bit for bit."""
    kw = {"wider heads": dict(head_dim=128), "narrower heads": dict(head_dim=64, hidden=512, ffn=2048)}.get(what, {})

    def change(eng):
        if what == "embedding off 16 bytes":
            eng.model.embed = off_16_bytes(eng.model.embed)
        elif what == "positions off 16 bytes":
            eng.model.pos_embed = off_16_bytes(eng.model.pos_embed)

    outs, taken = [], []
    for knob in (True, False):
        eng = engine(tmp_path, knob, graphs, **kw)
        outs.append(steps(eng, [list(range(3, 40)), list(range(5, 9))], change=change))
        taken.append(eng._one_launch(2))
        eng.close()
    assert taken == [what == "as it is", False]
    for x, y in zip(*outs):
        if taken[0]:
            assert float((x - y).norm()) <= 3 * 2.0 ** -7 * float(y.norm())  # the chain rounds its rows between launches, three layers of them
        else:
            assert torch.equal(x, y)


@pytest.mark.parametrize("graphs", [False, True])
def test_steps_on_two_streams(native_lib, tmp_path, graphs):
    """Eager steps of one engine, or its graphs of one row and of two, on two streams at a time: each has words of its own."""
    eng = engine(tmp_path, graphs=graphs)
    steps(eng, [[1, 2]], n=0)
    seqs = [eng.open_sequence(list(range(2, n))) for n in (30, 50, 400)]
    with torch.inference_mode():
        eng.kv_cache.k.normal_(), eng.kv_cache.v.normal_()
    for s in seqs:
        s._decode_slot = int(eng.kv.slots(s.seq_id, s.num_tokens - 1, 1)[0])
    parts = (seqs[:1], seqs[1:])
    want = [eng.decode(p).clone() for p in parts]
    streams = [torch.cuda.Stream() for _ in parts]
    torch.cuda.synchronize()
    for _ in range(20):
        got = []
        for s, p in zip(streams, parts):
            with torch.cuda.stream(s):
                got.append(eng.decode(p).clone())
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(got, want))
    eng.close()


def test_steps_beside_a_full_chip(native_lib):
    """Steps that start while another stream's attention holds nearly every CU do not go through with the few workgroups that run (one takes 7.7 ms, all 0.2): the
    attention's launches are 0.7 ms."""
    from llmctl import ops

    q, k, v = (torch.randn(4, 4096, 32, 128, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    a, ws, side = make(768, 12, [129]), ops.decode_layers_workspace(768, "cuda"), torch.cuda.Stream()
    run(a, ws), ops.flash_attention(q, k, v)
    torch.cuda.synchronize()
    took = []
    for _ in range(20):
        with torch.cuda.stream(side):
            for _ in range(20):
                ops.flash_attention(q, k, v)
        for _ in range(6):
            ev = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            ev[0].record()
            ops.decode_layers(*(a[n] for n in ("ids", "positions", "slots", "block_tables", "ctx_lens", "table", "pos_table", "weights", "k_cache", "v_cache", "eps")), ws)
            ev[1].record()
            ev[1].synchronize()
            took.append(ev[0].elapsed_time(ev[1]))
        side.synchronize()
    assert max(took) < 2.5, sorted(took)[-5:]


def test_a_lost_step_is_told(native_lib, tmp_path, monkeypatch):
    """A step whose waits run out (of one try here) ends with NaN rows and sets the host's word; the workspace serves the next one.  Through an engine: whoever asks for
    its tokens, or for the next step, is told, once."""
    import functools

    from llmctl import ops
    from llmctl.serve.scheduler import SamplingParams

    a, ws, lost = make(256, 2, [40, 9]), ops.decode_layers_workspace(256, "cuda"), torch.zeros(1, dtype=torch.int32, pin_memory=True)
    want = run(a, ws, lost=lost)
    torch.cuda.synchronize()
    assert int(lost) == 0
    out = run(a, ws, lost=lost, spins=1)[0]
    torch.cuda.synchronize()
    assert bool(torch.isnan(out).all()) and int(lost) == 1
    lost.zero_()
    got = run(a, ws, lost=lost)
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip(got, want)) and int(lost) == 0
    with pytest.raises(RuntimeError):
        run(a, ws, lost=torch.zeros(1, dtype=torch.int32))  # not pinned: no kernel could write it

    eng = engine(tmp_path, graphs=False)
    steps(eng, [[1, 2, 3]], n=2)
    seq = eng.open_sequence([5, 6, 7])
    seq._decode_slot = int(eng.kv.slots(seq.seq_id, 2, 1)[0])
    whole, short = ops.decode_layers, functools.partial(ops.decode_layers, spins=1)
    for ask in (lambda x: eng.sample(x, [seq]), lambda x: (torch.cuda.synchronize(), eng.decode([seq]))):
        monkeypatch.setattr(ops, "decode_layers", short)
        logits = eng.decode([seq])
        monkeypatch.setattr(ops, "decode_layers", whole)
        with pytest.raises(RuntimeError, match="lost"):
            ask(logits)
        assert bool(torch.isfinite(eng.decode([seq])).all())
    eng.scheduler.finish(seq, "stop")
    eng.add_request([4, 5, 6], SamplingParams(max_tokens=8, temperature=0.0))
    monkeypatch.setattr(ops, "decode_layers", short)
    with pytest.raises(RuntimeError, match="lost"):  # the step after it is under way by then, with its tokens
        for _ in range(4):
            eng.step()
    monkeypatch.setattr(ops, "decode_layers", whole)
    torch.cuda.synchronize()
    eng.close()

"""The work that users have this framework do, as measured cases: training steps, prompt (prefill) steps and
decode steps through the public engines (``TrainingEngine.train_step``, ``InferenceEngine.prefill`` / ``decode`` /
``forward_portions``), from a 2 x 128-token step of the test model to layers of GPT-7B and of three
hybrid families at the sizes of ``llmctl.benchmarks.hybrid``.  Depth is cut (the layers of one model are alike);
widths, heads, experts, vocabulary and sequence lengths are the real ones.

A case: ``kind`` (``train`` / ``prefill`` / ``decode``), ``model`` and sizes.  ``exact`` computes the same results
from the same inputs (weights, tokens, cache contents) in plain torch, float64.
"""

from __future__ import annotations

import dataclasses
import json
import math
import tempfile
from pathlib import Path

import torch
import torch.nn.functional as F

F64 = torch.float64
DENSE = ("tiny", "gpt2-125m", "gpt-7b")  # transformer templates; the others are hybrid families
BLOCK = 16  # tokens per cache block, the engine's default


def listed():
    return [
        # the smallest training step: the test / smoke model, where launches and host time count
        dict(name="train tiny", kind="train", model="tiny", layers=2, batch=2, seq=128),
        # the small GPT-2 style model (LayerNorm, GELU, learned positions, tied embeddings) at its usual length
        dict(name="train gpt2-125m", kind="train", model="gpt2-125m", layers=12, batch=8, seq=1024),
        # the flagship: GPT-7B layers at the training length
        dict(name="train gpt-7b layers", kind="train", model="gpt-7b", layers=2, batch=4, seq=2048),
        # time to first token: one 2048-token prompt
        dict(name="prefill gpt-7b 2048", kind="prefill", model="gpt-7b", layers=4, prompts="2048"),
        # the smallest call: one sequence of the small model, short context, one token
        dict(name="decode gpt2-125m x1", kind="decode", model="gpt2-125m", layers=12, batch=1, context=129),
        # steady serving: 16 sequences at 2k context
        dict(name="decode gpt-7b x16", kind="decode", model="gpt-7b", layers=4, batch=16, context=2048),
        # latent attention + mLSTM + group-limited experts, one prompt (the benchmark's medium size)
        dict(name="prefill lenitar 2048", kind="prefill", model="lenitar", width=2048, layers=4, prompts="2048"),
        dict(name="decode lenitar x16", kind="decode", model="lenitar", width=2048, layers=4, batch=16, context=2048),
        # gated linear attention + sigmoid attention + routed experts, a ragged packed batch of prompts
        dict(name="prefill malinex ragged", kind="prefill", model="malinex", width=2048, layers=3, prompts="1417,33,700,250,511"),
        dict(name="decode malinex x16", kind="decode", model="malinex", width=2048, layers=3, batch=16, context=2048),
        # windowed attention beside gated delta rule, Mamba-2, retention; ragged pair of prompts, and decode
        dict(name="prefill dumazen ragged", kind="prefill", model="dumazen", width=2048, layers=6, prompts="2048,1331"),
        dict(name="decode dumazen x16", kind="decode", model="dumazen", width=2048, layers=6, batch=16, context=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("train", "prefill", "prefill", "decode", "decode"))
    if kind == "train":
        model = rng.choice(("tiny", "gpt2-125m", "gpt-7b"))
        layers = {"tiny": 2, "gpt2-125m": 12, "gpt-7b": rng.randint(1, 2)}[model]
        seq = _log_int(rng, 64, 512 if model == "tiny" else 2048)
        if rng.random() < 0.5:  # the usual multiples beside odd lengths
            seq = max(64, seq // 64 * 64)
        most = 4096 if model == "tiny" else 8192
        return dict(kind=kind, model=model, layers=layers, batch=_log_int(rng, 1, max(1, min(8, most // seq))), seq=seq)
    model = rng.choice(("gpt2-125m", "gpt-7b", "lenitar", "malinex", "dumazen"))
    case = dict(kind=kind, model=model, layers={"gpt2-125m": 12, "gpt-7b": 4, "lenitar": 4, "malinex": 3, "dumazen": 6}[model])
    if model not in DENSE:
        case["width"] = rng.choice((1024, 2048))
    if kind == "prefill":
        n = rng.choice((1, 1, 2, 3, 5, 8))
        lens = [_log_int(rng, 16, 2047) for _ in range(n)]
        while sum(lens) > 4096:
            lens.pop()
        case["prompts"] = ",".join(str(v) for v in lens)
    else:
        case.update(batch=_log_int(rng, 1, 32), context=_log_int(rng, 17, 2048 if model == "gpt2-125m" else 4000) - 1)
    return case


# ------------------------------------------------------------------ what a user's program has in hand
def _prompts(case):
    return [int(v) for v in str(case["prompts"]).split(",")]


def _longest(case):
    return (max(_prompts(case)) if case["kind"] == "prefill" else int(case["context"])) + 8


def _config(case):
    """The model's configuration: the named template with this case's depth (hybrid: the benchmark's sizes)."""
    from llmctl.models import get_model_config

    m, n = case["model"], int(case["layers"])
    if m in DENSE:
        return dataclasses.replace(get_model_config(m), layers=n)
    w = int(case["width"])
    kw = dict(width=w, layers=n, heads=w // 128, vocab=32000)
    if m == "lenitar":
        from llmctl.models.lenitar import lenitar_template

        cfg = lenitar_template(every=4, experts=8, top=2, groups=2, keep=1, ff=w // 2, window=1024, **kw)
    elif m == "malinex":
        from llmctl.models.malinex import malinex_template

        cfg = malinex_template(kv_heads=w // 512, every=3, experts=8, top=2, expert_ff=w // 2, head_dim=128,
                               max_positions=4096, **kw)
    else:
        from llmctl.models.dumazen import dumazen_template

        cfg = dumazen_template(kv_heads=w // 512, every=3, ff=4 * w, head_dim=128, window=1024, **kw)
    cfg.max_position_embeddings = 4096
    return cfg


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _vectors(model, g):
    """Vectors (norm weights, biases, gates) as training leaves them: not all at their initial values."""
    with torch.no_grad():
        for name, p in model.named_parameters():
            if p.dim() != 1:
                continue
            r = torch.randn(p.shape, generator=g, device="cuda", dtype=torch.float32)
            if name.endswith("dist_a") or name.endswith("dist_b"):  # a distance penalty is a penalty
                p.copy_((0.02 + 0.1 * r.abs()).to(p.dtype))
            elif name.endswith("dt_bias"):  # steps well below one
                p.copy_((-2.0 + 0.5 * r).to(p.dtype))
            else:
                p.add_((0.1 * r).to(p.dtype))


def _specialise(model, cfg, g):
    """Routers that know their tokens, as trained ones do: every token's embedding carries the directions of two experts of
    one half, which the router's rows read.  With random routers a few tokens in a hundred sit on a tie between two experts, and
    bf16 rounding alone decides what they run."""
    W, scale = cfg.hidden, float(getattr(cfg, "embedding_scale", 1.0))
    routers = [m.w_router for m in model.modules() if hasattr(m, "w_router")]
    if not routers:
        return
    E, V = routers[0].shape[0], cfg.vocab_size
    u = torch.linalg.qr(torch.randn(W, E, generator=g, device="cuda"))[0].t()  # orthonormal rows
    first = torch.randint(0, E, (V,), generator=g, device="cuda")
    half = E // 2
    second = first // half * half + (first % half + torch.randint(1, half, (V,), generator=g, device="cuda")) % half
    with torch.no_grad():
        rows = model.embed.float() / model.embed.float().std() + 20.0 * (u[first] + 0.9 * u[second])
        model.embed.copy_((rows / scale).to(model.embed.dtype))
        for w in routers:
            w.mul_(0.1).add_(0.2 * u)


def _serving_engine(case, seed):
    from llmctl.serve.engine import InferenceEngine

    cfg = _config(case)
    with tempfile.TemporaryDirectory(prefix="llmctl_cases_") as d:
        path = Path(d) / "model.json"
        path.write_text(json.dumps(cfg.to_dict()))
        lens = _prompts(case) if case["kind"] == "prefill" else [int(case["context"])] * int(case["batch"])
        blocks = sum((n + 1 + BLOCK - 1) // BLOCK for n in lens) + 1
        eng = InferenceEngine(str(path), device="cuda", max_batch_size=len(lens), max_batch_tokens=1 << 20,
                              max_model_len=min(_longest(case), cfg.max_position_embeddings), block_size=BLOCK,
                              num_kv_blocks=blocks, prefix_caching=False, seed=int(seed))
    if eng.hybrid:
        _vectors(eng.model, _gen(seed + 1))
        _specialise(eng.model, cfg, _gen(seed + 2))
        with torch.device("cuda"):
            eng.model.load_named(eng.model.export_named())  # what a checkpoint holds: rows without a bias have none
    return eng, lens


def prepare(case, seed):
    g = _gen(seed)
    if case["kind"] == "train":
        from llmctl.runtime.engine import TrainingConfig, TrainingEngine

        cfg = _config(case)
        eng = TrainingEngine(TrainingConfig(
            model_name_or_path=case["model"], batch_size=int(case["batch"]), seq_len=int(case["seq"]), learning_rate=3e-4,
            weight_decay=0.1, scheduler="cosine", max_steps=1000, gradient_clipping=1.0, mixed_precision="bf16",
            device="cuda", seed=int(seed), log_level="warning"), cfg)
        ids = torch.randint(0, cfg.vocab_size, (int(case["batch"]), int(case["seq"]) + 1), generator=g, device="cuda")
        return dict(kind="train", eng=eng, batch=(ids[:, :-1].contiguous(), ids[:, 1:].contiguous()))
    eng, lens = _serving_engine(case, seed)
    V = eng.cfg.vocab_size
    ids = [torch.randint(0, V, (n,), generator=g, device="cuda").tolist() for n in lens]
    st = dict(kind=case["kind"], eng=eng, ids=ids)
    if case["kind"] == "prefill":
        # hybrid families: logits at up to 64 places of every prompt (scoring); the transformer: of the next tokens
        st["want"] = [sorted({n * (i + 1) // min(n, 64) - 1 for i in range(min(n, 64))}) for n in lens] if eng.hybrid else None
        return st
    # decode: every sequence's earlier tokens are in the cache; the next step runs its last token
    st["seqs"] = [eng.open_sequence(t) for t in ids]
    for s in st["seqs"]:
        s._decode_slot = int(eng.kv.slots(s.seq_id, s.num_tokens - 1, 1)[0])
    eng.decode(st["seqs"])  # a serving program's warm-up (captures the step where the engine does so)
    with torch.inference_mode():
        for t in _cache_tensors(eng):
            t.copy_(torch.randn(t.shape, generator=g, device="cuda", dtype=torch.float32) * (1.0 if t.dtype == torch.bfloat16 else 0.3))
    return st


def _cache_tensors(eng):
    """The tensors of the engine's cache, pools of rows and of states, layer by layer."""
    if not eng.hybrid:
        return [eng.kv_cache.k, eng.kv_cache.v]
    out = []
    for i in range(len(eng.kv_cache._layers)):
        e = eng.kv_cache.layer(i)
        for t in e if isinstance(e, tuple) else (e,):
            out += list(t) if isinstance(t, tuple) else [t]
    return out


def _open(eng, ids):
    return [eng.open_sequence(t) for t in ids]


def _finish(eng, seqs):
    for s in reversed(seqs):
        eng.scheduler.finish(s, "stop")


def run(state):
    eng = state["eng"]
    if state["kind"] == "train":
        out = eng.train_step([state["batch"]])
        o = eng.optimizer
        # the second moment is the square of what the first one shows (and moves the next pass's weights)
        return {"loss": out["loss"], "grad_norm": out["grad_norm"], "master": o.master, "exp_avg": o.exp_avg}
    if state["kind"] == "decode":
        logits = eng.decode(state["seqs"])
        return {"logits": logits, "states": [t for t in _cache_tensors(eng) if t.dtype == torch.float32] if eng.hybrid else []}
    from llmctl.serve.scheduler import PrefillChunk

    seqs = _open(eng, state["ids"])
    portions = [PrefillChunk(s, 0, s.num_tokens) for s in seqs]
    logits = eng.forward_portions(portions, state["want"]) if eng.hybrid else eng.prefill(portions)
    _finish(eng, seqs)
    return {"logits": logits, "cache": _cache_tensors(eng)}


# ------------------------------------------------------------------ what a pass cannot do without
def _shape(case):
    """(configuration, weights of the model, weights that one token multiplies, those of the head)."""
    with torch.device("meta"):
        cfg = _config(case)
        if case["model"] in DENSE:
            from llmctl.models import build_model

            model = build_model(cfg, device="meta")
        else:
            from llmctl.models.registry import family_of_config

            model = family_of_config(cfg).build(cfg, device="meta", dtype=torch.bfloat16, seed=0)
    total = used = 0
    for n, p in model.named_parameters():
        if p.dim() < 2 or n in ("pos_embed", "pos"):
            continue
        if n == "embed" and not cfg.tie_word_embeddings:
            continue
        total += p.numel()
        expert = ".experts_" in n or (case["model"] == "malinex" and n.endswith((".ff.w_up", ".ff.w_down")))
        used += p.numel() // 4 if expert else p.numel()  # two of eight experts
    return cfg, total, used, cfg.vocab_size * cfg.hidden


def work(case):
    cfg, total, used, head = _shape(case)
    m, W, n = case["model"], cfg.hidden, int(case["layers"])
    att = {"lenitar": n - n // 4, "malinex": n // 3, "dumazen": n // 3}.get(m, n)  # layers that attend
    kv = cfg.kv_heads * cfg.head_dim if m in DENSE else W // 4  # columns of keys (and of values) of a token
    if case["kind"] == "train":
        T, S = int(case["batch"]) * int(case["seq"]), int(case["seq"])
        flops = 6.0 * used * T + 6.0 * T * S * W * att
        # weights (read twice, bf16), gradients (written, read), master and moments (read, written), activations
        return {"bytes": float(total * (2 * 2 + 2 * 2 + 2 + 24) + T * (W * n * 16 + 2 * cfg.vocab_size)), "flops": flops}
    if case["kind"] == "prefill":
        lens = _prompts(case)
        T = sum(lens)
        rows = len(lens) if m in DENSE else sum(min(v, 64) for v in lens)
        flops = 2.0 * (used - head) * T + 2.0 * head * rows + sum(2.0 * v * min(v, 1024 if m in ("lenitar", "dumazen") else v) * W for v in lens) * att
        return {"bytes": float(2 * total + T * (2 * 2 * kv * att + 6 * W) + 4 * rows * cfg.vocab_size), "flops": flops}
    B, C = int(case["batch"]), int(case["context"])
    C = min(C, 1024) if m in ("lenitar", "dumazen") else C
    touched = min(1.0, 1.0 - 0.75 ** B)  # share of the experts that B tokens reach
    weights = used + (total - used) * (touched * 4 - 1) / 3 if total > used else total
    state = 0 if m in DENSE else (n - att + (att if m == "dumazen" else 0)) * (W // 128) * 64 * 128 * 8
    return {"bytes": float(2 * weights + B * (2 * 2 * C * kv * att + state + 4 * cfg.vocab_size)),
            "flops": 2.0 * used * B + 4.0 * B * C * W * att}


def tolerance(case):
    """bf16 activations through all layers: 0.005 to 0.02 off ``exact``, so two correct forms are up to 0.03 apart."""
    return {"rel": 0.03}


# ------------------------------------------------------------------ the same in plain torch, float64
def _rms(x, eps):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps)


def _ln(x, w, b, eps):
    return F.layer_norm(x, (x.shape[-1],), w, b, eps)


def _turn(x, pos, freq):
    """Rotary on half pairs of the first 2 * len(freq) entries; x [T, heads, d], pos [T]."""
    h = freq.shape[0]
    a = pos.to(F64)[:, None] * freq
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    u, v = x[..., :h], x[..., h:2 * h]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * h:]], -1)


def _freq(base, dims):
    return float(base) ** (-2.0 * torch.arange(dims // 2, dtype=F64, device="cuda") / dims)


def _scores(q, k, scale, first=0):
    """[G, r, Tq, Tk] scores of grouped heads and the distances i - j; query 0 sits at position ``first``."""
    Tq, H, d = q.shape
    G = k.shape[1]
    s = torch.matmul(q.transpose(0, 1).reshape(G, H // G, Tq, d), k.permute(1, 2, 0)[:, None].contiguous()) * scale
    dist = torch.arange(first, first + Tq, device="cuda")[:, None] - torch.arange(k.shape[0], device="cuda")[None]
    return s, dist


def _attend(w, v):
    """w [G, r, Tq, Tk], v [Tk, G, dv] -> [Tq, H, dv]."""
    o = torch.matmul(w, v.transpose(0, 1)[:, None].contiguous())
    return o.flatten(0, 1).transpose(0, 1)


def _softmax_attention(q, k, v, scale, first=0, window=None, sink=None):
    s, dist = _scores(q, k, scale, first)
    s = s.masked_fill((dist < 0) | (dist >= (window or 1 << 40)), -math.inf)
    if sink is not None:
        g = sink.view(s.shape[0], s.shape[1], 1, 1).expand(-1, -1, s.shape[2], 1)
        return _attend(torch.softmax(torch.cat([s, g], -1), -1)[..., :-1], v)
    return _attend(torch.softmax(s, -1), v)


# ---- the transformer
def _dense_layer(cfg, P, p, x, pos, past=None, attend=None):
    """One block on x [T, h]; returns (x, k, v).  ``past`` = (k, v) of the earlier tokens; ``attend(q, k, v)`` replaces the
    causal attention of one sequence."""
    T, D, eps = x.shape[0], cfg.head_dim, cfg.layer_norm_eps
    b = lambda n: P[p + n] if p + n in P else None
    norm = lambda y, n: (_ln(y, P[p + n + "_w"], P[p + n + "_b"], eps) if cfg.norm == "layernorm" else _rms(y, eps) * P[p + n + "_w"])
    z = F.linear(norm(x, "attn_norm"), P[p + "wqkv"], b("bqkv")).view(T, -1, D)
    q, k, v = z.split([cfg.heads, cfg.kv_heads, cfg.kv_heads], 1)
    if cfg.position == "rope":
        f = _freq((cfg.rope or {}).get("base", 10000), D)
        q, k = _turn(q, pos, f), _turn(k, pos, f)
    if past is not None:
        o = _softmax_attention(q, torch.cat([past[0], k]), torch.cat([past[1], v]), D ** -0.5, past[0].shape[0])
    elif attend is not None:
        o = attend(q, k, v)
    else:
        o = _softmax_attention(q, k, v, D ** -0.5)
    x = x + F.linear(o.reshape(T, -1), P[p + "wo"], b("bo"))
    h = norm(x, "mlp_norm")
    u = F.linear(h, P[p + "w_up"], b("b_up"))
    if cfg.gated_mlp:
        gate, up = u.chunk(2, -1)
        u = F.silu(gate) * up
    else:
        u = F.gelu(u, approximate="tanh")
    return x + F.linear(u, P[p + "w_down"], b("b_down")), k, v


def _dense_head(cfg, P, x):
    eps = cfg.layer_norm_eps
    x = _ln(x, P["final_norm_w"], P["final_norm_b"], eps) if cfg.norm == "layernorm" else _rms(x, eps) * P["final_norm_w"]
    return x @ (P["embed"] if cfg.tie_word_embeddings else P["lm_head"]).t()


def _dense_embed(P, ids, pos):
    x = P["embed"][ids]
    return x + P["pos_embed"][pos] if "pos_embed" in P else x


def _exact_train(case, st):
    eng = st["eng"]
    cfg, c = eng.model_config, eng.config
    P = {n: p.detach().to(F64).requires_grad_(True) for n, p in eng.model.named_parameters()}
    ids, labels = st["batch"]
    B, S = ids.shape
    pos = torch.arange(S, device="cuda").repeat(B)

    def attend(q, k, v):
        one = lambda t: t.view(B, S, t.shape[1], t.shape[2])
        return torch.cat([_softmax_attention(a, b, d, cfg.head_dim ** -0.5) for a, b, d in zip(one(q), one(k), one(v))])

    x = _dense_embed(P, ids.reshape(-1), pos)
    for i in range(cfg.layers):
        x = _dense_layer(cfg, P, f"layers.{i}.", x, pos, attend=attend)[0]
    loss = F.cross_entropy(_dense_head(cfg, P, x), labels.reshape(-1))
    grads = dict(zip(P, torch.autograd.grad(loss, list(P.values()))))
    norm = torch.sqrt(sum(v.square().sum() for v in grads.values()))
    coef = min(1.0, c.gradient_clipping / (float(norm) + 1e-6))
    flat, o = eng.flat, eng.optimizer
    out = {k: torch.zeros(o.master.numel(), dtype=F64, device="cuda") for k in ("master", "exp_avg")}
    for name, p in eng.model.named_parameters():
        at = slice(flat.offsets[id(p)], flat.offsets[id(p)] + p.numel())
        gr, w = grads.pop(name).reshape(-1) * coef, P[name].detach().reshape(-1)
        decay = c.weight_decay if p.dim() > 1 else 0.0
        out["exp_avg"][at] = (1 - c.betas[0]) * gr
        out["master"][at] = w * (1.0 - c.learning_rate * decay) - c.learning_rate * gr / (gr.abs() + c.eps)
    return {"loss": loss.detach(), "grad_norm": norm.reshape(o.last_grad_norm.shape if o.last_grad_norm is not None else (1,)), **out}


def _exact_dense_serving(case, st):
    eng = st["eng"]
    cfg = eng.cfg
    P = {n: p.detach().to(F64) for n, p in eng.model.named_parameters()}
    kc, vc = eng.kv_cache.k, eng.kv_cache.v
    L, KV, D = cfg.layers, cfg.kv_heads, cfg.head_dim
    flat = lambda t: t.view(L, -1, KV, D)
    rows = []
    if case["kind"] == "decode":
        for s in st["seqs"]:
            n = s.num_tokens - 1
            at = torch.from_numpy(eng.kv.slots(s.seq_id, 0, n).astype("int64")).cuda()
            pos = torch.tensor([n], device="cuda")
            x = _dense_embed(P, torch.tensor([s.all_ids[n]], device="cuda"), pos)
            for i in range(L):
                x = _dense_layer(cfg, P, f"layers.{i}.", x, pos, past=(flat(kc)[i, at].to(F64), flat(vc)[i, at].to(F64)))[0]
            rows.append(_dense_head(cfg, P, x))
        return {"logits": torch.cat(rows), "states": []}
    K, Vv = flat(torch.zeros_like(kc, dtype=F64)), flat(torch.zeros_like(vc, dtype=F64))
    for s, t in zip(_open(eng, st["ids"]), st["ids"]):
        at = torch.from_numpy(eng.kv.slots(s.seq_id, 0, len(t)).astype("int64")).cuda()
        pos = torch.arange(len(t), device="cuda")
        x = _dense_embed(P, torch.tensor(t, device="cuda"), pos)
        for i in range(L):
            x, k, v = _dense_layer(cfg, P, f"layers.{i}.", x, pos)
            K[i, at], Vv[i, at] = k, v
        rows.append(_dense_head(cfg, P, x[-1:]))
    return {"logits": torch.cat(rows), "cache": [K.view(kc.shape), Vv.view(vc.shape)]}


# ---- the hybrid families: W = tensors by checkpoint name, ``past`` = (rows of the earlier tokens or None, states or None)
def _lin(W, n, h):
    y = h @ W[n].t()
    return y + W[n + ".b"] if n + ".b" in W else y


def _conv(u, w, bias, before):
    """Causal convolution per channel; ``before`` [taps - 1, channels] are the inputs ahead of the first row."""
    ext, taps = torch.cat([before, u]), w.shape[1]
    y = sum(w[:, j] * ext[j:j + u.shape[0]] for j in range(taps))
    return (y if bias is None else y + bias), ext[-(taps - 1):]


def _latent(W, p, m, h, eps, pos, past):
    T, H, dn, dr, dv, rk = h.shape[0], m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
    f = _freq(m["rot"]["base"], m["rot"]["dims"])
    q = ((_rms(h @ W[p + "dq"].t(), eps) * W[p + "dq.norm"]) @ W[p + "uq"].t()).view(T, H, dn + dr)
    q = torch.cat([q[..., :dn], _turn(q[..., dn:], pos, f)], -1)
    d = h @ W[p + "dkv"].t()
    new = torch.cat([_rms(d[:, :rk], eps) * W[p + "dkv.norm"], _turn(d[:, None, rk:], pos, f)[:, 0]], -1)
    rows = new if past[0] is None else torch.cat([past[0], new])
    n = rows.shape[0]
    k = torch.cat([(rows[:, :rk] @ W[p + "uk"].t()).view(n, H, dn), rows[:, None, rk:].expand(-1, H, -1)], -1)
    v = (rows[:, :rk] @ W[p + "uv"].t()).view(n, H, dv)
    o = _softmax_attention(q, k, v, m["scale"], n - T, m["mask"]["size"], W[p + "sink"]).reshape(T, -1)
    return (o * torch.sigmoid(h @ W[p + "g"].t())) @ W[p + "o"].t(), new, ()


def _mlstm(W, p, m, h, eps, pos, past):
    T, H, dk, dv, cap = h.shape[0], m["heads"], m["dim"], m["vdim"], m["gate_cap"]
    q = (h @ W[p + "q"].t()).view(T, H, dk) * dk ** -0.5
    k, v = (h @ W[p + "k"].t()).view(T, H, dk), (h @ W[p + "v"].t()).view(T, H, dv)
    ig = cap * torch.tanh(_lin(W, p + "i", h) / cap)
    fg = F.logsigmoid(cap * torch.tanh(_lin(W, p + "f", h) / cap))
    S, n, mx = past[1] or (h.new_zeros(H, dk, dv), h.new_zeros(H, dk), h.new_zeros(H))
    out = []
    for t in range(T):
        top = torch.maximum(fg[t] + mx, ig[t])
        a, b = torch.exp(fg[t] + mx - top), torch.exp(ig[t] - top)
        kb = b[:, None] * k[t]
        S, n, mx = a[:, None, None] * S + kb[:, :, None] * v[t][:, None], a[:, None] * n + kb, top
        den = torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-mx)) + 1e-6
        out.append(torch.matmul(q[t][:, None], S)[:, 0] / den[:, None])
    o = _rms(torch.stack(out), eps).reshape(T, -1) * W[p + "norm"]
    return (o * torch.sigmoid(h @ W[p + "g"].t())) @ W[p + "o"].t(), None, (S, n, mx)


def _memory(q, k, v, decay, beta, S, delta=False):
    """o_t = S_t^T q_t with S_t = decay_t S_(t-1) + beta_t k_t v_t^T (``delta``: v less what the memory gives for k).  q, k [T, H,
    dk], v [T, H, dv], decay [T, H, 1 or dk], beta [T, H]."""
    out = []
    for t in range(q.shape[0]):
        S = decay[t][:, :, None] * S
        u = v[t] - torch.matmul(k[t][:, None], S)[:, 0] if delta else v[t]
        S = S + k[t][:, :, None] * (beta[t][:, None] * u)[:, None]
        out.append(torch.matmul(q[t][:, None], S)[:, 0])
    return torch.stack(out), S


def _gla(W, p, m, h, eps, pos, past):
    T, H, dk, dv = h.shape[0], m["heads"], m["dim"], m["vdim"]
    q, k = (_lin(W, p + n, h).view(T, H, dk) for n in ("q", "k"))
    v = _lin(W, p + "v", h).view(T, H, dv)
    alpha = torch.sigmoid(_lin(W, p + "a2", _lin(W, p + "a1", h))).pow(1.0 / m["tau"]).view(T, H, dk)
    S = past[1][0] if past[1] else h.new_zeros(H, dk, dv)
    o, S = _memory(q * dk ** -0.5, k, v, alpha, h.new_ones(T, H), S)
    o = (_rms(o, eps) * W[p + "norm"]).reshape(T, -1)
    return _lin(W, p + "o", o * F.silu(_lin(W, p + "g", h))), None, (S,)


def _sigmoid_attention(W, p, m, h, eps, pos, past):
    T, H, G, dk, dv = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k = (_rms(_lin(W, p + n, h), eps) * W[p + n + ".norm"] for n in ("q", "k"))
    qt = m["q_temp"]
    q = q * (1.0 + qt["coef"] * torch.log(torch.floor((pos + 1.0).to(F64) / qt["every"]) + 1.0))[:, None]
    new = torch.cat([_lin(W, p + "v", h).view(T, G, dv), k.view(T, G, dk)], -1)
    rows = new if past[0] is None else torch.cat([past[0].view(-1, G, dv + dk), new])
    s, dist = _scores(q.view(T, H, dk), rows[..., dv:], m["scale"], rows.shape[0] - T)
    by = lambda n: W[p + n].view(G, H // G, 1, 1)
    s = torch.sigmoid(s - by("r1") * torch.log(1.0 + by("r2") * dist.clamp(min=0)) + by("pb")).masked_fill(dist < 0, 0.0)
    o = _attend(s, rows[..., :dv]) * torch.sigmoid(_lin(W, p + "g", h))[:, :, None]
    return _lin(W, p + "o", o.reshape(T, -1)), new.reshape(T, -1), ()


def _window_attention(W, p, m, h, eps, pos, past):
    T, H, G, d, dv = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    r = m["rot"]
    f, sc = _freq(r["base"], r["dims"]), r["scaling"]
    turns = sc["original"] * f / (2.0 * math.pi)
    keep = ((turns - sc["low"]) / (sc["high"] - sc["low"])).clamp(0.0, 1.0)
    f = (1.0 - keep) * f / sc["factor"] + keep * f
    q, k = (_turn((_rms(_lin(W, p + n, h), eps) * W[p + n + ".norm"]).view(T, -1, d), pos, f) for n in ("q", "k"))
    new = torch.cat([_lin(W, p + "v", h).view(T, G, dv), k], -1)
    rows = new if past[0] is None else torch.cat([past[0].view(-1, G, dv + d), new])
    o = _softmax_attention(q, rows[..., dv:], rows[..., :dv], m["scale"], rows.shape[0] - T, m["mask"]["size"])
    return _lin(W, p + "o", o.reshape(T, -1)), new.reshape(T, -1), ()


def _delta_rule(W, p, m, h, eps, pos, past):
    T, H, G, d, dv = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    w = torch.cat([W[p + n + ".conv"] for n in ("q", "k", "v")])
    S, before = past[1] or (h.new_zeros(H, d, dv), h.new_zeros(w.shape[1] - 1, w.shape[0]))
    y, before = _conv(torch.cat([_lin(W, p + n, h) for n in ("q", "k", "v")], -1), w, None, before)
    q, k, v = F.silu(y).split([G * d, G * d, H * dv], -1)
    unit = lambda x: x / torch.sqrt(x.pow(2).sum(-1, keepdim=True) + 1e-6)
    q, k = (unit(x.view(T, G, d)).repeat_interleave(H // G, 1) for x in (q, k))
    decay = torch.exp(-torch.exp(W[p + "A_log"]) * F.softplus(_lin(W, p + "a", h) + W[p + "dt_bias"]))
    o, S = _memory(q * d ** -0.5, k, v.reshape(T, H, dv), decay[:, :, None], torch.sigmoid(_lin(W, p + "b", h)), S, delta=True)
    o = (_rms(o, eps) * W[p + "norm"]).reshape(T, -1)
    return _lin(W, p + "o", o * F.silu(_lin(W, p + "g", h))), None, (S, before)


def _pair(W, p, m, h, eps, pos, past):
    a, rows, _ = _window_attention(W, p + "left.", m["left"], h, eps, pos, past)
    b, _, states = _delta_rule(W, p + "right.", m["right"], h, eps, pos, past)
    return m["left_scale"] * a + m["right_scale"] * b, rows, states


def _mamba2(W, p, m, h, eps, pos, past):
    T, H, dv, N, G = h.shape[0], m["heads"], m["vdim"], m["state"], m["groups"]
    z, xbc, dt = _lin(W, p + "in", h).split([H * dv, H * dv + 2 * G * N, H], -1)
    w = W[p + "conv"]
    S, before = past[1] or (h.new_zeros(H, N, dv), h.new_zeros(w.shape[1] - 1, w.shape[0]))
    y, before = _conv(xbc, w, W[p + "conv.b"], before)
    x, B, C = F.silu(y).split([H * dv, G * N, G * N], -1)
    dt = F.softplus(dt + W[p + "dt_bias"])
    x = x.reshape(T, H, dv)
    B, C = (t.view(T, G, N).repeat_interleave(H // G, 1) for t in (B, C))
    o, S = _memory(C, B, x, torch.exp(-torch.exp(W[p + "A_log"]) * dt)[:, :, None], dt, S)
    y = (o + W[p + "D"][:, None] * x).reshape(T, -1) * F.silu(z)
    y = _rms(y.view(T, m["norm_groups"], -1), eps).reshape(T, -1) * W[p + "norm"]
    return _lin(W, p + "o", y), None, (S, before)


def _retention(W, p, m, h, eps, pos, past):
    T, H, d, dv = h.shape[0], m["heads"], m["dim"], m["vdim"]
    f = _freq(m["rot"]["base"], m["rot"]["dims"])
    q, k = (_turn(_lin(W, p + n, h).view(T, H, d), pos, f) for n in ("q", "k"))
    S = past[1][0] if past[1] else h.new_zeros(H, d, dv)
    decay = torch.tensor(m["decay"], dtype=F64, device="cuda").view(1, H, 1).expand(T, H, 1)
    o, S = _memory(q, k * d ** -0.5, _lin(W, p + "v", h).view(T, H, dv), decay, h.new_ones(T, H), S)
    return _lin(W, p + "o", _rms(o, eps).reshape(T, -1) * F.silu(_lin(W, p + "g", h))), None, (S,)


_MIXERS = {"latent_attention": _latent, "mlstm": _mlstm, "gla": _gla, "attention": _sigmoid_attention, "parallel": _pair,
           "mamba2": _mamba2, "retention": _retention}


def _experts(W, p, h, idx, w, n, one):
    y = torch.zeros_like(h)
    for e in range(n):
        t, slot = (idx == e).nonzero(as_tuple=True)
        y.index_add_(0, t, one(f"{p}e{e}.", h[t]) * w[t, slot][:, None])
    return y


def _lenitar_moe(W, p, f, h):
    r = f["router"]
    s = torch.sigmoid(h @ W[p + "router"].t())
    G, per = r["groups"]["count"], r["experts"] // r["groups"]["count"]
    best = s.view(-1, G, per).topk(min(2, per), -1).values.sum(-1).topk(r["groups"]["keep"], -1).indices
    ok = torch.zeros(s.shape[0], G, dtype=torch.bool, device="cuda").scatter_(1, best, True).repeat_interleave(per, 1)
    idx = s.masked_fill(~ok, -1.0).topk(r["top"], -1).indices
    one = lambda q, x: _lin(W, q + "down", F.silu(_lin(W, q + "gate", x)) * _lin(W, q + "up", x))
    return _experts(W, p, h, idx, s.gather(1, idx), r["experts"], one)


def _malinex_moe(W, p, f, h):
    r = f["router"]
    s = torch.softmax(h @ W[p + "router"].t(), -1)
    idx = (s + W[p + "correction"]).topk(r["top"], -1).indices
    w = s.gather(1, idx)
    one = lambda q, x: _lin(W, q + "down", F.relu(_lin(W, q + "up", x)).square())
    return _experts(W, p, h, idx, w / (w.sum(-1, keepdim=True) + 1e-20), r["experts"], one) + one(p + "shared.", h)


def _hybrid(cfg, W, ids, pos, past):
    """(the final normed stream of the given tokens, the head's weight, [(new rows, states) per layer])."""
    eps, kept = cfg["norm"]["eps"], []
    x = W["embed"][ids]
    fam = cfg["architecture"].lower()
    if fam == "lenitar":
        x = x * cfg["embedding"]["scale"]
    elif fam == "malinex":
        x = x + W["pos"][pos]
    for i, spec in enumerate(cfg["layers"]):
        p, mix, f = f"l{i}.", _MIXERS[spec["type"]], spec["mlp"]
        if fam == "lenitar":
            h = _ln(x, W[p + "norm1"], W[p + "norm1.b"], eps)
            y, rows, states = mix(W, p + "mix.", spec["mixer"], h, eps, pos, past[i])
            x = x + y + _lenitar_moe(W, p + "mlp.", f, h)
        elif fam == "malinex":
            h = _rms(x, eps) * W[p + "norm1"]
            y, rows, states = mix(W, p + "mix.", spec["mixer"], h, eps, pos, past[i])
            x = x + _rms(y * torch.sigmoid(_lin(W, p + "rg1", h)), eps) * W[p + "norm1b"]
            h = _rms(x, eps) * W[p + "norm2"]
            y = _malinex_moe(W, p + "mlp.", f, h) * torch.sigmoid(_lin(W, p + "rg2", h))
            x = x + _rms(y, eps) * W[p + "norm2b"]
        else:
            y, rows, states = mix(W, p + "mix.", spec["mixer"], x, eps, pos, past[i])
            x = x + cfg["residual_mult"] * _rms(y, eps) * (1.0 + W[p + "norm1"])
            y = _lin(W, p + "mlp.down", F.gelu(_lin(W, p + "mlp.up", x)))
            x = x + cfg["residual_mult"] * _rms(y, eps) * (1.0 + W[p + "norm2"])
        kept.append((rows, states))
    if fam == "lenitar":
        return _ln(x, W["final.norm"], W["final.norm.b"], eps), W["head"], kept
    w = W["final.norm"] if fam == "malinex" else 1.0 + W["final.norm"]
    return _rms(x, eps) * w, W["head"] if fam == "malinex" else W["embed"], kept


def _exact_hybrid(case, st):
    eng = st["eng"]
    cfg, n = eng.cfg.to_dict(), len(eng.kv_cache._layers)
    W = {k: v.to(F64) for k, v in eng.model.export_named().items()}
    split = []  # per layer (pool of rows or None, pools of states)
    for i in range(n):
        e = eng.kv_cache.layer(i)
        if not isinstance(e, tuple):
            e = (e, ())
        elif not (len(e) == 2 and isinstance(e[1], tuple)):
            e = (None, e)
        split.append(e)
    out = [(None if r is None else torch.zeros_like(r, dtype=F64), tuple(torch.zeros_like(s, dtype=F64) for s in ss)) for r, ss in split]
    decode = case["kind"] == "decode"
    seqs = st["seqs"] if decode else _open(eng, st["ids"])
    rows = []
    for j, s in enumerate(seqs):
        slot, first = (eng.kv_cache.slots.slot(s.seq_id), s.num_tokens - 1 if decode else 0)
        at = torch.from_numpy(eng.kv.slots(s.seq_id, 0, s.num_tokens).astype("int64")).cuda()
        past = [(None, None)] * n
        if decode:
            past = [(None if r is None else r.view(-1, r.shape[-1])[at[:first]].to(F64), tuple(t[slot].to(F64) for t in ss) or None)
                    for r, ss in split]
        ids = torch.tensor(s.all_ids[first:], device="cuda")
        x, head, kept = _hybrid(cfg, W, ids, torch.arange(first, s.num_tokens, device="cuda"), past)
        rows.append((x if decode else x[torch.tensor(st["want"][j], device="cuda")]) @ head.t())
        for (r, ss), (new, states) in zip(out, kept):
            if r is not None and not decode:
                r.view(-1, r.shape[-1])[at] = new
            for t, v in zip(ss, states):
                t[slot] = v
    # the mLSTM's stabiliser [slots, heads] is a free choice of scale for the memory beside it: it has no exact value of its own
    known = lambda ss: [None if t.dim() == 2 else t for t in ss]
    if decode:
        return {"logits": torch.cat(rows), "states": [t for _, ss in out for t in known(ss)]}
    return {"logits": torch.cat(rows), "cache": [t for r, ss in out for t in ([] if r is None else [r]) + known(ss)]}


def exact(case, seed):
    st = prepare(case, seed)
    if case["kind"] == "train":
        return _exact_train(case, st)
    with torch.inference_mode():
        return _exact_dense_serving(case, st) if case["model"] in DENSE else _exact_hybrid(case, st)

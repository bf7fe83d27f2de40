"""Linear layer with gradient *sinks*: weight gradients are written by the backward GEMM
directly into the flat gradient buffer.

With stock autograd, ``dW = dY^T X`` lands in a fresh tensor and AccumulateGrad then adds
it into ``param.grad`` (our flat-buffer view) — an extra read-read-write pass over every
weight gradient (~40 GB/step for GPT-7B, ~7 ms of HBM time on MI355X).  Here the backward
GEMM writes the flat view itself: ``mm(..., out=view)`` on the first micro-step after
``zero_grad`` (beta = 0, so the buffer never needs zeroing) and ``addmm_`` (hipBLASLt
beta = 1 epilogue, free accumulation) on later gradient-accumulation micro-steps.  The sink
then notifies the DP overlap engine that the parameter's gradient is ready — the same
signal ``register_post_accumulate_grad_hook`` gives for ordinary parameters.

Data gradients: up to 16384 tokens a step they run on the in-house 64-deep MFMA kernel, which reads W as it is (``gemm64_ex``,
llmctl/ops/csrc/gemm64.hip), as the weight gradients do (20-40 % over hipBLASLt on the GPT-7B shapes).  Beyond that, and for
shapes it does not take, large weights go through a transposed copy: ``dX = dY W`` (the "NN" GEMM) runs ~13 % slower on
hipBLASLt than the forward's "TN" layout at the GPT-7B shapes (``profiles/gemm_tunable_dgradT_r1.log``: 7.27 -> 6.37 ms per
layer).  Such weights keep a bf16 ``W^T`` copy, refreshed by the transpose HIP kernel the first time the weight is used after an
optimizer step (``GradSink.epoch``; under ZeRO-1/2 that is after the layer's all-gather has landed), and the backward
computes ``dX = F.linear(dY, W^T)``.  Cost: one bf16 copy of the projection weights and ~2 x 13.5 GB of HBM transpose traffic per
step.  The down projection's data gradient can carry the SwiGLU backward in its epilogue.  Knob ``dgrad64``, see
``dgrad64_shape_ok`` and ``weight_t_ok``.
"""

from __future__ import annotations

import contextlib
import functools
import threading
from typing import Callable, List, Optional, Tuple

import torch
import torch.nn.functional as F

from llmctl.config.knobs import knobs
from llmctl.ops._lib import native, use_native  # (once: an import in a function is 0.5 us a call)


# gemm64_ex config: knob gemm64_config (see gemm64_config below).  A tuning cache
# (llmctl.plugins.tuning_cache) can override it per layout or per exact shape.
DGRAD64_TOKENS = 16384  # see dgrad64_shape_ok
GEMM64_CONFIGS: dict = {}  # layout -> config
GEMM64_SHAPE_CONFIGS: dict = {}  # (layout, M, N, K) -> config


def gemm64_config(layout: str, M: int, N: int, K: int) -> int:
    """Config of one gemm64 call: a tuning-cache entry for the exact shape or the layout, else
    knob ``gemm64_config`` (default 304: the persistent 4-wave kernel; the down projection's
    weight gradient with the SwiGLU backward as a side job runs the one-shot 4-wave kernel --
    3 rounds of bench.py: 1051.9 vs 1053.3 ms/step for 904 on every wgrad,
    profiles/ab_wgrad_persistent_r4.txt)."""
    c = GEMM64_SHAPE_CONFIGS.get((layout, M, N, K), GEMM64_CONFIGS.get(layout))
    if c is not None:
        return c
    return knobs().gemm64_config


def _gemm64_enabled() -> bool:
    return knobs().gemm64  # False: A/B against hipBLASLt


def _rows_ok(*ts: torch.Tensor) -> bool:
    for t in ts:
        if t.stride(1) != 1 or t.stride(0) % 8 or t.data_ptr() % 16:
            return False
    return True


def _gemm64_ok(M: int, N: int, K: int, *ts: torch.Tensor) -> bool:
    """Shapes the 64-deep MFMA kernel (llmctl/ops/csrc/gemm64.hip) takes: M, N multiples of
    256, K of 128, bf16 GPU operands with 16-byte aligned unit-stride rows."""
    if not _gemm64_enabled() or M % 256 or N % 256 or K % 128 or K == 0:
        return False
    if not all(t.is_cuda and t.dtype == torch.bfloat16 for t in ts):
        return False
    from llmctl.ops._lib import use_native

    return use_native(ts[0]) and _rows_ok(*ts)


def fwd64_pick(M: int, N: int, K: int) -> bool:
    """Forward ``x W^T`` shapes routed to gemm64: the wide up-projection up to 8192 tokens and the
    QKV / down projections at <= 2048 tokens (serving prefill chunks); hipBLASLt keeps the
    training shapes (24576 tokens) and the rest.  Standalone sweep:
    profiles/gemm64_fwd_small_m_r2.jsonl (up at 2048: 0.278 vs 0.422 ms); in situ, inside a
    GPT-7B 2k prefill, hipBLASLt picks a better up-projection kernel (0.268 ms) and the gain is
    ~1.5 ms per prefill (TTFT p50 28.0 vs 29.5 ms, profiles/ttft_fwd64_r2.txt).
    Knob ``fwd64``: ``off`` disables, ``all`` forces every supported shape (A/B)."""
    mode = knobs().fwd64
    if mode == "off" or not _gemm64_enabled():
        return False
    if mode == "all":
        return True
    return (N >= 16384 and M <= 8192) or (M <= 2048 and (N >= 8192 or K >= 8192))


def forward_linear(x: torch.Tensor, w: torch.Tensor, b: Optional[torch.Tensor] = None, layout: str = "eager") -> torch.Tensor:
    """``x @ w^T (+ b)``: small products on gemm_small (``small_pays``), those of one to a few rounds of tiles on gemm_rows (``rows_form``), gemm64 for the shapes ``fwd64_pick`` selects, hipBLASLt otherwise."""
    N, K = w.shape
    M = x.numel() // K if x.shape[-1] == K else 0
    if M > 32 or layout != "eager":
        y = small_linear(x, w, b, layout)
        if y is None:
            y = rows_linear(x, w, b, None, 0, layout == "eager")
        if y is not None:
            return y
    if M and fwd64_pick(M, N, K) and x.dtype == torch.bfloat16:
        x2 = x.reshape(M, K)
        if _gemm64_ok(M, N, K, x2, w) and 256 * x2.stride(0) * 2 < 2**31 and 256 * w.stride(0) * 2 < 2**31:
            from llmctl.ops._lib import native

            y = torch.empty(M, N, dtype=x.dtype, device=x.device)
            native().gemm64_ex(x2, w, y, False, False, False, gemm64_config("fwd", M, N, K))
            if b is not None:
                y += b
            return y.view(*x.shape[:-1], N)
    return F.linear(x, w, b)


class _Steps(threading.local):
    recorded = False


_steps = _Steps()


@contextlib.contextmanager
def recorded_step():
    """This thread's products are those of a step that is recorded, or of the eager ones ahead of the recording: launches that the host does not feed, so the ``eager`` rules take
    nothing for its sake.  Said by who records, not asked of the stream: a recording has to take the routes of the steps ahead of it, where the library makes its handle and loads its kernels (a
    library product that a recording is the first to call ends the process)."""
    was, _steps.recorded = _steps.recorded, True
    try:
        yield
    finally:
        _steps.recorded = was


@functools.lru_cache(maxsize=4096)
def small_pays(layout: str, M: int, N: int, K: int, bias: bool = False) -> bool:
    """Is ``gemm_small`` (csrc/gemm_small.hip) the fastest form of this product of a training step?  ``fwd``: M tokens, N outputs; ``dgrad``: K
    outputs, N inputs; ``wgrad``: M outputs, N inputs, K tokens, ``bias``: and the bias's gradient, which else takes two launches more below 256
    tokens.  Where the tiles of 32 are about one round of the chip; beyond that each operand is read too often.  us in a graph, the next best / here:
    fwd 1024 tokens 512 x 256 5.8 / 5.5, 768 x 256 5.9 / 6.3; 200 768 x 768 7.5 / 6.1, 384 7.7 / 8.8; 64 768 x 3072 10.1 / 13.5; 512 1024 x 512 7.8 / 7.0;
    dgrad 128 tokens 768 x 3072 10.1 / 8.2, 200 9.1 / 10.7, 512 768 x 768 12.9 / 8.4, 640 8.1 / 8.4; beyond K 1024 the 256-row tiles are what is left behind:
    256 1408 x 256 12.8 / 8.0, 2304 x 768 16.2 / 11.1, 128 1536 x 512 8.2 / 8.7, 48 3072 x 768 9.1 / 11.7;
    wgrad 4096 tokens 768 x 256 18.5 / 15.1, 1408 x 256 27.6 / 25.7, 1024 768 x 768 16.9 / 10.9, 128 2304 x 768 11.3 / 10.3, 256 9.2 / 10.7, 48 7.2 / 9.4;
    with a bias 200 2304 x 768 13.5 / 10.5, 128 3072 x 768 15.9 / 14.2.
    ``eager``: the forward of a prompt, whose launches the host feeds one by one: a library product takes it 20 us, this 9, so every product of at most
    some 16 us (gpt2-125m, a prompt of 100 tokens 2130 / 1400, of 300 2140 / 1400, of 800 2205 / 2035; the tiny model, 470 504 / 396)."""
    w = -(-M // 32) * -(-N // 32)
    if layout == "eager":
        return M > 32 and (K * -(-w // 256) <= 3072 if w <= 512 else K * -(-w // 1024) <= 1536)
    if layout == "fwd":
        return (w <= 256 and K <= 1024) or (w <= 512 and K <= 512)
    if layout == "dgrad":
        return (w <= 256 or (w <= 384 and K <= 1024) or (w <= 704 and K <= 256)) and (K <= 1024 or (K <= 3072 and M % 256 == 0))
    return ((w <= 384 and K <= 4096) or (w <= 1024 and K <= 1024) or (w <= 1792 and 64 <= K <= 128)
            or (bias and w <= 2304 and 64 <= K < 256))


_PLAIN = (torch.Tensor, torch.nn.Parameter)
_is_wrapped, _is_legacy_batched = torch._C._functorch.is_functorch_wrapped_tensor, torch._C._functorch.is_legacy_batchedtensor


_modes, _function_modes, _tracing = torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack, torch._C._is_tracing
_any_autocast, _forward_ad = torch._C._is_any_autocast_enabled, torch.autograd.forward_ad


def _calls_are_seen() -> bool:
    """Something in this thread traces, counts or replaces the library's calls (which take symbolic sizes, and other ones when a trace is run).  0.3 us."""
    return _modes() or _function_modes() or _tracing()


def _small_operand(t: torch.Tensor, dtypes=(torch.bfloat16,)) -> bool:
    """A matrix of aligned rows that ``gemm_small`` reads, and no tensor of a transform (vmap)."""
    if type(t) not in _PLAIN or not t.is_cuda or t.dtype not in dtypes or t.dim() != 2 or _is_wrapped(t) or _is_legacy_batched(t):
        return False
    st = t.stride()
    return st[1] == 1 and st[0] & 7 == 0 and st[0] >= t.shape[1] and t.data_ptr() & 15 == 0


def _small_bias(b: torch.Tensor, N: int) -> bool:
    """The same of a bias."""
    return (type(b) in _PLAIN and b.is_cuda and b.dtype is torch.bfloat16 and not _is_wrapped(b) and not _is_legacy_batched(b) and b.shape == (N,)
            and b.is_contiguous() and b.data_ptr() & 7 == 0)


def _small_ok(layout: str, M: int, N: int, K: int, *ts: torch.Tensor) -> bool:
    """``gemm_small`` takes operands of these sizes; sizes with a tuned gemm64 config stay with that."""
    return (M > 0 and N > 0 and K > 0 and N & 7 == 0 and ((M if layout == "wgrad" else K) & 7) == 0 and _gemm64_enabled()
            and not (layout in GEMM64_CONFIGS or (layout, M, N, K) in GEMM64_SHAPE_CONFIGS)
            and all(map(_small_operand, ts)) and use_native(ts[0]))


def small_linear(x: torch.Tensor, w: torch.Tensor, b: Optional[torch.Tensor] = None, layout: str = "fwd", act: int = 0) -> Optional[torch.Tensor]:
    """``act(x @ w^T (+ b))`` on ``gemm_small`` where it takes it and no gradient is wanted of it (the forward of an autograd function, serving); else
    None.  ``layout``: the rule of ``small_pays``; ``act``: as in csrc/stream_linear.h (0: none)."""
    N, K = w.shape
    M = x.numel() // K if K and x.shape[-1] == K else 0
    if not M or type(M * N) is not int or not small_pays(layout, M, N, K) or _calls_are_seen() or not w.is_cuda or knobs().fwd64 != "auto":
        return None  # (symbolic and traced sizes are no ints)
    if layout == "eager" and not small_pays("fwd", M, N, K) and _steps.recorded:
        return None
    if (type(x) is not torch.Tensor or _is_legacy_batched(x) or not x.is_contiguous() or _any_autocast()
            or (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad or (b is not None and b.requires_grad)))
            or _forward_ad._current_level >= 0 or torch.compiler.is_compiling()):
        return None
    x2 = x if x.dim() == 2 else x.view(M, K)
    if not _small_ok("fwd", M, N, K, x2, w) or not (b is None or _small_bias(b, N)):
        return None
    y = torch.empty(M, N, dtype=x.dtype, device=x.device)
    native().gemm_small(x2, w, y, False, False, False, b, None, False, act)
    return y if x.dim() == 2 else y.view(*x.shape[:-1], N)


def small_linear_f32(x: torch.Tensor, w: torch.Tensor) -> Optional[torch.Tensor]:
    """``x @ w^T`` of a prompt's rows with an fp32 result on ``gemm_small``, by the rules of :func:`small_linear`'s ``eager`` form, up to 2 Mi outputs;
    else None.  Decay logits of gated linear attention (K 64), us, library / here: 200 x 1024 1.8 / 1.7, 2000 x 512 2.6 / 4.1, 2911 x 1024 4.8 / 9.1; a library product takes the host 24 us, this
    9: malinex width 2048, 200 tokens 797 / 753, width 1024, 3800 tokens 964 / 924; 2911 tokens of width 2048 1375 / 1381, so left."""
    if x.dim() != 2 or w.dim() != 2 or x.shape[1] != w.shape[1] or type(x.shape[0]) is not int or _calls_are_seen() or not w.is_cuda or knobs().fwd64 != "auto":
        return None
    M, (N, K) = x.shape[0], w.shape
    if (M * N > 2 << 20 or not small_pays("eager", M, N, K) or _steps.recorded or _any_autocast() or (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad))
            or _forward_ad._current_level >= 0 or torch.compiler.is_compiling() or not _small_ok("fwd", M, N, K, x, w)):
        return None
    y = torch.empty(M, N, dtype=torch.float32, device=x.device)
    native().gemm_small(x, w, y, False, False, False)
    return y


_CUS = 256  # of an MI355X


def _rounds_us(items: int, ktiles: float, empty: float, full: float, fixed: float) -> float:
    """Workgroups of one to a CU: a round's K-tiles at ``empty`` us and ``full`` more on a full chip, and a fixed part."""
    whole, rest = divmod(items, _CUS)
    return whole * (ktiles * (empty + full) + fixed) + (ktiles * (empty + full * rest / _CUS) + fixed if rest else 0.0)


def _tile_rows(M: int, form: int) -> int:
    return -(-M // 128) if form == 2 else 1 if M <= 288 else (M - 33) // 256 + 1


@functools.lru_cache(maxsize=8192)
def rows_form(M: int, N: int, K: int, act: bool = False, eager: bool = False) -> int:
    """How ``gemm_rows`` (csrc/gemm_rows.hip) multiplies M rows of width K to N outputs where that is faster than the library: tiles (1 = 256 rows, 2 = 128) + 4 (ranges of K - 1);
    else 0.  ``act``: an activation follows, which costs the library's product a pass; ``eager``: launches that the host feeds one by one.
    Up to 1024 rows: :func:`_few_rows_form`, and nothing else.  Beyond, one range of K: a model of either's workgroups and of the library's products, us: 12 and 1300 TFLOP/s, small ones 6 and 550,
    fitted to kernel times with operands from HBM (``profiles/prompt_products.txt``, to 4096 rows, 256 to 12288 outputs, K 256 to 8192).  Of its 73 sizes of more than 1024
    rows the rule takes 31, in 21 % less time; one of these takes longer, 1049 x 256 x 256 5.3 / 5.6.  In ``profiles/short_prompt_products.txt`` (42 such sizes) 19, in 8 % less; four take longer,
    1300 x 3072 x 1024 15.4 / 18.1, the others up to 0.7 us.
    us, library / here: 2048 x 2048 x 2048 25.8 / 17.8, 2048 x 3712 x 2048 35.5 / 29.0, 2911 x 2048 x 1024 23.2 / 16.8, 1128 x 3584 x 1664 21.4 / 15.5; left to the library: 1.1 rounds,
    2911 x 3072 x 2048 36.8 / 46.0; large products, 3379 x 8192 x 2048 94 / 109."""
    if M <= 32 or N <= 0 or N & 7 or K & 127 or K < 256:
        return 0
    if M <= 1024:
        return _few_rows_form(M, N, K, act, eager)
    cols, kt = -(-N // 128), K / 64
    tall = _rounds_us(_tile_rows(M, 1) * cols, kt, 0.47, 0.36, 5.0 + act * _ACT_TILE[1])
    half = _rounds_us(_tile_rows(M, 2) * cols, kt, 0.28, 0.18, 4.0 + act * _ACT_TILE[2])
    gflop = 2e-9 * M * N * K
    if min(tall, half) >= (0.95 if K <= 2304 else 0.85) * min(12.0 + gflop / 1.3, 6.0 + gflop / 0.55) + act * _act_us(M, N):
        return 0
    return 1 if tall <= half else 2


_ACT_TILE = {1: 3.9, 2: 2.1}  # GELUs of a tile in its epilogue, us: nothing else runs on its CU meanwhile


def _act_us(M: int, N: int) -> float:
    return 3.0 + 1e-6 * M * N  # an activation pass of its own, us


def _few_rows_form(M: int, N: int, K: int, act: bool, eager: bool) -> int:
    """:func:`rows_form` of up to 1024 rows.  Their tiles are few, so K is cut into ranges of 256 at least: rounds of 256 workgroups, a K-tile of 64 1.06 us on tiles of 256 rows and 0.82 on those of
    128, 3.1 us and the fp32 sums' bytes for the pass that adds the ranges, and the weight's stream at the least; against the library's products, which K beyond 4096 makes slow.  The
    constants are fitted to the choice, not to either time, at 1200 sizes (fitted to one half of them they do as well on the other; ``profiles/few_rows_products.txt``, ``short_prompt_products.txt``
    and ``prompt_products.txt``): the library's own times jump by a half from one size to the next (256 x 6144 x 2048 27.4, 288 rows 18.8).  573 of the sizes timed are taken, in 18 % less
    time; 38 of these take longer, by 3.6 us at most but for one (579 x 8448 x 6272 76 / 85), nine by more than a tenth (201 x 256 x 6144 11.2 / 14.0).  All sizes together take 3 % more than with
    the better choice everywhere, and 9 % less than in the library.
    ``eager``: a step's launches are the host's time, and a library product takes it 24 us, this 9 (13 with the pass that adds the ranges): of up to 6 Mi outputs and 38 us also what may take
    the chip a few us longer, 8 and 0.3 of the library's time by the model, 5.2 at most of the sizes timed but for that one (350 x 3712 x 2048 16.3 / 21.5; all 1003 that are taken, in 11 % less).
    us, library / here: 600 x 2048 x 8192 47 / 36, 128 x 4096 x 11008 79 / 46, 288 x 8256 x 2048 29 / 22; left to the library 900 x 2048 x 2048 16.3 / 20.3, 288 x 32000 x 2048 68 / 81, 128 x 12288 x
    4096 45 / 53; for the host's sake 256 x 2048 x 2048 11.3 / 14.9.  Prompts, us a step, with every product the library's / here: dumazen width 2048 100 tokens 1387 / 1118, 450 1331 / 1110; lenitar 300
    982 / 880; malinex 200 948 / 809."""
    # Of nine sizes of as many outputs six are the library's, by 4 to 33 %; three of K up to 512 would be faster here (1000 x 11008 x 512 43 / 27) and stay where the rule of large products had them.
    if not act and M * N > 10 << 20:
        return 0
    cols, best, code = -(-N // 128), 1e9, 0
    for splits in (1, 2, 3, 4, 6, 8, 12, 16):
        if splits > 1 and (splits > K // 256 or splits * cols * _tile_rows(M, 1) > 512):
            break
        for form, step in ((1, 1.06), (2, 0.82)):
            rounds = -(-splits * cols * _tile_rows(M, form) // _CUS)
            t = rounds * (K / 64 / splits * step + (act * _ACT_TILE[form] if splits == 1 else 0.0)) + (3.1 + splits * M * N * 4e-6 if splits > 1 else 0.0)
            if t < best:
                best, code = t, form + 4 * (splits - 1)
    mb, gflop = N * K * 2e-6, 2e-9 * M * N * K
    best = max(best, mb / 1.8)
    library = min(7.2 + 0.22 * mb + 0.88 * gflop + 20.0 * max(0, K - 4096) / 1024, 75.0 + 0.68 * gflop) + act * _act_us(M, N)
    return code if best < library or (eager and M * N <= 6 << 20 and best <= min(1.3 * library + 8.0, 38.0)) else 0


def rows_linear(x: torch.Tensor, w: torch.Tensor, b: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None, act: int = 0,
                eager: bool = True) -> Optional[torch.Tensor]:
    """``act(x @ w^T (+ b))`` (into ``out`` ``[M, groups, N / groups]``, whose rows and groups may lie apart) on ``gemm_rows`` where it takes it, pays (:func:`rows_form`) and no gradient is wanted of it (the forward of an autograd function, serving); else
    None.  ``act``: 0 none, 1 erf GELU, 2 tanh GELU (without ``out``).  A library product takes the host 24 us, this 9: Lenitar's prompt of 2048 tokens, sixteen of them,
    1198 us, so 1127 (kernels 1190 / 1106); gpt2-125m's of 700 and 300 tokens 2195 / 1870."""
    if w.dim() != 2:  # (a vector: the library's)
        return None
    N, K = w.shape
    M = x.numel() // K if K and x.shape[-1] == K else 0
    code = rows_form(M, N, K, act != 0, eager and not _steps.recorded) if M and type(M * N) is int else 0  # (symbolic and traced sizes are no ints)
    if not code or _calls_are_seen() or not w.is_cuda or knobs().fwd64 != "auto":
        return None
    if (type(x) is not torch.Tensor or _is_legacy_batched(x) or not (x.dim() == 2 or x.is_contiguous()) or _any_autocast()
            or (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad or (b is not None and b.requires_grad)))
            or _forward_ad._current_level >= 0 or torch.compiler.is_compiling()):
        return None
    x2 = x if x.dim() == 2 else x.view(M, K)
    if (not _small_ok("fwd", M, N, K, x2, w) or not (b is None or (_small_bias(b, N) and b.data_ptr() & 15 == 0))
            or 512 * x2.stride(0) >= 1 << 30 or 512 * w.stride(0) >= 1 << 30):
        return None
    if out is not None:
        if not (type(out) is torch.Tensor and out.dtype is torch.bfloat16 and out.shape[2] & 7 == 0 and out.stride(2) == 1 and out.stride(0) & 7 == 0
                and out.stride(1) & 7 == 0 and out.data_ptr() & 15 == 0):
            return None
        native().gemm_rows_into(x2, w, b, code & 3, out, (code >> 2) + 1)
        return out
    y = native().gemm_rows(x2, w, b, code & 3, (code >> 2) + 1, act)
    return y if x.dim() == 2 else y.view(*x.shape[:-1], N)


@functools.lru_cache(maxsize=1024)
def _prompt_form(M: int, N: int, K: int, act: bool) -> Optional[int]:
    """The route of an eager prompt's product through ``ops.functional.decode_linear`` as csrc/dense_prompt.cpp names it; None: another one."""
    if N & 7 or K & 7:
        return None
    if small_pays("eager", M, N, K):
        return -1
    code = rows_form(M, N, K, act, True)
    return None if not code and (fwd64_pick(M, N, K) or (act and rows_form(M, N, K, False, True))) else code


def prompt_forms(x: torch.Tensor, sizes) -> Optional[List[int]]:
    """The routes of the products ``(N, K, activation)`` of one eager prompt's rows ``x [M, .]``, where nothing that those routes look at asks for others; else None."""
    M, kn = x.shape[0], knobs()
    if (type(x) is not torch.Tensor or M <= 32 or type(M) is not int or not x.is_cuda or x.dtype is not torch.bfloat16 or _calls_are_seen() or _any_autocast()
            or _is_legacy_batched(x) or _is_wrapped(x) or torch.is_grad_enabled() or _forward_ad._current_level >= 0 or torch.compiler.is_compiling()
            or kn.fwd64 != "auto" or kn.skinny_gemm != "auto" or not _gemm64_enabled() or GEMM64_CONFIGS or GEMM64_SHAPE_CONFIGS or not use_native(x)
            or _steps.recorded or torch.cuda.is_current_stream_capturing()):
        return None
    forms = [_prompt_form(M, *s) for s in sizes]
    return None if None in forms else forms


def small_dgrad(dy2: torch.Tensor, w: torch.Tensor, out: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """``dy2 @ w`` on ``gemm_small`` (into ``out``) where it takes it; else None.  Weights whose sink was made to keep W^T copies stay with them."""
    if _calls_are_seen():
        return None
    M, (O, I) = dy2.shape[0], w.shape
    if dy2.dim() != 2 or dy2.shape[1] != O or not small_pays("dgrad", M, I, O) or knobs().dgrad64 != "auto" or torch.is_grad_enabled():
        return None
    sink = getattr(w, "_llmctl_grad_sink", None)
    if (sink is not None and sink.always_transpose) or not _small_ok("dgrad", M, I, O, dy2, w, *(() if out is None else (out,))):
        return None
    dx = torch.empty(M, I, dtype=dy2.dtype, device=dy2.device) if out is None else out
    native().gemm_small(dy2, w, dx, False, True, False)
    return dx


def small_wgrad(g: torch.Tensor, dy2: torch.Tensor, x2: torch.Tensor, accumulate: bool, gb: Optional[torch.Tensor] = None, add: bool = False) -> bool:
    """``g (+)= dy2^T x2`` (and ``gb (+)= dy2.sum(0)``) on ``gemm_small`` where it takes them; False: nothing done."""
    if _calls_are_seen():
        return False
    M, N, K = dy2.shape[1], x2.shape[1], dy2.shape[0]
    if not small_pays("wgrad", M, N, K, gb is not None) or not knobs().wgrad_kernel or torch.is_grad_enabled():
        return False
    if not _small_ok("wgrad", M, N, K, dy2, x2) or not _small_operand(g, (torch.bfloat16, torch.float32)):
        return False
    if gb is not None and not (gb.dtype == g.dtype and gb.is_contiguous() and gb.is_cuda and gb.numel() == M):
        return False
    native().gemm_small(dy2, x2, g, True, True, accumulate, None, gb, add)
    return True


def small_back(dy2: torch.Tensor, p: torch.nn.Parameter, w: torch.Tensor, x2: torch.Tensor,
               b: Optional[torch.nn.Parameter] = None) -> Optional[torch.Tensor]:
    """Both gradients of a sinked ``p`` (``w``: its values) and of its bias in one launch of ``gemm_small``'s tiles, where they take the two products and the weight's
    are no more than a round or two: the weight's (and bias's) into the sink, ``dy2 @ w`` returned; None: nothing done.  256 tokens, a step of the tiny model 306 us in two launches a
    layer's product, so 279."""
    sink: Optional[GradSink] = getattr(p, "_llmctl_grad_sink", None)
    T, (O, I) = dy2.shape[0], w.shape
    if (sink is None or _calls_are_seen() or sink.always_transpose or dy2.dim() != 2 or dy2.shape[1] != O or x2.shape != (T, I) or -(-O // 32) * -(-I // 32) > 512
            or not small_pays("dgrad", T, I, O) or not small_pays("wgrad", O, I, T) or torch.is_grad_enabled()
            or knobs().dgrad64 != "auto" or not knobs().wgrad_kernel):
        return None
    gb, add = None, False
    if b is not None:
        if getattr(b, "_llmctl_grad_sink", None) is not sink:
            return None
        gb, add = sink.open(b)
    g, more = sink.open(p)
    if (not _small_ok("dgrad", T, I, O, dy2, w) or not _small_ok("wgrad", O, I, T, x2) or not _small_operand(g, (torch.bfloat16, torch.float32))
            or not (gb is None or (gb.dtype == g.dtype and gb.is_contiguous() and gb.is_cuda and gb.numel() == O))):
        return None
    dx = torch.empty(T, I, dtype=dy2.dtype, device=dy2.device)
    native().gemm_small_back(dy2, w, dx, x2, g, more, gb, add)
    sink.close(p)
    if b is not None:
        sink.close(b)
    return dx


@functools.lru_cache(maxsize=4096)
def _back_splits(T: int, O: int, I: int, bias: bool) -> int:
    """The rule of ``gemm_tall_back`` (csrc/gemm_tall.hip), by size: ranges of the weight gradient, 0: two launches are as fast."""
    return native().gemm64_back_splits(T, O, I, bias)


def tall_back(dy2: torch.Tensor, p: torch.nn.Parameter, w: torch.Tensor, x2: torch.Tensor,
              b: Optional[torch.nn.Parameter] = None) -> Optional[torch.Tensor]:
    """:func:`small_back` on the 256 x 128 tiles (``gemm_tall_back``): both gradients of a sinked ``p`` in one launch where that takes less time than two; None: nothing
    done.  Steps of gpt2-125m, us: 8192 tokens 11450, so 11240; 3912 8360 / 7830; 1920 5750 / 5130; 1326 4880 /
    4440 (the data gradient was the library's there)."""
    sink: Optional[GradSink] = getattr(p, "_llmctl_grad_sink", None)
    T, (O, I) = dy2.shape[0], w.shape
    if (sink is None or O & 255 or I & 255 or T < 256 or T > DGRAD64_TOKENS or not w.is_cuda or _calls_are_seen() or sink.always_transpose or dy2.dim() != 2
            or dy2.shape[1] != O or x2.shape != (T, I) or not _back_splits(T, O, I, b is not None) or torch.is_grad_enabled() or knobs().dgrad64 != "auto"
            or not knobs().wgrad_kernel or gemm64_config("wgrad", O, I, T) // 100 != 3 or gemm64_config("dgrad", T, I, O) // 100 != 3):
        return None
    gb, add = None, False
    if b is not None:
        if getattr(b, "_llmctl_grad_sink", None) is not sink:
            return None
        gb, add = sink.open(b)
    g, more = sink.open(p)
    if (not _small_ok("dgrad", T, I, O, dy2, w) or not _small_ok("wgrad", O, I, T, x2) or not _small_operand(g, (torch.bfloat16, torch.float32))
            or not (gb is None or (gb.dtype == g.dtype and gb.is_contiguous() and gb.is_cuda and gb.numel() == O))
            or max(T * dy2.stride(0), T * x2.stride(0), O * w.stride(0)) >= 1 << 30):
        return None
    dx = torch.empty(T, I, dtype=dy2.dtype, device=dy2.device)
    native().gemm_tall_back(dy2, w, dx, x2, g, more, _back_splits(T, O, I, b is not None), gb, add)
    sink.close(p)
    if b is not None:
        sink.close(b)
    return dx


def dgrad64_shape_ok(tokens: int, w: torch.Tensor, fused: bool = False) -> bool:
    """Will ``dx = dy W`` for ``tokens`` rows run on gemm64?  (Decided at forward time: the
    weight's W^T copy is only kept for layers whose data gradient cannot.)  ``fused``: the
    down-projection data gradient with the SwiGLU backward in its epilogue.
    Knob ``dgrad64``: auto (default) = every data gradient that fits up to ``DGRAD64_TOKENS`` rows, beyond that as fused; fused = only
    the SwiGLU-fused down-projection data gradient on gemm64, the rest on hipBLASLt's forward layout through the W^T copies; all =
    every data gradient on gemm64 (no W^T copies, ~10 GB less memory for GPT-7B); off = none.  Whole steps, ms, gemm64 / W^T copies:
    tiny model, 256 tokens 1.89 / 2.84; gpt2-125m 1024 tokens 8.31 / 12.24, 8192 13.0 / 13.2; two GPT-7B layers 1024 tokens
    8.02 / 8.69, 8192 25.9 / 26.4, 16384 46.7 / 47.1, 24576 67.0 / 67.1 (a copy costs a pass over the weight, a launch and an event whatever
    the batch).  Beyond the limit nothing is gained: the full GPT-7B, two runs each, 24576 tokens 816.6, 818.0 / 816.5, 817.6, 32768 1073.8,
    1075.0 / 1071.1, 1071.3 (``profiles/dgrad_routes_full_model.txt``)."""
    out, inn = w.shape
    mode = knobs().dgrad64
    if mode == "off" or (not fused and (mode == "fused" or (mode == "auto" and tokens > DGRAD64_TOKENS))):
        return False
    return _gemm64_ok(tokens, inn, out, w) and out * w.stride(0) * 2 < 2**31


def dgrad64_rows(tokens: int, w: torch.Tensor) -> int:
    """Rows of a large weight's data gradient that gemm64 takes when ``tokens`` is no multiple of its 256-row tiles (knob dgrad64 = auto;
    else 0): whole tiles, the library multiplies the rest, which streams the weight once more and so takes 1536 rows to pay.  One
    GPT-7B layer, whole step, ms, this / W^T copies / W as it is: 540 tokens 5.36 / 5.36 / 5.14, 1000 6.10 / 6.06 / 5.91, 1710 7.54 / 7.81
    / 7.59, 3414 10.1 / 10.4 / 10.8, 8196 19.0 / 21.2 / 21.1."""
    rows = tokens // 256 * 256
    if knobs().dgrad64 != "auto" or tokens < 1536 or rows == tokens or w.numel() < 1 << 24 or not dgrad64_shape_ok(rows, w):
        return 0
    return rows


def _tied(w: torch.Tensor) -> bool:
    """A weight that is the embedding and the output projection.  It keeps no W^T copy: its data gradient runs on gemm64 whatever the tokens, us, W^T copy made
    and read / gemm64: 50304 x 768 16640 tokens 1510 / 1271, 20480 1529 / 1098, 50304 x 1024 20480 1630 / 1447, 32000 x 2048 20480 2511 / 1736."""
    return getattr(w, "_llmctl_writes", 1) > 1


def weight_t_ok(tokens: int, w: torch.Tensor) -> bool:
    """Does the data gradient of a sinked ``w`` for ``tokens`` rows go through a W^T copy?  Where it does not run on gemm64, and
    (knob dgrad64 = auto, unless its sink was made to keep copies) the layout's gain on the product covers the copy: weights of 2^24
    entries at 8192 rows and more.  Whole steps, ms, W^T copies / hipBLASLt reading W as it is: two GPT-7B layers 1024 tokens 8.69 /
    8.51, 4096 16.2 / 16.0, 8192 26.4 / 26.7, 16384 47.1 / 48.2; gpt2-125m (weights of at most 2^21.2 entries) 1024 tokens 12.2 /
    8.8, 8192 13.2 / 12.9, 32768 37.5 / 37.1."""
    sink = getattr(w, "_llmctl_grad_sink", None)
    if sink is None or _tied(w) or dgrad64_shape_ok(tokens, w):
        return False
    if sink.always_transpose or knobs().dgrad64 != "auto":
        return True
    return not dgrad64_rows(tokens, w) and tokens >= 8192 and w.numel() >= 1 << 24


def dgrad64_ok(dy2: torch.Tensor, w: torch.Tensor, fused: bool = False) -> bool:
    """``dx = dy W`` on gemm64 (W read K-major through ds_read_b64_tr_b16: no W^T copy)."""
    return (dy2.dim() == 2 and dy2.shape[1] == w.shape[0] and dgrad64_shape_ok(dy2.shape[0], w, fused)
            and dy2.is_cuda and dy2.dtype == torch.bfloat16 and _rows_ok(dy2))


def dgrad64(dy2: torch.Tensor, w: torch.Tensor, rows: Optional[int] = None) -> torch.Tensor:
    """``dy2 @ w`` on gemm64, rows from ``rows`` on (``dgrad64_rows``) in the library."""
    from llmctl.ops._lib import native

    T = dy2.shape[0]
    rows = T if rows is None else rows
    dx = torch.empty(T, w.shape[1], dtype=dy2.dtype, device=dy2.device)
    cfg = gemm64_config("dgrad", rows, w.shape[1], w.shape[0])
    native().gemm64_ex(dy2[:rows], w, dx[:rows], False, True, False, cfg)
    if rows < T:
        torch.mm(dy2[rows:], w, out=dx[rows:])
    return dx


def dgrad64_part(dy2: torch.Tensor, w: torch.Tensor) -> int:
    """``dgrad64_rows`` for these operands (0: not this way); weights whose sink keeps W^T copies stay with them."""
    sink = getattr(w, "_llmctl_grad_sink", None)
    if sink is None or sink.always_transpose or not (dy2.is_cuda and dy2.dtype == torch.bfloat16 and _rows_ok(dy2)):
        return 0
    return dgrad64_rows(dy2.shape[0], w)


def _gemm_ex_ok(g: torch.Tensor, dy2: torch.Tensor, x2: torch.Tensor) -> bool:
    """Shapes/layouts the hand-written MFMA wgrad kernel (llmctl/ops/csrc/gemm_bf16.hip) takes:
    M = out and N = in multiples of 256, K = tokens a multiple of 32, bf16, unit inner stride."""
    if not (g.is_cuda and g.dtype == torch.bfloat16 and dy2.dtype == torch.bfloat16 and x2.dtype == torch.bfloat16):
        return False
    from llmctl.ops._lib import use_native

    if not use_native(g) or not knobs().wgrad_kernel:  # off: hipBLASLt (A/B)
        return False
    M, N, K = dy2.shape[1], x2.shape[1], dy2.shape[0]
    if M % 256 or N % 256 or K % 32 or K == 0:
        return False
    for t in (g, dy2, x2):
        if t.stride(1) != 1 or t.stride(0) % 8 or t.data_ptr() % 16:
            return False
    # 32-bit buffer offsets inside the kernel
    return dy2.stride(0) * K * 2 < 2**31 and x2.stride(0) * K * 2 < 2**31


def _wgrad_whole(g: torch.Tensor, dy2: torch.Tensor, x2: torch.Tensor) -> bool:
    """Whether a weight whose rows are no multiple of 256 (a vocabulary) has its gradient made by gemm64 all the same: whole tiles, and a tile of their own for the
    rows behind them (``_whole_pays``)."""
    M, N, K = dy2.shape[1], x2.shape[1], dy2.shape[0]
    return (M % 256 != 0 and M % 8 == 0 and _whole_pays(M, N, K) and _gemm64_ok(M // 256 * 256, N, K, g, dy2, x2) and K * dy2.stride(0) * 2 < 2**31
            and K * x2.stride(0) * 2 < 2**31)


def _whole_pays(M: int, N: int, K: int) -> bool:
    """The second product and its copies are 16 us and more, so products from about 100 us on.  us, library / so: 8192 tokens 50304 x 768 642 / 499, 32136 x 4096 1935 / 1590; 3072
    tokens 50304 x 768 268 / 220, x 512 190 / 160, 8200 x 2048 127 / 102, but 12008 x 512 53 / 59, 32136 x 256 60 / 66, 32136 x 768 153 / 160; 6144 tokens 8200 x 768 91 / 102, 50304 x 256
    198 / 166; 2048 tokens 50304 x 768 204 / 204, 1024 107 / 107; 8192 tokens 5000 x 768 87 / 90, 40008 x 256 183 / 222."""
    return M >= 8192 and K >= 3072 and M * N * K >= (65e9 if M >= 40000 or N >= 2048 else 90e9) and (N >= 512 or M >= 49152)


def wgrad_into(g: torch.Tensor, dy2: torch.Tensor, x2: torch.Tensor, accumulate: bool) -> None:
    """``g (+)= dy2^T @ x2``: the MFMA kernels read both K-major operands through
    ds_read_b64_tr_b16 (gemm64: +20-40 % over hipBLASLt on the GPT-7B shapes,
    profiles/gemm64_variants_r2.jsonl; the 32-deep gemm_ex where K is not a multiple of 128);
    other shapes go to hipBLASLt."""
    M, N, K = dy2.shape[1], x2.shape[1], dy2.shape[0]
    if small_wgrad(g, dy2, x2, accumulate):
        return
    if g.dtype == torch.float32:  # fp32 main gradient: accumulate without a bf16 rounding
        if (_gemm64_ok(M, N, K, dy2, x2) and g.is_cuda and g.stride(1) == 1 and g.stride(0) % 4 == 0
                and g.data_ptr() % 16 == 0 and K * dy2.stride(0) * 2 < 2**31 and K * x2.stride(0) * 2 < 2**31):
            from llmctl.ops._lib import native

            native().gemm64_ex(dy2, x2, g, True, True, accumulate, gemm64_config("wgrad", M, N, K))
        elif K % 128 and wgrad_bias_into(g, dy2, x2, accumulate, None, False):
            pass
        elif accumulate:
            g.add_(dy2.t().matmul(x2))
        else:
            g.copy_(dy2.t().matmul(x2))
        return
    if (_gemm64_ok(M, N, K, g, dy2, x2) and K * dy2.stride(0) * 2 < 2**31 and K * x2.stride(0) * 2 < 2**31):
        from llmctl.ops._lib import native

        native().gemm64_ex(dy2, x2, g, True, True, accumulate, gemm64_config("wgrad", M, N, K))
    elif K % 128 and wgrad_bias_into(g, dy2, x2, accumulate, None, False):
        pass
    elif _gemm_ex_ok(g, dy2, x2):
        from llmctl.ops._lib import native

        native().gemm_ex(dy2, x2, g, True, True, accumulate)
    elif _wgrad_whole(g, dy2, x2):
        from llmctl.ops._lib import native

        whole = M // 256 * 256
        last = torch.empty(256, N, dtype=torch.float32, device=g.device)  # a tile that ends at the last row
        if accumulate:  # (the library's add of fp32 rows to bf16 ones takes 47 us, the two copies 3 each)
            last.copy_(g[M - 256:])
        native().gemm64_ex(dy2[:, :whole], x2, g[:whole], True, True, accumulate, gemm64_config("wgrad", whole, N, K))
        native().gemm64_ex(dy2[:, M - 256:], x2, last, True, True, accumulate, gemm64_config("wgrad", 256, N, K))
        g[whole:].copy_(last[256 - (M - whole):])
    elif accumulate:
        g.addmm_(dy2.t(), x2)
    else:
        torch.mm(dy2.t(), x2, out=g)


@functools.lru_cache(maxsize=4096)
def _bias_rides(M: int, N: int, K: int, bias: bool) -> bool:
    """Whether the 256 x 128 tiles take a weight gradient of these sizes (``gemm64_wgrad_splits``).  Kept by size: a call that was refused cost the host 5 us, and a
    backward that is bound by its launches two of them a layer (300 tokens, 8192 x 2048 with a bias 43.5 us, so 31)."""
    from llmctl.ops._lib import native

    return native().gemm64_wgrad_splits(M, N, K, bias) > 0


def wgrad_bias_into(g: torch.Tensor, dy2: torch.Tensor, x2: torch.Tensor, accumulate: bool, gb: Optional[torch.Tensor], add: bool) -> bool:
    """``g (+)= dy2^T x2`` and ``gb (+)= dy2.sum(0)`` in one kernel where the 256 x 128 tiles take the weight gradient, over any number of tokens from 256 on
    (without ``gb`` where they are no multiple of 128); False: nothing done."""
    M, N, K = dy2.shape[1], x2.shape[1], dy2.shape[0]
    if gb is not None and small_wgrad(g, dy2, x2, accumulate, gb, add):
        return True
    if M % 256 or N % 256 or K < 256 or not dy2.is_cuda or not _bias_rides(M, N, K, gb is not None):  # (most refusals end here)
        return False
    if not (_gemm64_ok(M, N, 128, dy2, x2) and g.is_cuda and g.dtype in (torch.bfloat16, torch.float32)
            and (gb is None or (gb.dtype == g.dtype and gb.is_contiguous()))
            and g.stride(1) == 1 and g.stride(0) % 8 == 0 and g.data_ptr() % 16 == 0
            and K * dy2.stride(0) * 2 < 2**31 and K * x2.stride(0) * 2 < 2**31 and gemm64_config("wgrad", M, N, K) // 100 == 3):
        return False
    from llmctl.ops._lib import native

    return native().gemm64_wgrad_bias(dy2, x2, g, accumulate, gb, add)


def side_chunks(M: int, N: int, K: int, T: int, F: int) -> int:
    """Chunks of 1024 elements per K-tile that ``gemm64_wgrad_swiglu``'s side job needs to cover
    ``T * F`` elements over the K-tiles of an ``[M, N] x K`` weight gradient (0: unsupported) —
    as ``side_chunks`` in gemm64.hip."""
    ktiles = (M // 256) * (N // 256) * (K // 64)
    E = T * F
    if E * 4 >= 2**31 or F % 2:
        return 0
    for ch in (1, 2):
        if ktiles * 1024 * ch >= E and ktiles * 1024 * ch < 2**32 and F >= 1024 * ch:
            return ch
    return 0


def swiglu_side_mode() -> str:
    """Where the MLP's SwiGLU backward runs (knob ``swiglu_bwd``): ``side`` (default) = as a side
    job of the down projection's weight-gradient GEMM (``gemm64_wgrad_swiglu``), the data
    gradient a plain GEMM; ``epilogue`` = in the data-gradient GEMM's store epilogue
    (``gemm64_swiglu_dgrad``, round 2); ``separate`` = separate elementwise kernel."""
    return knobs().swiglu_bwd


def wgrad_swiglu_ok(w: torch.nn.Parameter, tokens: int, F: int) -> bool:
    """Can ``w``'s (down projection, [H, F]) weight gradient over ``tokens`` rows carry the SwiGLU
    backward as a side job?  Needs the grad sink (the GEMM writes the flat gradient view)."""
    if swiglu_side_mode() != "side" or getattr(w, "_llmctl_grad_sink", None) is None or not w.is_cuda:
        return False
    H = w.shape[0]
    return (_gemm64_enabled() and w.dtype == torch.bfloat16 and H % 256 == 0 and F % 256 == 0
            and tokens % 128 == 0 and tokens > 0 and side_chunks(H, F, tokens, tokens, F) > 0)


def wgrad_swiglu_into(g: torch.Tensor, dy2: torch.Tensor, x2: torch.Tensor, accumulate: bool,
                      dact: torch.Tensor, gu: torch.Tensor) -> Optional[torch.Tensor]:
    """``g (+)= dy2^T x2`` with ``dgu = swiglu_bwd(dact, gu)`` computed by the same kernel
    (returned); None when the operands do not fit (the caller falls back)."""
    M, N, K = dy2.shape[1], x2.shape[1], dy2.shape[0]
    if not (_gemm64_ok(M, N, K, dy2, x2) and g.is_cuda and g.dtype in (torch.bfloat16, torch.float32)
            and g.stride(1) == 1 and g.stride(0) % 8 == 0 and g.data_ptr() % 16 == 0
            and K * dy2.stride(0) * 2 < 2**31 and K * x2.stride(0) * 2 < 2**31
            and dact.is_contiguous() and gu.is_contiguous() and dact.shape == (K, N) and gu.shape == (K, 2 * N)
            and dact.dtype == torch.bfloat16 and gu.dtype == torch.bfloat16
            and side_chunks(M, N, K, K, N) > 0):
        return None
    from llmctl.ops._lib import native

    return native().gemm64_wgrad_swiglu(dy2, x2, g, accumulate, dact, gu, gemm64_config("wgrad", M, N, K))


class GradSink:
    def __init__(self, transpose_dgrad: Optional[bool] = None):
        self.callbacks: List[Callable[[torch.nn.Parameter], None]] = []
        self.always_transpose = bool(transpose_dgrad)  # asked for here: whatever the sizes
        if transpose_dgrad is None:
            transpose_dgrad = knobs().dgrad_transpose
        self.transpose_dgrad = transpose_dgrad
        self.epoch = 0  # bumped by the engine after every optimizer step / weight load

    def weight_t(self, w: torch.nn.Parameter) -> Optional[torch.Tensor]:
        """The up-to-date ``W^T`` copy of a 2-D bf16 GPU weight (None if not applicable)."""
        if not (self.transpose_dgrad and w.is_cuda and w.dim() == 2 and w.dtype == torch.bfloat16):
            return None
        from llmctl.ops._lib import native, use_native

        if not use_native(w) or w.shape[0] % 8 or w.shape[1] % 8:
            return None
        wt = getattr(w, "_llmctl_wt", None)
        if wt is None:
            wt = torch.empty(w.shape[1], w.shape[0], dtype=w.dtype, device=w.device)
            w._llmctl_wt = wt
            w._llmctl_wt_epoch = -1
        if w._llmctl_wt_epoch != self.epoch:
            if self._side_stream_ok():
                # the copy is only read by the backward's data-gradient GEMM: transpose on a side
                # stream under the forward's compute-bound GEMMs; wait_weight_t() orders the
                # backward after it (and, through the backward, the next optimizer step)
                cur = torch.cuda.current_stream(w.device)
                side = self._side_stream(w.device)
                side.wait_stream(cur)
                with torch.cuda.stream(side):
                    native().transpose_(w.detach(), wt)
                ev = torch.cuda.Event()
                ev.record(side)
                w._llmctl_wt_event = ev
            else:
                native().transpose_(w.detach(), wt)
                w._llmctl_wt_event = None
            w._llmctl_wt_epoch = self.epoch
        return wt

    @staticmethod
    def wait_weight_t(w: torch.nn.Parameter) -> None:
        """Order the current stream after the side-stream refresh of ``w``'s W^T copy."""
        ev = getattr(w, "_llmctl_wt_event", None)
        if ev is not None:
            torch.cuda.current_stream(w.device).wait_event(ev)

    _streams: dict = {}

    @staticmethod
    def _side_stream_ok() -> bool:
        return knobs().wt_side_stream and not torch.cuda.is_current_stream_capturing()

    @classmethod
    def _side_stream(cls, device) -> "torch.cuda.Stream":
        s = cls._streams.get(device)
        if s is None:
            s = cls._streams[device] = torch.cuda.Stream(device=device)
        return s

    def attach(self, p: torch.nn.Parameter, writes: int = 1) -> None:
        """``writes``: the gradients that one backward writes (2: an embedding that is the output projection too); the last of them
        is what the callbacks are told of."""
        p._llmctl_grad_sink = self
        p._llmctl_writes = p._llmctl_pending = writes
        p._llmctl_fresh = True

    def reset(self, p: torch.nn.Parameter) -> None:
        p._llmctl_fresh = True
        p._llmctl_pending = p._llmctl_writes

    @staticmethod
    def _target(p: torch.nn.Parameter) -> torch.Tensor:
        g = getattr(p, "main_grad", None)
        if g is None:
            g = p.grad
        if g is None:
            raise RuntimeError("grad sink parameter has no flat .grad view")
        return g

    def _written(self, p: torch.nn.Parameter) -> None:
        p._llmctl_fresh = False
        p._llmctl_pending -= 1
        if p._llmctl_pending > 0:
            return
        p._llmctl_pending = p._llmctl_writes
        for cb in self.callbacks:
            cb(p)

    def open(self, p: torch.nn.Parameter) -> Tuple[torch.Tensor, bool]:
        """A vector's flat gradient for a kernel to write, and whether it adds to it; ``close`` follows the launch."""
        return self._target(p), not p._llmctl_fresh

    close = _written

    def add(self, p: torch.nn.Parameter, g: torch.Tensor) -> None:
        """A gradient computed elsewhere (CPU and fp32 paths)."""
        t = self._target(p)
        t.copy_(g) if p._llmctl_fresh else t.add_(g)
        self._written(p)

    def write(self, p: torch.nn.Parameter, dy2: torch.Tensor, x2: torch.Tensor) -> None:
        wgrad_into(self._target(p), dy2, x2, accumulate=not p._llmctl_fresh)
        self._written(p)

    def write_with_bias(self, p: torch.nn.Parameter, dy2: torch.Tensor, x2: torch.Tensor, b: torch.nn.Parameter) -> bool:
        """``write`` with the bias ``b``'s gradient summed by the same kernel; False: it does not take them, nothing is written."""
        if getattr(b, "_llmctl_grad_sink", None) is not self:
            return False
        gb, add = self.open(b)
        if not wgrad_bias_into(self._target(p), dy2, x2, not p._llmctl_fresh, gb, add):
            return False
        self._written(p)
        self.close(b)
        return True

    def write_swiglu(self, p: torch.nn.Parameter, dy2: torch.Tensor, x2: torch.Tensor, dact: torch.Tensor,
                     gu: torch.Tensor) -> Optional[torch.Tensor]:
        """``write`` with the SwiGLU backward riding on the weight-gradient GEMM: returns
        ``dgu = swiglu_bwd(dact, gu)``, or None (nothing written) if the kernel cannot take it."""
        dgu = wgrad_swiglu_into(self._target(p), dy2, x2, not p._llmctl_fresh, dact, gu)
        if dgu is not None:
            self._written(p)
        return dgu


def bias_grad(b: torch.nn.Parameter, dy2: torch.Tensor) -> Optional[torch.Tensor]:
    """Column sums of ``dy2``: into ``b``'s flat gradient if it has a sink (returns None), else as an ordinary gradient."""
    from llmctl import ops

    sink: Optional[GradSink] = getattr(b, "_llmctl_grad_sink", None)
    if sink is not None:
        g, add = sink.open(b)
        ops.col_sum_(dy2, g, add)
        sink.close(b)
        return None
    if torch.is_grad_enabled():  # a backward that is differentiated itself (create_graph)
        return dy2.sum(0)
    db = torch.empty(b.shape, dtype=dy2.dtype, device=dy2.device)
    ops.col_sum_(dy2, db, False)
    return db


class _Linear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, b):
        ctx.save_for_backward(x, w)
        # keep the Parameter object itself: tensors coming back from saved_tensors can be
        # aliases (e.g. under activation checkpointing) that do not carry the sink
        ctx.wparam, ctx.bparam = w, b
        sink = getattr(w, "_llmctl_grad_sink", None)
        ctx.wt = None
        if ctx.needs_input_grad[0] and weight_t_ok(x.numel() // x.shape[-1], w):
            ctx.wt = sink.weight_t(w)
        return forward_linear(x, w, b, "fwd")

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        dy2 = dy.reshape(-1, dy.shape[-1])
        x2 = x.reshape(-1, x.shape[-1])
        dw = None
        bias = ctx.bparam is not None and ctx.needs_input_grad[2]
        if ctx.needs_input_grad[0] and ctx.needs_input_grad[1] and ctx.wt is None:
            dx = small_back(dy2, ctx.wparam, w, x2, ctx.bparam if bias else None)
            if dx is None:
                dx = tall_back(dy2, ctx.wparam, w, x2, ctx.bparam if bias else None)
            if dx is not None:
                return dx.view(*dy.shape[:-1], w.shape[1]), None, None
        if ctx.needs_input_grad[1]:
            sink: Optional[GradSink] = getattr(ctx.wparam, "_llmctl_grad_sink", None)
            if sink is not None and bias and sink.write_with_bias(ctx.wparam, dy2, x2, ctx.bparam):
                bias = False
            elif sink is not None:
                sink.write(ctx.wparam, dy2, x2)  # weight grad first: lets its bucket's comm start earlier
            else:  # an ordinary gradient (AccumulateGrad adds it), still on the MFMA kernels when they fit
                dw = torch.empty_like(w)
                wgrad_into(dw, dy2, x2, accumulate=False)
        dx = None
        if ctx.needs_input_grad[0]:
            # an unsinked or tied weight keeps no W^T copy, so its alternative is hipBLASLt's slower "NN"
            # layout: gemm64 (W read K-major) whenever the shape fits, unless knob dgrad64 is off
            free = (getattr(ctx.wparam, "_llmctl_grad_sink", None) is None or _tied(ctx.wparam)) and knobs().dgrad64 != "off"
            dx = small_dgrad(dy2, w) if ctx.wt is None else None
            if dx is not None:
                dx = dx.view(*dy.shape[:-1], w.shape[1])
            elif dgrad64_ok(dy2, w) or (free and dy2.is_cuda and dy2.dtype == torch.bfloat16 and _rows_ok(dy2)
                                      and _gemm64_ok(dy2.shape[0], w.shape[1], w.shape[0], w)
                                      and w.shape[0] * w.stride(0) * 2 < 2**31):
                dx = dgrad64(dy2, w).view(*dy.shape[:-1], w.shape[1])
            elif dgrad64_part(dy2, ctx.wparam):
                dx = dgrad64(dy2, w, dgrad64_part(dy2, ctx.wparam)).view(*dy.shape[:-1], w.shape[1])
            elif ctx.wt is not None:
                GradSink.wait_weight_t(ctx.wparam)
                dx = F.linear(dy, ctx.wt)
            else:
                dx = dy.matmul(w)
        db = bias_grad(ctx.bparam, dy2) if bias else None
        return dx, dw, db


def linear(x: torch.Tensor, w: torch.Tensor, b: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``x @ w^T (+ b)`` (``forward_linear``: gemm64 or hipBLASLt); weight grads go through the
    parameter's sink if any.  Whenever a gradient is needed the call goes through ``_Linear`` — the
    gemm64 forward is a plain kernel call that autograd cannot see, so an unsinked weight (MoE
    experts, tied heads) taking that route from ``forward_linear`` directly would get no gradient."""
    needs_grad = torch.is_grad_enabled() and (x.requires_grad or w.requires_grad
                                              or (b is not None and b.requires_grad))
    if not needs_grad:
        return forward_linear(x, w, b)
    return _Linear.apply(x, w, b)


class _Embedding(torch.autograd.Function):
    @staticmethod
    def forward(ctx, ids, w):
        from llmctl import ops

        ctx.save_for_backward(ids)
        ctx.wparam = w
        return ops.embed_rows(ids, w)

    @staticmethod
    def backward(ctx, dy):
        from llmctl import ops

        (ids,) = ctx.saved_tensors
        if ctx.needs_input_grad[1]:
            w = ctx.wparam
            sink: GradSink = w._llmctl_grad_sink
            dy2 = dy.reshape(-1, dy.shape[-1])
            g, add = sink.open(w)
            ok = ops.embed_grad_ok(ids, dy2, g)
            if ok and ops.embed_grad_pays(dy2.shape[0], dy2.shape[1], g.shape[0]):
                ops.embed_grad_(ids, dy2, g, add)
                sink.close(w)
            else:
                if ok and (add or g.dtype == torch.float32):  # (the sums in fp32 up to the flat gradient, as the kernel holds them)
                    dy2 = dy2.float()
                sink.add(w, torch.ops.aten.embedding_dense_backward(dy2, ids, w.shape[0], -1, False))
        return None, None


def embedding(ids: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``w[ids]`` for ids ``[T]``; the gradient of a weight with a sink goes straight into its flat gradient."""
    if torch.is_grad_enabled() and w.requires_grad and getattr(w, "_llmctl_grad_sink", None) is not None:
        return _Embedding.apply(ids, w)
    return F.embedding(ids, w)


def data_grad(dy: torch.Tensor, w: torch.nn.Parameter) -> torch.Tensor:
    """``dy @ w`` for hand-written backward passes: gemm64 when the shape fits, else through
    the weight's transposed copy when its sink keeps one."""
    dy2 = dy.reshape(-1, dy.shape[-1])
    dx = small_dgrad(dy2, w)
    if dx is not None:
        return dx.view(*dy.shape[:-1], w.shape[1])
    if dgrad64_ok(dy2, w):
        return dgrad64(dy2, w).view(*dy.shape[:-1], w.shape[1])
    if dgrad64_part(dy2, w):
        return dgrad64(dy2, w, dgrad64_part(dy2, w)).view(*dy.shape[:-1], w.shape[1])
    wt = w._llmctl_grad_sink.weight_t(w) if weight_t_ok(dy2.shape[0], w) else None
    if wt is not None:
        GradSink.wait_weight_t(w)
        return F.linear(dy, wt)
    return dy.matmul(w)


def data_grad_into(dy2: torch.Tensor, w: torch.nn.Parameter, out: torch.Tensor) -> None:
    """``out = dy2 @ w`` into a preallocated (row-slice) output: gemm64 writes it directly."""
    if small_dgrad(dy2, w, out) is not None:
        return
    if dgrad64_ok(dy2, w) and _rows_ok(out):
        from llmctl.ops._lib import native

        native().gemm64_ex(dy2, w, out, False, True, False, gemm64_config("dgrad", dy2.shape[0], w.shape[1], w.shape[0]))
        return
    out.copy_(data_grad(dy2, w))


def swiglu_data_grad(dy: torch.Tensor, w: torch.nn.Parameter, gu: torch.Tensor) -> torch.Tensor:
    """``swiglu_bwd(dy @ w, gu)`` for the MLP down projection: on gemm64 the SwiGLU backward runs
    in the data-gradient GEMM's epilogue (``gemm64_swiglu_dgrad``: dgate / dup from the fp32 dAct
    tile, no dAct tensor); otherwise the data gradient and the elementwise kernel separately."""
    dy2 = dy.reshape(-1, dy.shape[-1])
    gu2 = gu.reshape(-1, gu.shape[-1])
    if (dgrad64_ok(dy2, w, fused=True) and gu2.is_contiguous() and gu2.data_ptr() % 16 == 0
            and swiglu_side_mode() != "separate"):  # separate: unfused (A/B)
        from llmctl.ops._lib import native

        cfg = gemm64_config("dgrad", dy2.shape[0], w.shape[1], w.shape[0])
        return native().gemm64_swiglu_dgrad(dy2, w, gu2, cfg).view(gu.shape)
    from llmctl.ops._lib import native, use_native
    from llmctl.ops import ref

    dact = data_grad(dy, w)
    return native().swiglu_bwd(dact, gu) if use_native(gu) else ref.swiglu_bwd(dact, gu)


def weight_grad(w: torch.nn.Parameter, dy2: torch.Tensor, x2: torch.Tensor) -> Optional[torch.Tensor]:
    """For hand-written backward passes: route ``dy2^T x2`` through ``w``'s sink (returns
    None) or return it as an ordinary gradient."""
    sink = getattr(w, "_llmctl_grad_sink", None)
    if sink is not None:
        sink.write(w, dy2, x2)
        return None
    return dy2.t().matmul(x2)

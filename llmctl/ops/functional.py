"""Autograd-facing fused ops.  GPU tensors run the hand-written CDNA4 HIP kernels in
``csrc/`` (``torch.ops.llmctl.*``); CPU tensors run the fp32 oracle in :mod:`.ref`.

Every op keeps the layouts the GEMMs (hipBLASLt) produce/consume so no transposes or
copies are needed between kernels:

* activations are token-major ``[T, features]`` (T = batch*seq);
* attention takes ``q [B,S,Hq,D]``, ``k/v [B,S,Hkv,D]`` (GQA), returns ``o [B,S,Hq,D]``
  which *is* the ``[T, Hq*D]`` input of the output projection;
* RoPE is fused with the QKV split: ``[T,(Hq+2Hkv)D] -> q,k (rotated), v``.
"""

from __future__ import annotations

import functools
from typing import List, Optional, Tuple

import torch

from llmctl.config.knobs import knobs

from . import ref
from ._lib import native, use_native


# =============================================================================== norms
def _norm_grads(ctx, dy2, x2, w, mu, rstd, dres2):
    """(dx, dw, db) of a norm over the rows ``x2`` (``mu`` None: RMS norm, db None).  Every vector for itself: one that needs a gradient
    and has a sink (``llmctl.exec.linear.GradSink``) has it written into the flat gradient, by the kernel, and gets None; one without a
    sink gets an ordinary gradient; a frozen one gets None and leaves the other as it is."""
    params, needed = ctx.norm_params, ctx.needs_input_grad[ctx.norm_at:ctx.norm_at + len(ctx.norm_params)]
    sinks = [getattr(p, "_llmctl_grad_sink", None) if need else None for p, need in zip(params, needed)]
    if use_native(dy2) and any(s is not None for s in sinks):
        outs = [s.open(p) if s is not None else None for p, s in zip(params, sinks)]
        kind = next(o[0].dtype for o in outs if o is not None)  # (the kernel's two sums share a type)
        outs = [(torch.empty(p.shape, dtype=kind, device=dy2.device), False) if o is None else o for p, o in zip(params, outs)]
        (dw, add_w), (db, add_b) = outs[0], (outs[1] if mu is not None else (None, False))
        dx = native().norm_bwd_into(dy2, x2, w, mu, rstd, dres2, dw, add_w, db, add_b)
        grads = [None if s is not None or not need else o[0].to(p.dtype) for p, s, need, o in zip(params, sinks, needed, outs)]
        for p, s in zip(params, sinks):
            if s is not None:
                s.close(p)
    else:
        k = native() if use_native(dy2) else ref
        if mu is None:
            dx, *sums = k.rmsnorm_bwd(dy2, x2, w, rstd, dres2)
        else:
            dx, *sums = k.layernorm_bwd(dy2, x2, w, mu, rstd, dres2)
        grads = []
        for p, s, need, g in zip(params, sinks, needed, sums):
            if s is not None:
                s.add(p, g)
            grads.append(g if need and s is None else None)
    return dx, grads[0], grads[1] if mu is not None else None


class _RMSNorm(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, eps):
        x2 = x.reshape(-1, x.shape[-1])
        if use_native(x):
            y, rstd = native().rmsnorm_fwd(x2, w, eps)
        else:
            y, rstd = ref.rmsnorm_fwd(x2, w, eps)
        ctx.save_for_backward(x2, w, rstd)
        ctx.shape, ctx.norm_params, ctx.norm_at = x.shape, (w,), 1
        return y.view(x.shape)

    @staticmethod
    def backward(ctx, dy):
        x2, w, rstd = ctx.saved_tensors
        dy2 = dy.reshape(-1, x2.shape[-1]).contiguous()
        dx, dw, _ = _norm_grads(ctx, dy2, x2, w, None, rstd, None)
        return dx.view(ctx.shape), dw, None


class _AddRMSNorm(torch.autograd.Function):
    """res_out = x + residual ; y = rmsnorm(res_out) * w.  One HBM pass for both."""

    @staticmethod
    def forward(ctx, x, residual, w, eps):
        H = x.shape[-1]
        x2, r2 = x.reshape(-1, H), residual.reshape(-1, H)
        if use_native(x):
            y, res_out, rstd = native().add_rmsnorm_fwd(x2, r2, w, eps)
        else:
            res_out = (x2.float() + r2.float()).to(x.dtype)
            y, rstd = ref.rmsnorm_fwd(res_out, w, eps)
        ctx.save_for_backward(res_out, w, rstd)
        ctx.shape, ctx.norm_params, ctx.norm_at = x.shape, (w,), 2
        return y.view(x.shape), res_out.view(x.shape)

    @staticmethod
    def backward(ctx, dy, dres):
        res_out, w, rstd = ctx.saved_tensors
        H = res_out.shape[-1]
        dy2 = dy.reshape(-1, H).contiguous()
        dres2 = dres.reshape(-1, H).contiguous() if dres is not None else None
        dx, dw, _ = _norm_grads(ctx, dy2, res_out, w, None, rstd, dres2)
        dx = dx.view(ctx.shape)
        return dx, dx, dw, None


class _LayerNorm(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, b, eps):
        x2 = x.reshape(-1, x.shape[-1])
        if use_native(x):
            y, mu, rstd = native().layernorm_fwd(x2, w, b, eps)
        else:
            y, mu, rstd = ref.layernorm_fwd(x2, w, b, eps)
        ctx.save_for_backward(x2, w, mu, rstd)
        ctx.shape, ctx.norm_params, ctx.norm_at = x.shape, (w, b), 1
        return y.view(x.shape)

    @staticmethod
    def backward(ctx, dy):
        x2, w, mu, rstd = ctx.saved_tensors
        dy2 = dy.reshape(-1, x2.shape[-1]).contiguous()
        dx, dw, db = _norm_grads(ctx, dy2, x2, w, mu, rstd, None)
        return dx.view(ctx.shape), dw, db, None


class _AddLayerNorm(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, residual, w, b, eps):
        H = x.shape[-1]
        x2, r2 = x.reshape(-1, H), residual.reshape(-1, H)
        if use_native(x):
            y, res_out, mu, rstd = native().add_layernorm_fwd(x2, r2, w, b, eps)
        else:
            res_out = (x2.float() + r2.float()).to(x.dtype)
            y, mu, rstd = ref.layernorm_fwd(res_out, w, b, eps)
        ctx.save_for_backward(res_out, w, mu, rstd)
        ctx.shape, ctx.norm_params, ctx.norm_at = x.shape, (w, b), 2
        return y.view(x.shape), res_out.view(x.shape)

    @staticmethod
    def backward(ctx, dy, dres):
        res_out, w, mu, rstd = ctx.saved_tensors
        H = res_out.shape[-1]
        dy2 = dy.reshape(-1, H).contiguous()
        dres2 = dres.reshape(-1, H).contiguous() if dres is not None else None
        dx, dw, db = _norm_grads(ctx, dy2, res_out, w, mu, rstd, dres2)
        dx = dx.view(ctx.shape)
        return dx, dx, dw, db, None


def rmsnorm(x, w, eps: float = 1e-5):
    return _RMSNorm.apply(x, w, eps)


def add_rmsnorm(x, residual, w, eps: float = 1e-5):
    return _AddRMSNorm.apply(x, residual, w, eps)


def layernorm(x, w, b, eps: float = 1e-5):
    return _LayerNorm.apply(x, w, b, eps)


def add_layernorm(x, residual, w, b, eps: float = 1e-5):
    return _AddLayerNorm.apply(x, residual, w, b, eps)


# =============================================================================== rope
class _RopeQKV(torch.autograd.Function):
    @staticmethod
    def forward(ctx, qkv, cos, sin, nq, nkv, seq_len, positions):
        if use_native(qkv):
            q, k, v = native().rope_qkv_fwd(qkv, cos, sin, nq, nkv, seq_len, positions)
        else:
            q, k, v = ref.rope_qkv_fwd(qkv, cos, sin, nq, nkv, seq_len, positions)
        ctx.save_for_backward(cos, sin, positions if positions is not None else torch.empty(0))
        ctx.has_pos = positions is not None
        ctx.seq_len = seq_len
        return q, k, v

    @staticmethod
    def backward(ctx, dq, dk, dv):
        cos, sin, pos = ctx.saved_tensors
        pos = pos if ctx.has_pos else None
        dq, dk, dv = dq.contiguous(), dk.contiguous(), dv.contiguous()
        if use_native(dq):
            dqkv = native().rope_qkv_bwd(dq, dk, dv, cos, sin, ctx.seq_len, pos)
        else:
            dqkv = ref.rope_qkv_bwd(dq, dk, dv, cos, sin, ctx.seq_len, pos)
        return dqkv, None, None, None, None, None, None


def rope_qkv(qkv, cos, sin, nq: int, nkv: int, seq_len: int, positions: Optional[torch.Tensor] = None):
    """``qkv [T,(nq+2nkv)*D]`` -> ``q [T,nq,D], k [T,nkv,D], v [T,nkv,D]`` with RoPE on q,k."""
    return _RopeQKV.apply(qkv, cos, sin, nq, nkv, seq_len, positions)


def rope_qkv_cache(qkv, cos, sin, nq: int, nkv: int, seq_len: int, positions, k_cache, v_cache, slots):
    """Inference: ``rope_qkv`` that also writes the rotated K and V rows into the paged cache at
    ``slots`` (int64 [T], -1 = skip) in the same pass."""
    if use_native(qkv):
        return native().rope_qkv_cache_fwd(qkv, cos, sin, nq, nkv, seq_len, positions, k_cache, v_cache, slots)
    q, k, v = ref.rope_qkv_fwd(qkv, cos, sin, nq, nkv, seq_len, positions)
    ref.kv_cache_write(k, v, k_cache, v_cache, slots)
    return q, k, v


# =============================================================================== attention
class _FlashAttn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, scale, causal, doc_start):
        if use_native(q):
            o, lse = native().flash_attn_fwd(q, k, v, scale, causal, doc_start)
        else:
            o, lse = ref.attention_fwd(q, k, v, scale, causal, doc_start)
        ctx.save_for_backward(q, k, v, o, lse)
        ctx.scale, ctx.causal, ctx.doc_start = scale, causal, doc_start
        return o

    @staticmethod
    def backward(ctx, do):
        q, k, v, o, lse = ctx.saved_tensors
        do = do.contiguous()
        if use_native(do):
            dq, dk, dv = native().flash_attn_bwd(do, q, k, v, o, lse, ctx.scale, ctx.causal, ctx.doc_start)
        else:
            dq, dk, dv = ref.attention_bwd(do, q, k, v, o, lse, ctx.scale, ctx.causal, ctx.doc_start)
        return dq, dk, dv, None, None, None


def flash_attention(q, k, v, causal: bool = True, softmax_scale: Optional[float] = None,
                    doc_start: Optional[torch.Tensor] = None):
    """Causal flash attention.  q ``[B,S,Hq,D]``, k/v ``[B,S,Hkv,D]`` (Hq % Hkv == 0).
    ``doc_start`` (int32 ``[B,S]``, packed sequences): attention stays inside each document."""
    scale = softmax_scale if softmax_scale is not None else q.shape[-1] ** -0.5
    return _FlashAttn.apply(q, k, v, scale, causal, doc_start)


class _RopeFlashAttn(torch.autograd.Function):
    """``rope_qkv`` + ``flash_attention`` with the RoPE backward fused into the attention
    backward's dQ / dK stores (``flash_attn_bwd_qkv``): the backward writes the QKV-projection
    gradient dqkv [T, (nq+2nkv)*D] directly — no dq/dk/dv tensors and no rope_bwd pass."""

    @staticmethod
    def forward(ctx, qkv, cos, sin, nq, nkv, B, S, positions, doc_start, inplace=False):
        if inplace:
            # the caller owns qkv (a projection output nothing else saved): rotate its q / k heads
            # in place and attend strided views of it — V is neither copied nor re-read
            native().rope_qk_inplace_(qkv, cos, sin, nq, nkv, S, positions)
            D = qkv.shape[-1] // (nq + 2 * nkv)
            qkv4 = qkv.view(B, S, nq + 2 * nkv, D)
            q, k, v = qkv4[:, :, :nq], qkv4[:, :, nq:nq + nkv], qkv4[:, :, nq + nkv:]
        else:
            q, k, v = native().rope_qkv_fwd(qkv, cos, sin, nq, nkv, S, positions)
            D = q.shape[-1]
            q, k, v = q.view(B, S, nq, D), k.view(B, S, nkv, D), v.view(B, S, nkv, D)
        scale = D ** -0.5
        o, lse = native().flash_attn_fwd(q, k, v, scale, True, doc_start)
        pos = positions.reshape(-1).int().contiguous() if positions is not None else None
        ctx.save_for_backward(q, k, v, o, lse, cos, sin, pos if pos is not None else torch.empty(0))
        ctx.has_pos, ctx.S, ctx.scale, ctx.doc_start = pos is not None, S, scale, doc_start
        return o

    @staticmethod
    def backward(ctx, do):
        q, k, v, o, lse, cos, sin, pos = ctx.saved_tensors
        dqkv = native().flash_attn_bwd_qkv(do.contiguous(), q, k, v, o, lse, ctx.scale, True, ctx.doc_start, cos, sin,
                                           pos if ctx.has_pos else None, ctx.S)
        return dqkv, None, None, None, None, None, None, None, None, None


def rope_flash_attention(qkv, cos, sin, nq: int, nkv: int, B: int, S: int, positions=None, doc_start=None,
                         inplace: bool = False):
    """Causal attention on the QKV projection output: RoPE(q, k) -> flash attention -> o
    ``[B,S,nq,D]``; the backward returns d(qkv) in one fused pass on the HIP path.  ``inplace``
    (HIP path; the caller's qkv must not be needed afterwards): RoPE rotates qkv's q / k heads in
    place and attention reads strided views (knob ``rope_inplace`` off disables)."""
    if use_native(qkv) and qkv.is_contiguous():
        inplace = inplace and knobs().rope_inplace
        return _RopeFlashAttn.apply(qkv, cos, sin, nq, nkv, B, S, positions, doc_start, inplace)
    q, k, v = rope_qkv(qkv, cos, sin, nq, nkv, S, positions)
    D = q.shape[-1]
    return flash_attention(q.view(B, S, nq, D), k.view(B, S, nkv, D), v.view(B, S, nkv, D), causal=True,
                           doc_start=doc_start)


class _QKVFlashAttn(torch.autograd.Function):
    """Causal flash attention of strided views of the QKV projection output (no rotation); the backward writes the
    projection's gradient dqkv [T, (nq+2nkv)*D] directly."""

    @staticmethod
    def forward(ctx, qkv, nq, nkv, B, S, doc_start):
        D = qkv.shape[-1] // (nq + 2 * nkv)
        q, k, v = qkv.view(B, S, nq + 2 * nkv, D).split((nq, nkv, nkv), dim=2)
        o, lse = native().flash_attn_fwd(q, k, v, D ** -0.5, True, doc_start)
        ctx.save_for_backward(qkv, o, lse)
        ctx.dims, ctx.doc_start = (B, S, nq, nkv, D), doc_start
        return o

    @staticmethod
    def backward(ctx, do):
        qkv, o, lse = ctx.saved_tensors
        B, S, nq, nkv, D = ctx.dims
        q, k, v = qkv.view(B, S, nq + 2 * nkv, D).split((nq, nkv, nkv), dim=2)
        dqkv = native().flash_attn_bwd_qkv(do.contiguous(), q, k, v, o, lse, D ** -0.5, True, ctx.doc_start, None, None, None, S)
        return dqkv, None, None, None, None, None


def qkv_flash_attention(qkv, nq: int, nkv: int, B: int, S: int, doc_start=None):
    """Causal attention on the QKV projection output ``[B*S, (nq+2nkv)*D]`` of a model without rotary positions -> o
    ``[B,S,nq,D]``.  On the HIP path nothing is copied: attention reads views of qkv, and its backward returns d(qkv) (with
    q, k and v sliced apart, a gpt2-125m layer of 8192 tokens spent 64 us on three copies, and 90 on the slices' backward:
    three copies, three fills and two adds)."""
    D = qkv.shape[-1] // (nq + 2 * nkv)
    if use_native(qkv) and qkv.is_contiguous() and qkv.data_ptr() % 16 == 0:
        return _QKVFlashAttn.apply(qkv, nq, nkv, B, S, doc_start)
    x = qkv.view(B, S, nq + 2 * nkv, D)
    q, k, v = (t.contiguous() for t in x.split((nq, nkv, nkv), dim=2))
    return flash_attention(q, k, v, causal=True, doc_start=doc_start)


# =============================================================================== MLP
class _SwiGLU(torch.autograd.Function):
    @staticmethod
    def forward(ctx, gu):
        ctx.save_for_backward(gu)
        return native().swiglu_fwd(gu) if use_native(gu) else ref.swiglu_fwd(gu)

    @staticmethod
    def backward(ctx, dact):
        (gu,) = ctx.saved_tensors
        dact = dact.contiguous()
        return native().swiglu_bwd(dact, gu) if use_native(dact) else ref.swiglu_bwd(dact, gu)


class _GELU(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        ctx.save_for_backward(x)
        return native().gelu_fwd(x) if use_native(x) else ref.gelu_fwd(x)

    @staticmethod
    def backward(ctx, dy):
        (x,) = ctx.saved_tensors
        dy = dy.contiguous()
        return native().gelu_bwd(dy, x) if use_native(dy) else ref.gelu_bwd(dy, x)


def swiglu(gu):
    """``gu [..., 2F]`` laid out ``[gate | up]`` -> ``silu(gate) * up``."""
    return _SwiGLU.apply(gu)


def gelu(x):
    return _GELU.apply(x)


# =============================================================================== loss
class _CrossEntropy(torch.autograd.Function):
    @staticmethod
    def forward(ctx, logits, labels, ignore_index, denom):
        if use_native(logits):
            loss, lse = native().cross_entropy_fwd(logits, labels, ignore_index)
        else:
            loss, lse = ref.cross_entropy_fwd(logits, labels, ignore_index)
        ctx.save_for_backward(logits, lse, labels)
        ctx.ignore_index, ctx.denom = ignore_index, denom
        if use_native(logits) and type(denom) in (int, float) and denom and not torch.jit.is_tracing() and loss.numel() <= 32768:
            return native().loss_mean(loss, denom)
        return loss.sum() / denom

    @staticmethod
    def backward(ctx, g):
        logits, lse, labels = ctx.saved_tensors
        if (use_native(logits) and type(g) is torch.Tensor and g.dtype is torch.float32 and g.is_cuda and type(ctx.denom) in (int, float)
                and ctx.denom and not torch.is_grad_enabled()):
            return native().cross_entropy_bwd_mean(g, ctx.denom, logits, lse, labels, ctx.ignore_index, True), None, None, None
        dloss = (g / ctx.denom).float().expand(labels.shape).contiguous()
        if use_native(logits):
            # logits are dead after this: write dlogits in place (saves a [T,V] buffer)
            dl = native().cross_entropy_bwd(dloss, logits, lse, labels, ctx.ignore_index, True)
        else:
            dl = ref.cross_entropy_bwd(dloss, logits, lse, labels, ctx.ignore_index)
        return dl, None, None, None


def cross_entropy(logits, labels, ignore_index: int = -100, reduction_denom: Optional[float] = None):
    """Mean token cross-entropy over non-ignored labels; logits ``[T,V]`` bf16/fp32."""
    if reduction_denom is None:
        reduction_denom = float(max(int((labels != ignore_index).sum()), 1)) if not labels.is_cuda else None
    if reduction_denom is None:
        # avoid a host sync on GPU: callers that know the count pass it; default = all tokens
        reduction_denom = float(labels.numel())
    return _CrossEntropy.apply(logits, labels, ignore_index, reduction_denom)


# =============================================================================== optimizer
def adamw_step_(param, master, grad, exp_avg, exp_avg_sq, *, lr: float, beta1: float, beta2: float,
                eps: float, weight_decay: float, step: int, grad_scale: Optional[torch.Tensor] = None):
    """One fused AdamW update over flat buffers (bf16 param, fp32 master/m/v, bf16|fp32 grad).
    ``grad_scale`` is a 1-element fp32 device tensor (e.g. the clip coefficient) so clipping
    needs no host sync."""
    bc1 = 1.0 - beta1 ** step
    bc2 = 1.0 - beta2 ** step
    if use_native(param):
        native().adamw_step_(param, master, grad, exp_avg, exp_avg_sq, lr, beta1, beta2, eps, weight_decay,
                             bc1, bc2, grad_scale)
    else:
        gs = float(grad_scale) if grad_scale is not None else 1.0
        ref.adamw_step_(param, master, grad, exp_avg, exp_avg_sq, lr, beta1, beta2, eps, weight_decay, step, gs)


def embed_rows(ids: torch.Tensor, table: torch.Tensor, pos: Optional[torch.Tensor] = None,
               pos_table: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``table[ids]`` (``+ pos_table[pos]``) of a serving step's tokens (no gradients)."""
    if (use_native(table) and all(t.dtype == torch.bfloat16 and t.is_contiguous() and t.shape[1] % 8 == 0 and t.data_ptr() % 16 == 0
                                  for t in (table, pos_table) if t is not None)
            and ids.dim() == 1 and ids.is_contiguous() and ids.dtype == torch.int64
            and (pos_table is None or (pos.is_contiguous() and pos.dtype in (torch.int32, torch.int64)))):
        return native().embed_rows(ids, table, pos if pos_table is not None else None, pos_table)
    x = torch.nn.functional.embedding(ids, table)
    return x if pos_table is None else x + pos_table[pos]


def clip_scale(nsq: torch.Tensor, skipped: torch.Tensor, divisor: float, max_norm: float):
    """``(norm, scale, skipped)`` of an optimizer step from the summed squares of its gradients, on the device: ``norm = sqrt(nsq) /
    divisor``; ``scale = min(1, max_norm / (norm + 1e-6)) / divisor`` (``1 / divisor`` with ``max_norm`` 0), NaN for a norm that is not
    finite, which leaves everything untouched in ``adamw_step_``; ``skipped`` counts such steps."""
    if use_native(nsq):
        return native().clip_scale(nsq, skipped, divisor, max_norm)
    norm = torch.sqrt(nsq) / divisor
    if max_norm > 0:
        coef = torch.clamp(max_norm / (norm + 1e-6), max=1.0) / divisor
    else:
        coef = torch.ones_like(norm) / divisor
    finite = torch.isfinite(norm)
    coef = torch.where(finite, coef, torch.full_like(coef, float("nan")))
    return norm, coef, skipped + (~finite).to(torch.int32).reshape(skipped.shape)


def col_sum_ok(x, out) -> bool:
    """Whether ``col_sum_`` (csrc/col_sum.hip) takes these rows and this output; the rest is a plain sum."""
    return (use_native(x) and x.dim() == 2 and x.dtype == torch.bfloat16 and x.shape[0] > 0 and x.stride(1) == 1 and x.shape[1] % 8 == 0
            and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0 and out.is_contiguous()
            and out.dtype in (torch.bfloat16, torch.float32))


def col_sum_(x, out, add: bool):
    """``out (+)= x.sum(0)`` for rows ``x [T, N]``: a bias gradient, summed in fp32 into a bf16 or fp32 vector."""
    if col_sum_ok(x, out):
        native().col_sum_(x, out, add)
    elif add:
        out.add_(x.sum(0))
    else:
        out.copy_(x.sum(0))


EMBED_GRAD_TOKENS = 65536  # csrc/embed_grad.hip ranks the tokens by comparing all pairs


def embed_grad_pays(T: int, H: int, V: int) -> bool:
    """Is ``embed_grad_`` faster than the library's dense gradient and what adds it?  Ranking all pairs grows with the square of the tokens, the library's sort
    and passes with the tokens, their rows and the table's (in us, on the right; a small table's rows repeat and stay in cache).  us, library / here, ids drawn
    evenly: 16384 tokens 32000 x 64 79 / 64, 256 x 64 72 / 63; 24576 32000 x 64 92 / 120, x 256 124 / 125, x 4096 980 / 248; 32768 32000 x 512 187 / 208, x 1024
    314 / 221; 50000 50304 x 1024 474 / 531, x 2048 927 / 612; 65536 32000 x 64 106 / 724, x 2048 826 / 865.  Ids as often as in text (1 / rank): 24576 32000 x 64
    144 / 141, 32768 x 512 219 / 239, x 1024 283 / 248, 65536 x 64 253 / 779; all the same 65536 x 64 1725 / 1337."""
    return T <= EMBED_GRAD_TOKENS and 1.65e-7 * T * T <= 25 + 2.2e-3 * T + 2.9e-6 * min(T, 8 * V) * H + 1.4e-6 * V * H


def embed_grad_ok(ids, dy, g) -> bool:
    """Whether ``embed_grad_`` (csrc/embed_grad.hip) takes these ids, rows and gradient."""
    return (use_native(dy) and dy.dim() == 2 and dy.dtype == torch.bfloat16 and dy.stride(1) == 1 and dy.shape[1] % 8 == 0
            and dy.stride(0) % 8 == 0 and dy.data_ptr() % 16 == 0 and 0 < dy.shape[0] <= EMBED_GRAD_TOKENS
            and ids.dim() == 1 and ids.dtype == torch.int64 and ids.is_contiguous() and ids.is_cuda
            and g.is_cuda and g.is_contiguous() and g.data_ptr() % 16 == 0 and g.dtype in (torch.bfloat16, torch.float32))


def embed_grad_(ids, dy, g, add: bool):
    """``g [V, H] (+)=`` the rows of ``dy [T, H]`` summed by their ids, in fp32 and in the same order every time: an embedding's gradient."""
    if not add:
        g.zero_()
    native().embed_grad_(ids, dy, g, add)


def l2norm_sq(t: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Sum of squares of ``t`` accumulated (fp32) into ``out`` (allocated if None)."""
    if out is None:
        out = torch.zeros(1, dtype=torch.float32, device=t.device)
    if use_native(t):
        native().l2norm_sq_(t, out)
    else:
        out += ref.l2norm_sq(t)
    return out


# =============================================================================== serving
def transpose_(src: torch.Tensor, dst: torch.Tensor) -> torch.Tensor:
    """``dst[C, R] = src[R, C]`` (bf16, HIP kernel on GPU)."""
    if use_native(src):
        native().transpose_(src, dst)
    else:
        dst.copy_(src.t())
    return dst


def kv_cache_write(k, v, k_cache, v_cache, slot_mapping):
    if use_native(k):
        native().kv_cache_write(k, v, k_cache, v_cache, slot_mapping)
    else:
        ref.kv_cache_write(k, v, k_cache, v_cache, slot_mapping)


def qkv_split_cache(qkv, nq: int, nkv: int, k_cache, v_cache, slots):
    """``qkv [T, (nq + 2 nkv) D]`` of a model without rotary positions: K and V rows to the paged cache at ``slots`` (-1 =
    skip), q as ``[T, nq, D]``; returns (q, k, v), k and v as views of ``qkv`` where that is possible."""
    T = qkv.shape[0]
    x = qkv.view(T, nq + 2 * nkv, -1)
    q, k, v = x[:, :nq], x[:, nq:nq + nkv], x[:, nq + nkv:]
    if use_native(qkv) and qkv.is_contiguous() and x.shape[2] % 8 == 0:
        return native().qkv_split_cache(qkv, nq, nkv, k_cache, v_cache, slots), k, v
    q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    kv_cache_write(k, v, k_cache, v_cache, slots)
    return q, k, v


def paged_attention_decode(q, k_cache, v_cache, block_tables, context_lens, scale: Optional[float] = None):
    scale = scale if scale is not None else q.shape[-1] ** -0.5
    if use_native(q):
        return native().paged_attention_decode(q, k_cache, v_cache, block_tables, context_lens, scale)
    return ref.paged_attention_decode(q, k_cache, v_cache, block_tables, context_lens, scale)


def attn_merge_(o_acc, lse_acc, o_j, lse_j) -> None:
    """Merge a partial attention output into an fp32 accumulator by log-sum-exp (in place)."""
    if use_native(o_acc):
        native().attn_merge_(o_acc, lse_acc, o_j, lse_j)
    else:
        ref.attn_merge_(o_acc, lse_acc, o_j, lse_j)


def prefill_work_list(cu_q, q_block: int = 128) -> List[int]:
    """(sequence << 16) | q-block items for ``paged_prefill_attention``, heaviest (longest
    causal span: the last q-blocks of long chunks) first."""
    items = []
    for n in range(len(cu_q) - 1):
        qlen = int(cu_q[n + 1]) - int(cu_q[n])
        for b in range((qlen + q_block - 1) // q_block):
            items.append((b * q_block, (n << 16) | b))
    items.sort(key=lambda t: -t[0])
    return [w for _, w in items]


def paged_prefill_attention(q, k_cache, v_cache, block_tables, cu_q, ctx_lens, scale: Optional[float] = None,
                            work=None):
    """Chunked / prefix-reusing prefill attention over the paged KV cache (see
    ``csrc/paged_prefill.hip``).  ``cu_q`` / ``ctx_lens`` / ``block_tables`` int32; ``work``
    (optional) is the precomputed :func:`prefill_work_list` as an int32 tensor."""
    scale = scale if scale is not None else q.shape[-1] ** -0.5
    if use_native(q):
        if work is None:
            work = torch.tensor(prefill_work_list(cu_q.tolist()), dtype=torch.int32, device=q.device)
        return native().paged_prefill_attention(q, k_cache, v_cache, block_tables, cu_q, ctx_lens, work, scale)
    return ref.paged_prefill_attention(q, k_cache, v_cache, block_tables, cu_q, ctx_lens, scale)


SKINNY_CONFIGS: dict = {}  # (M, N, K) -> tuned config (0 = hipBLASLt), from a tuning cache


_ROW_ACTS = {None: 0, "gelu": 2}  # the tanh form, as :func:`gelu`


def wants_grad(*ts) -> bool:
    """Will autograd want a gradient through an op of these operands?  (The kernels of serving have no backward.)"""
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in ts)


def stream_takes(x, w, b=None) -> bool:
    """Does ``csrc/stream_linear.h`` take this product?  At most 32 rows, bf16, K a multiple of 8, aligned rows, no gradient.  (Asked for every
    projection of an eager step: one look at each property.)"""
    if not (x.is_cuda and x.dtype is torch.bfloat16 and w.dtype is torch.bfloat16):
        return False
    xs, ws, (M, K) = x.stride(), w.stride(), x.shape
    return (1 <= M <= 32 and xs[1] == 1 and ws[1] == 1 and (xs[0] | ws[0] | K) & 7 == 0 and (x.data_ptr() | w.data_ptr()) & 15 == 0
            and (b is None or (b.dtype is torch.bfloat16 and b.is_contiguous())) and use_native(x) and not wants_grad(x, w, b))


def stream_ok(x, w, b=None) -> bool:
    """``stream_takes``, and it is faster than the library's product (:func:`stream_pays`)."""
    return x.dim() == 2 and 1 <= x.shape[0] <= 32 and stream_pays(x.shape[0], w.shape[0], x.shape[1]) and stream_takes(x, w, b)


@functools.lru_cache(maxsize=4096)
def stream_pays(M: int, N: int, K: int) -> bool:
    """Is the weight stream faster than the library's product?  In a graph, weights from HBM, us, library / here, beside each line.  (The
    library splits K over the chip at some sizes and not at others: 16 rows 4096 x 8192 15.0, 4096 x 11008 37.)"""
    if M > 16:  # a fragment of x more for every one of W: 32 rows 4240 x 2048 12.2 / 9.7, 12288 x 1024 12.4 / 9.4, 16384 x 512 8.8 / 7.2, but 12288 x 256 5.3 / 5.8,
        # 28672 x 768 13.9 / 15.7, 6144 x 3072 13.1 / 14.2, 50304 x 768 20.7 / 25.2, 102400 x 256 17.6 / 18.4; 24 rows 4096 x 4096 13.6 / 13.1, 12288 x 2048 15.8 / 15.0
        if N > 40960:  # where the last of the library's rounds of 256-wide tiles leaves CUs idle: 32 rows 152064 x 3072 295 / 202, 128256 x 2304 110 / 131
            return N >= 102400 and (512 if M > 24 else 0) <= K <= 4096 and 0 < -(-N // 256) % 256 <= 192
        if N > 8192:
            return 512 <= K <= (2048 if N <= 12288 and M <= 24 else 1024) and (N <= 24576 or 31744 <= N <= 32000)
        return K <= 2048 or (M <= 24 and N <= 4096 and K <= 4096)
    if K > 4096 and K % 8192 == 0:  # rows of W that lie a multiple of 8192 entries apart crowd the same channels: 8 rows 2048 x 8192 13.0 / 12.4, 6144 x 8192
        # 23.7 / 25.6, 16384 x 16384 101 / 129; 4 rows 12288 x 8192 48 / 51, 16384 x 8192 63 / 55, 32000 x 8192 111 / 94; 16 rows 2048 x 8192 13.6 / 15.4
        return (M <= 8 and N <= (4096 if K == 8192 else 2304)) or (M <= 5 and K == 8192 and 16384 <= N <= 40960)
    if K > 4096 and M > 8:  # a workgroup reads all of x for its few rows of W: 16 rows 3648 x 6144 13.2 / 14.8, 1024 x 5120 7.5 / 9.3, 6144 x 7168 19.8 / 22.5, 12288 x 10240
        # 58 / 51, 32000 x 6144 86 / 77, 50304 x 12288 220 / 237; 14 rows 1024 x 5120 12.5 / 8.2; 12 rows 6144 x 7168 19.8 / 21.2
        if 24576 < N <= 30720 and 10240 < K < 12288:
            return False
        return (8192 if M > 12 and K <= 10240 else 4096) < N <= 40960 or (N <= 2304 and K < 6144 and (M <= 14 or N > 1024))
    if K > 4096:  # 8 rows 2048 x 6144 11.2 / 10.1, 4096 x 12288 23.0 / 24.5, 3072 x 14336 20.2 / 23.8, 12288 x 12288 61 / 57, 50304 x 5120 94 / 102; 4 rows 50304 x 11008 195 / 234, 24576 x
        # 20480 176 / 201
        if 40960 < N < 61440 or (M <= 4 and 24576 < N <= 30720 and 10240 <= K <= 12288) or (K > 16384 and N >= 18432):
            return False
        return M <= 4 or not (K % 2048 == 0 and 12288 <= K < 16384 and 2304 < N <= (4096 if K == 12288 else 3840))
    # 16 rows 2048 x 2048 11.1 / 6.1, 8256 x 2048 14.2 / 11.0, 32000 x 2048 35 / 30, 50304 x 768 20.0 / 21.8, 50304 x 3072 62 / 68, 102400 x 2048 147 / 86, 65024 x 3072
    # 76 / 81, 152064 x 3072 295 / 183; 4 rows 50304 x 768 19.7 / 19.3
    return M <= 4 or N <= 40960 or N >= 61440


@functools.lru_cache(maxsize=4096)
def decode_form(M: int, N: int, K: int) -> str:
    """The form of :func:`decode_linear` by size: ``stream``, ``skinny`` (``csrc/skinny_gemm.hip``) or ``library``.  Beside
    :func:`stream_pays`, us in a graph, stream / skinny:"""
    # short rows: 1 row 2304 x 768 3.63 / 3.32, 8192 x 768 5.66 / 5.30; 16 rows 768 x 512 3.48 / 3.07, 512 x 768 3.8 / 3.4, but 2304 x 768 4.10 / 4.06 and 768 x 768 3.88 / 3.97; 24
    # rows 4096 x 768 4.87 / 4.57.  (More than 4096 outputs that are a multiple of 64 take skinny's other tiles: 16 rows 5120 x 512 4.6 / 6.8, but 5152 x 512 4.5 / 4.1.)
    if K < (768 if 4 < M <= 16 and 512 < N < 3072 else 1024) and N <= (16384 if M <= 4 else 5152 if M <= 16 and N % 64 else 4096):
        return "skinny"
    if M <= 4 and 2304 <= N <= 4096 and K <= 1280:  # 4 rows 3072 x 1280 4.9 / 4.7, 3648 x 1280 5.1 / 4.7
        return "skinny"
    if 4 < M <= 16 and N % 64 and 8192 < N <= 10240 and K < (1024 if M <= 8 else 512):  # 8 rows 9248 x 256 4.4 / 3.6, x 896 7.3 / 6.8; 16 rows x 384 5.5 / 4.5
        return "skinny"
    # few long rows, of which skinny splits K over the chip: 8 rows 1024 x 12288 15.0 / 13.3, 1280 x 11008 14.8 / 13.4, 16 rows 768 x 10240 15.5 / 13.6, 1536 x 10240 17.5 / 14.9,
    # 12 rows 2048 x 28672 42.6 / 37.1, 16 rows 2048 x 14336 24.7 / 21.5
    if 4 < M <= 16 and K > (8192 if N <= (1024 if M < 8 else 1280 if M < 12 else 1536) else 12288) and N <= (2048 if M >= 8 else 1024):
        return "skinny"
    # (the library's own times jump here: 12 rows 2048 x 11008 35.8, stream 18.2; 2048 x 10240 13.1 and 13.1)
    return "stream" if stream_pays(M, N, K) or (M <= 16 and N <= 4096 and K % 8192) else "library"


def decode_linear(x, w, b=None, act: Optional[str] = None):
    """``act(x @ w^T (+ b))`` for decode-shaped inputs (``act``: None or ``gelu``): the form that is fastest on uncached weights
    (``decode_form``): a stream of the weight with bias and activation in the same launch (``csrc/stream_linear.h``),
    ``csrc/skinny_gemm.hip``, or the library.  A tuned configuration or knob ``skinny_gemm`` = ``all`` picks
    ``csrc/skinny_gemm.hip``, ``off`` the library.  Other inputs: the library and an activation pass."""
    from llmctl.exec.linear import forward_linear, rows_linear, small_linear

    mode = knobs().skinny_gemm
    (M, K), N = x.shape if x.dim() == 2 else (0, 0), w.shape[0]
    y = None
    tuned = SKINNY_CONFIGS.get((M, N, w.shape[1])) if SKINNY_CONFIGS and x.dim() == 2 else None
    if tuned is not None and mode == "auto" and use_native(x):
        if tuned == 0:
            y = torch.nn.functional.linear(x, w, b)
        elif x.is_contiguous() and w.is_contiguous() and x.dtype == w.dtype == torch.bfloat16:
            y = native().skinny_linear_cfg(x, w, b, tuned)
    form = "skinny" if mode == "all" else "library" if mode == "off" or not 1 <= M <= 32 else decode_form(M, N, K)
    if y is None and form == "skinny":
        if (use_native(x) and M <= 32 and x.dtype == w.dtype == torch.bfloat16 and N % 16 == 0 and K % 128 == 0
                and x.is_contiguous() and w.is_contiguous() and (b is None or b.is_contiguous())
                and not (mode == "auto" and act is not None)):  # (an activation pass of its own costs more than the kernels differ by)
            y = native().skinny_linear(x, w, b)
        elif mode == "auto":
            form = "stream"
    if form == "library" and mode == "auto" and act is not None and M * N % 8:
        form = "stream"  # (the activation pass takes multiples of 8)
    if y is None and form == "stream" and x.dim() == 2 and stream_takes(x, w, b):
        return native().stream_linear(x, w, b, _ROW_ACTS[act])
    if y is None and act == "gelu" and M > 32:
        y = small_linear(x, w, b, "eager", _ROW_ACTS[act])
        if y is None:
            y = rows_linear(x, w, b, None, _ROW_ACTS[act])
        if y is not None:
            return y
    if y is None:
        y = forward_linear(x, w, b)
    return gelu(y) if act == "gelu" else y


def norm_linear_ok(x, res, nw, nb, w, b, split: bool = False) -> bool:
    """Does ``csrc/norm_linear.hip`` take this LayerNorm and product, and does it pay?  Every workgroup repeats the norm, so for few and
    short rows and up to 8192 outputs: up to 12 rows of 1024 (8 of 2048); ``split``: four more, as the launch that splits QKV goes too.
    us in a graph, fused / separate: K 768, N 3072: 1 row 4.8 / 6.7, 8 rows 6.3 / 7.2, 12 rows 7.3 / 7.4, 16 rows 8.3 / 7.6; K 2048, N 3072:
    1 row 8.0 / 9.8, 8 rows 10.0 / 10.8, 12 rows 11.8 / 11.0; N 16384, K 768: 1 row 11.8 / 10.8."""
    if nb is None or not (x.dim() == 2 and stream_ok(x, w, b)) or wants_grad(res, nw, nb):
        return False
    (M, K), N = x.shape, w.shape[0]
    bf = all(t.dtype == torch.bfloat16 and t.is_contiguous() and t.data_ptr() % 16 == 0 for t in (x, nw, nb) + (() if res is None else (res,)))
    return (bf and K <= 2048 and M <= (12 if K <= 1024 else 8) + 4 * split and N <= 8192 and N % 4 == 0 and knobs().skinny_gemm == "auto"
            and (M, N, K) not in SKINNY_CONFIGS)


def decode_norm_linear(x, res, nw, nb, eps: float, w, b=None, act: Optional[str] = None):
    """``act(LN(x + res) w^T (+ b))`` of a decode step (``res`` None: nothing is added); returns it and the new residual ``x +
    res``.  Few short rows take one launch."""
    if norm_linear_ok(x, res, nw, nb, w, b):
        y, r = native().norm_linear(x, res, nw, nb, eps, w, b, _ROW_ACTS[act])
        return y, (x if res is None else r)
    xn, r = (layernorm(x, nw, nb, eps), x) if res is None else add_layernorm(x, res, nw, nb, eps)
    return decode_linear(xn, w, b, act=act), r


def decode_norm_qkv_cache(x, res, nw, nb, eps: float, w, b, nq: int, nkv: int, k_cache, v_cache, slots):
    """``decode_norm_linear`` for the QKV projection of a model without rotary positions, K and V rows written to the paged cache at
    ``slots``; returns (q ``[T, nq, D]``, the new residual)."""
    if norm_linear_ok(x, res, nw, nb, w, b, True) and w.shape[0] // (nq + 2 * nkv) % 8 == 0:
        q, r = native().norm_qkv_cache(x, res, nw, nb, eps, w, b, nq, nkv, k_cache, v_cache, slots)
        return q, (x if res is None else r)
    xn, r = (layernorm(x, nw, nb, eps), x) if res is None else add_layernorm(x, res, nw, nb, eps)
    return qkv_split_cache(decode_linear(xn, w, b), nq, nkv, k_cache, v_cache, slots)[0], r


def decode_layers_ok(hidden: int, heads: int, kv_heads: int, ffn: int, layers: int, rows: int, cache) -> bool:
    """Does ``csrc/decode_layers.hip`` run a whole decode step of this size in one launch (LayerNorm, biases, GELU and learned positions are the caller's to
    know), and does it pay?  Up to four rows, where the launches are most of a step: gpt2-125m, us a step, a launch per product / this: one row at context 129
    381 / 203, 2000 432 / 252, at 129 two rows 396 / 239, four 420 / 297; four layers of 256, one row 127 / 78, of 1024, four rows 171 / 153."""
    return (knobs().decode_layers and use_native(cache) and cache.dtype == torch.bfloat16 and cache.is_contiguous() and 1 <= rows <= 4 and 1 <= layers <= 32
            and cache.dim() == 5 and cache.shape[-1] == 64 and cache.data_ptr() % 16 == 0 and cache[0].numel() < 1 << 35
            and hidden % 256 == 0 and 256 <= hidden <= 1024 and heads == kv_heads and heads * 64 == hidden and ffn == 4 * hidden
            and torch.cuda.get_device_properties(cache.device).multi_processor_count >= 128)


def decode_layers_workspace(hidden: int, device) -> torch.Tensor:
    """The words that the workgroups of a step exchange (``decode_layers``), for steps that follow one another: a graph's, or one eager step's."""
    return torch.zeros(native().decode_layers_words(hidden), dtype=torch.int64, device=device)


def decode_layers(ids, positions, slots, block_tables, ctx_lens, table, pos_table, weights, k_cache, v_cache, eps: float, workspace, workgroups: int = 128,
                  gate_us: Optional[int] = None, lost: Optional[torch.Tensor] = None, spins: int = 1 << 21):
    """The final norm's rows of a decode step: embedding, all layers with their paged cache, final norm.  ``weights``: per layer the attention norm (weight,
    bias), QKV, output projection, MLP norm, up and down (weight and bias each), then the final norm; ``k_cache`` / ``v_cache``: all layers' ``[L, blocks,
    block, heads, 64]``.  ``workgroups``: fewer than 128 each do the work of several; ``gate_us``: how long it waits for those that do not run yet, for every round of
    shares that the others would take beyond the first (None: about as long as that round, 5 us a layer and 2.5 a further row).  ``lost``: an int32 of pinned host memory
    that becomes 1 when a workgroup's wait for the others runs out (``spins`` tries, seconds); the rows are NaN then and the cache rows void."""
    if gate_us is None:
        gate_us = 5 * (len(weights) // 12) * (ids.shape[0] + 1) // 2
    return native().decode_layers(ids, positions, slots, block_tables, ctx_lens, table, pos_table, weights, k_cache, v_cache, eps, workspace, workgroups, gate_us,
                                  lost, spins)


def _dequant(w, w_scale, dtype):
    """bf16 image of an fp8 (e4m3fn) weight with fp32 row scales (fallback paths)."""
    return w if w_scale is None else (w.float() * w_scale.float().unsqueeze(1)).to(dtype)


def decode_linear_fp8(x, w, w_scale, b=None):
    """``x @ (w * w_scale[:, None])^T (+ b)`` for decode-shaped inputs with fp8 (OCP e4m3fn)
    weights and fp32 row scales (W8A16: ``csrc/skinny_gemm.hip``'s fp8 weight stream, half the
    bytes of the bf16 one)."""
    if decode_fused_ok(x, w):
        return native().decode_linear_fp8(x, w, w_scale, b)
    return decode_linear(x, _dequant(w, w_scale, x.dtype), b)


def decode_fused_ok(x, w) -> bool:
    """Can this decode projection run with a fused epilogue (``csrc/skinny_gemm.hip``: the v2
    weight-streaming GEMM's K-chunk partials summed by a finalize pass that also applies RoPE +
    paged-cache write, SwiGLU or residual + RMSNorm)?  <= 16 tokens, bf16, out features a
    multiple of 64, in features of 128.  Knob ``decode_fused`` off disables (A/B)."""
    return (knobs().decode_fused and use_native(x) and x.dim() == 2
            and 1 <= x.shape[0] <= 16 and x.dtype == torch.bfloat16
            and w.dtype in (torch.bfloat16, torch.float8_e4m3fn) and x.is_contiguous()
            and w.is_contiguous() and w.shape[0] % 64 == 0 and x.shape[1] % 128 == 0)


def decode_qkv_rope_cache(x, w, b, cos, sin, nq: int, nkv: int, positions, k_cache, v_cache, slots,
                          w_scale=None):
    """Decode QKV projection + RoPE + paged-cache write of K/V in one finalize pass; returns
    ``q [T, nq, D]``.  Same result as ``rope_qkv_cache(decode_linear(x, w, b), ...)[0]``.
    ``w_scale``: fp32 row scales of an fp8 (e4m3fn) ``w``."""
    if decode_fused_ok(x, w):
        return native().decode_qkv_rope_cache(x, w, b, cos, sin, nq, nkv, positions.to(torch.int32).contiguous(),
                                              k_cache, v_cache, slots, w_scale)
    return rope_qkv_cache(decode_linear(x, _dequant(w, w_scale, x.dtype), b), cos, sin, nq, nkv, 0, positions,
                          k_cache, v_cache, slots)[0]


def decode_attention_qkv(x, w, b, cos, sin, nq: int, nkv: int, positions, k_cache, v_cache, slots, block_tables,
                         ctx_lens, scale: Optional[float] = None, w_scale=None):
    """Decode QKV projection -> RoPE -> paged-cache write (one finalize pass) -> paged attention.
    (Round 2's variant that summed the projection partials inside the attention kernel measured
    0.1-0.2 ms slower per 16 x 2k GPT-7B step, profiles/serve_r2_session6.txt, and was retired.)"""
    D = w.shape[0] // (nq + 2 * nkv)
    scale = scale if scale is not None else D ** -0.5
    q = decode_qkv_rope_cache(x, w, b, cos, sin, nq, nkv, positions, k_cache, v_cache, slots, w_scale)
    return paged_attention_decode(q, k_cache, v_cache, block_tables, ctx_lens, scale)


def _gemm64_fwd_takes(x, w, b=None) -> bool:
    """The operands of ``gemm64_fwd`` (csrc/gemm64.hip), which takes any number of rows."""
    return (x.dim() == 2 and x.dtype is torch.bfloat16 and w.dtype is torch.bfloat16 and x.shape[1] % 128 == 0 and x.shape[1] >= 256 and x.stride(1) == 1
            and w.stride(1) == 1 and x.stride(0) % 8 == 0 and w.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
            and x.stride(0) >= x.shape[1] and w.stride(0) >= w.shape[1] and 512 * max(x.stride(0), w.stride(0)) < 2**31
            and (b is None or (b.dtype is torch.bfloat16 and b.is_contiguous() and b.data_ptr() % 8 == 0)) and use_native(x) and not wants_grad(x, w, b))


def odd_linear(x, w, b=None):
    """``x @ w^T (+ b)`` for layers whose outputs fill no whole tiles of 256: the in-house kernel where the library's products lose to it (:func:`odd_pays`), else the
    library's."""
    if odd_pays(x.shape[0], w.shape[0], x.shape[1]) and _gemm64_fwd_takes(x, w, b):
        return native().gemm64_fwd(x, w, b)
    return torch.nn.functional.linear(x, w, b)


@functools.lru_cache(maxsize=4096)
def odd_pays(T: int, N: int, K: int) -> bool:
    """Rule of :func:`odd_linear`: from 9 * 2^20 outputs on, unless the tiles of 256 x 256 leave the second round of 256, or with a long K the only one, short.  us, library / here: K 2048
    3379 x 4240 64.5 / 49.2, 3379 x 9248 132 / 114, 4090 x 12008 201 / 145, 2911 x 8256 93 / 87; K 1024 2911 x 4240 42 / 28; below: 1331 x 4240 29 / 39, 1800 x 5152 44 / 42; 1.2
    to 1.5 rounds: K 1024 6000 x 3208 50.8 / 55.5, K 3072 1800 x 10504 105 / 114, K 2048 1800 x 12008 86 / 92, 3379 x 6200 83 / 88; less than one: K 4096 1000 x 10504 78 / 85, 1331 x 8256 79 / 87.  (Outputs in
    whole tiles: 3379 x 6144 73 / 86, 3379 x 8192 88 / 95.)"""
    tiles = -(-T // 256) * -(-N // 256)
    return N % 256 != 0 and N % 8 == 0 and K >= 1024 and T * N >= 9 << 20 and not 307 < tiles < 384 and not (tiles < 200 and K >= 4096)


@functools.lru_cache(maxsize=4096)
def ragged_swiglu_pays(T: int, F: int) -> bool:
    """Does the gated kernel take a projection to 2 F outputs of a number of tokens that is no multiple of 256?  From 11 * 2^20 entries on, unless a third of its tile rows is
    empty or its tiles of 256 x 128 pairs make about one and a half rounds of 256.  us, library and SwiGLU pass / here: 4096 -> 2 x 11008 500 tokens 93 / 85, 700 144 /
    118, 1331 308 / 210, 2911 503 / 394, 4095 680 / 528; 4096 -> 2 x 8192 700 86 / 84, 2911 296 / 288, but 1331 160 / 181, 1500 168 / 177; 2048 -> 2 x 4096 1500 50 / 46, but 1023 40 /
    43; 8192 -> 2 x 28672 300 312 / 347."""
    rows = -(-T // 256)
    return F % 128 == 0 and 2 * T * F >= 11 << 20 and 3 * T >= 2 * 256 * rows and not 346 <= rows * (F // 128) <= 410


def up_swiglu(x, w, b=None):
    """``silu(gate) * up`` of the gate/up projection ``x @ w^T (+ b)`` (w = [W_gate; W_up]).
    Serving prefill: tokens a multiple of 256 run the gemm64 kernel with the SwiGLU in its
    epilogue (``gemm64_swiglu_fwd``: gate and matching up rows in one output tile, only the
    [T, F] activation stored — no gu tensor, no SwiGLU pass), and so do other numbers of tokens where that pays (:func:`ragged_swiglu_pays`).  Knob ``prefill_swiglu``
    off disables (A/B)."""
    x2 = x.reshape(-1, x.shape[-1])
    T, F = x2.shape[0], w.shape[0] // 2
    if (b is None and knobs().prefill_swiglu and use_native(x) and T % 256 == 0
            and F % 128 == 0 and x2.shape[1] % 128 == 0 and x2.dtype == w.dtype == torch.bfloat16
            and x2.stride(1) == 1 and x2.stride(0) % 8 == 0 and x2.data_ptr() % 16 == 0 and w.is_contiguous()
            and w.data_ptr() % 16 == 0):
        from llmctl.exec.linear import gemm64_config

        act = native().gemm64_swiglu_fwd(x2, w, gemm64_config("fwd", T, 2 * F, x2.shape[1]) % 1000)
        return act.view(*x.shape[:-1], F)
    if b is None and knobs().prefill_swiglu and w.shape[0] % 2 == 0 and ragged_swiglu_pays(T, F) and _gemm64_fwd_takes(x2, w):
        return native().gemm64_fwd(x2, w, None, True).view(*x.shape[:-1], F)
    from llmctl.exec.linear import forward_linear

    return swiglu(forward_linear(x, w, b))


def decode_up_swiglu(x, w, b=None, w_scale=None):
    """Decode gate/up projection with SwiGLU in its finalize pass: ``silu(g) * u`` of
    ``x @ w^T (+ b)`` (gate = first half of the out features)."""
    if decode_fused_ok(x, w):
        return native().decode_up_swiglu(x, w, b, w_scale)
    return swiglu(decode_linear(x, _dequant(w, w_scale, x.dtype), b))


# ----------------------------------------------------------- prefill with the RMSNorm folded in
# Serving prefill (llmctl/serve/engine.py ``_prefill_layers_folded``): rmsnorm(h) * w_n @ W^T equals
# rstd(h)[:, None] * (h @ (W * w_n)^T), so with the norm weight folded into the projection's K
# columns (once, at engine start) the norm reduces to a per-row statistic that the GEMM applies in its
# epilogue, and no normalised copy of h is written or read.

def rms_rstd(x, eps: float):
    """``rsqrt(mean(x^2, -1) + eps)`` per row of a 2-D bf16 ``x`` (fp32 [T])."""
    if use_native(x):
        return native().rms_rstd(x.contiguous(), eps)
    return torch.rsqrt(x.float().pow(2).mean(-1) + eps)


def rowscale_ok(x, w) -> bool:
    """Shapes the row-scaled gemm64 forms take: x [T, K], w [N, K], T and N multiples of 256, K of
    128 and >= 256, bf16 GPU operands, 16-byte aligned rows."""
    return (use_native(x) and x.dim() == 2 and w.dim() == 2 and x.dtype == w.dtype == torch.bfloat16
            and x.shape[0] % 256 == 0 and x.shape[0] > 0 and w.shape[0] % 256 == 0 and x.shape[1] == w.shape[1]
            and x.shape[1] % 128 == 0 and x.shape[1] >= 256 and x.stride(1) == 1 and x.stride(0) % 8 == 0
            and x.data_ptr() % 16 == 0 and w.is_contiguous() and w.data_ptr() % 16 == 0)


def linear_rowscale(x, w, rstd):
    """``(x @ w^T) * rstd[:, None]`` rounded once to bf16 (gemm64 persistent kernel, row scale in
    its epilogue)."""
    if rowscale_ok(x, w):
        from llmctl.exec.linear import gemm64_config

        return native().gemm64_rs(x, w, rstd, gemm64_config("fwd", x.shape[0], w.shape[0], x.shape[1]))
    return ((x.float() @ w.float().t()) * rstd.float()[:, None]).to(x.dtype)


def up_swiglu_rowscale(x, w, rstd):
    """``silu(g) * u`` of ``(x @ w^T) * rstd[:, None]`` (w = [W_gate; W_up]): the SwiGLU and the row
    scale in the gate/up GEMM's epilogue."""
    F = w.shape[0] // 2
    if rowscale_ok(x, w) and F % 128 == 0:
        from llmctl.exec.linear import gemm64_config

        return native().gemm64_swiglu_fwd(x, w, gemm64_config("fwd", x.shape[0], w.shape[0], x.shape[1]) % 1000, rstd)
    gu = ((x.float() @ w.float().t()) * rstd.float()[:, None]).to(x.dtype)
    return swiglu(gu)


def linear_acc_(x, w, out):
    """``out += x @ w^T`` in place (the residual add riding on the projection's epilogue)."""
    if rowscale_ok(x, w) and out.is_contiguous() and out.shape == (x.shape[0], w.shape[0]):
        from llmctl.exec.linear import gemm64_config

        native().gemm64_ex(x, w, out, False, False, True, gemm64_config("fwd", x.shape[0], w.shape[0], x.shape[1]))
        return out
    return out.addmm_(x, w.t())


def decode_linear_add_rmsnorm(x, w, b, residual, norm_w, eps: float, w_scale=None):
    """Decode row projection + residual add + RMSNorm in one finalize pass:
    ``(rmsnorm(y + residual) * norm_w, y + residual)`` with ``y = x @ w^T (+ b)``."""
    if decode_fused_ok(x, w) and w.shape[0] <= 16384:
        return native().decode_linear_add_rmsnorm(x, w, b, residual, norm_w, eps, w_scale)
    y = decode_linear(x, _dequant(w, w_scale, x.dtype), b)
    return add_rmsnorm(y, residual, norm_w, eps)


def sample(logits, temperature, top_k, top_p, uniform):
    if use_native(logits):
        return native().sample(logits, temperature, top_k, top_p, uniform)
    return ref.sample(logits, temperature, top_k, top_p, uniform)


__all__ = [
    "transpose_",
    "rmsnorm", "add_rmsnorm", "layernorm", "add_layernorm", "rope_qkv", "flash_attention", "rope_flash_attention",
    "swiglu",
    "gelu", "cross_entropy", "adamw_step_", "clip_scale", "embed_rows", "l2norm_sq", "kv_cache_write", "qkv_split_cache", "paged_attention_decode",
    "sample", "decode_linear", "decode_linear_fp8", "decode_fused_ok", "decode_qkv_rope_cache", "decode_up_swiglu", "decode_attention_qkv", "up_swiglu",
    "decode_linear_add_rmsnorm", "rope_qkv_cache", "paged_prefill_attention", "prefill_work_list", "attn_merge_",
    "rms_rstd", "rowscale_ok", "decode_layers_ok", "decode_layers", "decode_layers_workspace", "linear_rowscale", "up_swiglu_rowscale", "linear_acc_",
]

"""TrainingEngine: one process per GPU, plan-driven TP × PP × DP (+SP, ZeRO-1/2/3).

Reference: ``llmctl/runtime/engine.py:72-411`` (HF model + accelerate DDP).  Kept
compatible: ``TrainingConfig`` carries every reference field (``engine.py:30-70``) and the
checkpoint directory layout (``checkpoint-<step>/``, ``final/``, ``training_state.json``) is
preserved and extended (``llmctl.io.checkpoint``).  Fixed reference defects:
loss scaled once under accumulation, DP sync only on the final micro-step, seeds applied,
bf16 weights when bf16 is requested, checkpoints written on CPU runs too, full resume.
"""

from __future__ import annotations

import json
import logging
import math
import os
import time
from dataclasses import asdict, dataclass, field
from pathlib import Path
from typing import Any, Dict, Iterator, List, Optional, Tuple

import torch
import torch.distributed as dist

from llmctl.comms.overlap import GradSyncEngine
from llmctl.models import ModelConfig, ParallelContext, build_model, get_model_config
from llmctl.parallel.groups import ProcessGroups, build_process_groups
from llmctl.runtime.faults import FaultInjector
from llmctl.runtime.flat import FlatParameters
from llmctl.runtime.optimizer import FlatAdamW, LRSchedule
from llmctl.runtime.step_graph import StepGraphs
from llmctl.utils.env import dist_env
from llmctl.utils.seed import set_seed

log = logging.getLogger("llmctl.engine")


@dataclass
class TrainingConfig:
    # ---- reference fields (engine.py:30-70; defaults kept) -------------------------
    model_name_or_path: str = "gpt2"
    dataset_path: str = "synthetic"
    output_dir: str = "./outputs"
    learning_rate: float = 5e-5
    batch_size: int = 8  # micro-batch per DP rank
    gradient_accumulation_steps: int = 1
    num_epochs: int = 3
    max_steps: int = -1
    warmup_steps: int = 0
    weight_decay: float = 0.01
    optimizer: str = "adamw"
    scheduler: str = "linear"
    gradient_clipping: float = 1.0
    mixed_precision: str = "bf16"
    distributed_backend: str = "auto"  # auto => nccl(RCCL) on GPU, gloo on CPU
    deepspeed_config: Optional[str] = None  # accepted for CLI compatibility; ZeRO is native
    save_steps: int = 500
    eval_steps: int = 500
    save_total_limit: int = 3
    resume_from_checkpoint: Optional[str] = None
    logging_steps: int = 10
    log_level: str = "info"
    seed: int = 42
    deterministic: bool = False
    # ---- plan / MI355X additions ---------------------------------------------------
    seq_len: int = 2048
    tensor_parallel: int = 1
    pipeline_parallel: int = 1
    context_parallel: int = 1  # CP: sequence split over cp ranks (llmctl.parallel.context_parallel)
    context_parallel_mode: str = "ulysses"  # ulysses (all-to-all, xGMI-mesh friendly) | ring
    expert_parallel: int = 1  # MoE: experts sharded over groups of this many DP ranks (llmctl.models.moe)
    pack_sequences: bool = False  # documents packed into sequences: attention/positions reset at separators
    doc_separator: int = 0  # token that ends a document (byte tokenizer / tokenize_to_bin use 0)
    sequence_parallel: bool = False
    zero_stage: int = 0
    activation_checkpoint: str = "none"  # none | selective | full
    num_microbatches: int = 0  # pipeline micro-batches per step (0 => 2*pp)
    virtual_stages: int = 1  # interleaved pipeline: model chunks per pipeline rank (1 = plain 1F1B)
    tuning_cache: Optional[str] = None  # autotuner results to apply (else $LLMCTL_TUNING_CACHE)
    bucket_mb: float = 256.0
    # gradient accumulation / reduction dtype: "fp32" keeps fp32 main gradients (GEMM epilogues
    # accumulate in fp32, DP reductions in fp32; ~2x gradient memory and bucket bytes), "bf16"
    # the parameter dtype; "auto" = fp32 whenever micro-batches accumulate (grad accumulation or
    # pipeline micro-batches) with bf16 parameters, where repeated bf16 rounding of the running
    # sum loses low-order gradient bits (Megatron's default for bf16)
    main_grads: str = "auto"
    betas: Tuple[float, float] = (0.9, 0.95)
    eps: float = 1e-8
    device: str = "auto"
    samples_per_epoch: int = 0  # synthetic dataset size (0 => unbounded / max_steps driven)
    eval_batches: int = 2
    async_checkpoint: bool = True
    sharded_checkpoint: bool = True
    keep_latest: int = 0
    profile_dir: Optional[str] = None  # torch.profiler (ROCm/roctracer activities) Chrome traces per rank
    profile_schedule: str = "wait=1,warmup=1,active=2"  # or "step(N)" (telemetry.profiling.schedule)
    collective_timeout_s: float = 1800.0  # RCCL/gloo watchdog: a dead peer fails the job instead of hanging it
    plan_file: Optional[str] = None
    # performance knobs (llmctl.config.knobs.PerfKnobs field -> value): kernel / schedule choices,
    # resolved at engine init (+ LLMCTL_KNOBS overrides) and recorded in the run manifest
    perf_knobs: Dict[str, Any] = field(default_factory=dict)
    extra: Dict[str, Any] = field(default_factory=dict)

    @property
    def dtype(self) -> torch.dtype:
        return {"bf16": torch.bfloat16, "fp16": torch.float16, "no": torch.float32, "fp32": torch.float32}[
            self.mixed_precision]


def create_training_config(**kw) -> TrainingConfig:
    known = set(TrainingConfig.__dataclass_fields__)
    extra = {k: v for k, v in kw.items() if k not in known}
    cfg = TrainingConfig(**{k: v for k, v in kw.items() if k in known})
    cfg.extra.update(extra)
    return cfg


class TrainingEngine:
    def __init__(self, config: TrainingConfig, model_config: Optional[ModelConfig] = None):
        self.config = c = config
        logging.basicConfig(level=getattr(logging, c.log_level.upper(), logging.INFO),
                            format="%(asctime)s %(levelname)s %(name)s: %(message)s")
        from llmctl.config import knobs as perf

        self.knobs = perf.configure(c.perf_knobs)  # tuning-cache values below may refine it
        self.env = dist_env()
        self._setup_distributed()
        set_seed(c.seed, c.deterministic)
        self.model_config = model_config or get_model_config(c.model_name_or_path)
        from llmctl.plugins import tuning_cache

        tc = tuning_cache.resolve(c.tuning_cache)
        self.tuned = tuning_cache.apply_training(tc, c) if tc is not None else {}
        if self.tuned:
            log.info("tuning cache %s applied: %s", tc, self.tuned)
        self.knobs = perf.knobs()  # config + tuning cache + LLMCTL_KNOBS
        self.global_step = 0
        self.epoch = 0
        self.consumed_samples = 0
        self.metrics_hooks: List = []
        self.step_graphs = StepGraphs()
        self._build()
        self.faults = FaultInjector(self.rank, c.output_dir)

    # ------------------------------------------------------------------ setup
    def _setup_distributed(self) -> None:
        c = self.config
        if c.device == "auto":
            self.device = torch.device("cuda", self.env.local_rank) if torch.cuda.is_available() else torch.device("cpu")
        else:
            self.device = torch.device(c.device)
            if self.device.type == "cuda" and self.device.index is None:
                self.device = torch.device("cuda", self.env.local_rank)
        if self.device.type == "cuda":
            torch.cuda.set_device(self.device)
            from llmctl.exec.gemm_tuning import enable_tuned_gemms

            enable_tuned_gemms()
            if os.environ.get("LLMCTL_STREAM_CHECK") == "1":
                # stream-race checker: every tensor access is tracked per stream and an access
                # not ordered after the last conflicting one (event/wait_stream) raises
                from torch.cuda._sanitizer import enable_cuda_sanitizer

                enable_cuda_sanitizer()
        backend = c.distributed_backend
        if backend == "auto":
            backend = "nccl" if self.device.type == "cuda" else "gloo"
        self.backend = backend
        if self.env.world_size > 1 and not dist.is_initialized():
            import datetime

            kw = {"timeout": datetime.timedelta(seconds=c.collective_timeout_s)}
            if backend == "nccl":
                kw["device_id"] = self.device
                # surface collective timeouts/errors as exceptions (torchrun then restarts)
                os.environ.setdefault("TORCH_NCCL_ASYNC_ERROR_HANDLING", "1")
                # RCCL streams at high priority: the bucketed reduce-scatters / all-gathers
                # overlapped with backward / forward get their workgroups dispatched ahead of
                # the GEMM grids, so the last buckets are not left exposed after backward
                os.environ.setdefault("TORCH_NCCL_HIGH_PRIORITY", "1")
            from llmctl.utils.env import init_process_group

            init_process_group(backend, **kw)
        if self.env.world_size > 1 and backend == "gloo" and self.device.type == "cuda":
            # single-GPU multi-rank rehearsal: device tensors cross gloo through host copies
            from llmctl.comms import host_staging

            host_staging.install()
        if c.pack_sequences and c.context_parallel > 1:
            raise NotImplementedError("pack_sequences with context parallelism is not supported")
        if c.expert_parallel > 1 and (c.tensor_parallel > 1 or c.pipeline_parallel > 1 or c.context_parallel > 1
                                      or c.zero_stage >= 3):
            raise NotImplementedError("expert_parallel composes with DP / ZeRO-1/2 only")
        self.pg: ProcessGroups = build_process_groups(tp=c.tensor_parallel, pp=c.pipeline_parallel,
                                                      cp=c.context_parallel, ep=c.expert_parallel)
        self.rank = self.pg.rank
        self.is_main = self.rank == 0

    def _build(self) -> None:
        c, mc = self.config, self.model_config
        pg = self.pg
        L = mc.layers
        pp, pp_rank = pg.layout.pp, pg.pp_rank
        # balanced contiguous layer split (embedding / head stages get one fewer layer
        # when the count does not divide; the planner's shard_map uses the same rule)
        from llmctl.partition.shard_map import split_layers

        V = max(int(c.virtual_stages or 1), 1) if pp > 1 else 1
        ranges = None
        if V > 1:  # rank r owns virtual stages r, r + pp, ... (chunks of the pp*V-way split)
            if L < pp * V:
                raise ValueError(f"{L} layers cannot fill pipeline_parallel*virtual_stages = {pp * V} stages")
            if c.zero_stage >= 3:
                raise NotImplementedError("virtual pipeline stages with ZeRO-3 are not supported")
            split = split_layers(L, pp * V)
            ranges = [split[v * pp + pp_rank] for v in range(V)]
            lo, hi = ranges[0][0], ranges[-1][1]
        else:
            lo, hi = split_layers(L, pp)[pp_rank]
        if mc.is_moe and pp > 1:
            # the pipeline stages compute only the LM loss: the router aux loss would be dropped
            raise NotImplementedError("MoE models with pipeline parallelism are not supported")
        pc = ParallelContext(
            tp_group=pg.tp_group, tp_size=pg.layout.tp, tp_rank=pg.tp_rank,
            sequence_parallel=c.sequence_parallel and pg.layout.tp > 1,
            layer_start=lo, layer_end=hi, has_embedding=pp_rank == 0, has_head=pp_rank == pp - 1, layer_ranges=ranges,
            activation_checkpoint=c.activation_checkpoint,
            cp_group=pg.cp_group, cp_size=pg.layout.cp, cp_rank=pg.cp_rank, cp_mode=c.context_parallel_mode,
            cp_zigzag=self._cp_zigzag(),
            ep_group=pg.ep_group, ep_size=pg.layout.ep, ep_rank=pg.ep_rank)
        # identical init on every DP replica (seeded; TP ranks get different shards, so
        # their seeds differ by tp_rank/pp_rank only)
        torch.manual_seed(c.seed + 1000 * pg.tp_rank + 100000 * pp_rank)
        self.model = build_model(mc, device=self.device, dtype=c.dtype, pc=pc)
        self.pc = pc
        dp = pg.layout.dp
        align = 64 * max(dp, 1)
        grad_dtype = self._main_grad_dtype()
        self.grad_dtype = grad_dtype
        if grad_dtype != c.dtype and self.is_main:
            n = sum(p.numel() for p in self.model.parameters())
            log.info("main gradients in %s (main_grads=%s: grad accumulation / PP): +%.2f GB of gradient memory "
                     "and %dx the DP bucket bytes vs %s", str(grad_dtype).replace("torch.", ""), c.main_grads,
                     n * (4 - torch.tensor([], dtype=c.dtype).element_size()) / 1e9,
                     4 // torch.tensor([], dtype=c.dtype).element_size(), str(c.dtype).replace("torch.", ""))
        bucket_numel = int(c.bucket_mb * 2**20 / torch.tensor([], dtype=grad_dtype).element_size())
        self.grad_sink = None
        if c.zero_stage >= 3 and dp > 1:
            if pp > 1 and mc.tie_word_embeddings:
                # the tied copy would need its ZeRO-3 unit gathered for the broadcast and its
                # grad reduced from the unit's flat shard: not implemented, so refuse loudly
                raise NotImplementedError("ZeRO-3 with pipeline parallelism and tied word embeddings is not supported")
            from llmctl.parallel.zero import Zero3Model

            self.zero3 = Zero3Model(self.model, dp_group=pg.dpcp_group, dtype=c.dtype)
            self.flat = self.zero3.flat
        else:
            self.zero3 = None
            named = list(self.model.named_parameters())
            if pg.layout.ep > 1:  # expert shards: their own flat buffer, reduced over expert-DP
                named = [(n, p) for n, p in named if not getattr(p, "expert", False)]
            solo = ("embed", "lm_head") if (pp > 1 and mc.tie_word_embeddings) else ()
            self.flat = FlatParameters(named, bucket_numel=bucket_numel, align=align, solo=solo,
                                       grad_dtype=grad_dtype)
            # kernel-written gradients (no AccumulateGrad pass)
            from llmctl.exec.linear import GradSink

            tied = mc.tie_word_embeddings
            leafs = ("wqkv", "wo", "w_up", "w_down") + (() if tied else ("lm_head",))
            # norm weights and biases too (their kernels write the flat gradient: no add and no fill per vector), the biases
            # where every one of them goes through ``linear``
            leafs += ("attn_norm_w", "mlp_norm_w", "final_norm_w", "attn_norm_b", "mlp_norm_b", "final_norm_b")
            if pg.layout.tp == 1 and not mc.is_moe and not mc.gated_mlp:
                leafs += ("bqkv", "bo", "b_up", "b_down")
            # the embedding, where its rows are not shared out among ranks; tied, the output projection writes it too, and has to be here
            if pg.layout.tp == 1 and not (tied and pp > 1):
                leafs += ("embed",)
            self.grad_sink = GradSink()
            self.flat.install_sinks(self.grad_sink, lambda n, p: 0 if n.split(".")[-1] not in leafs else 2 if tied and n == "embed" else 1)
        if pp > 1 and mc.tie_word_embeddings:
            from llmctl.parallel.pipeline import broadcast_tied_embedding

            broadcast_tied_embedding(self.model, pg)  # before FlatAdamW snapshots the masters
        norm_group = pg.pp_group if pp > 1 else None
        self.optimizer = FlatAdamW(self.flat, lr=c.learning_rate, betas=tuple(c.betas), eps=c.eps,
                                   weight_decay=c.weight_decay, max_grad_norm=c.gradient_clipping,
                                   dp_group=pg.dpcp_group, zero_stage=min(c.zero_stage, 2) if self.zero3 is None else 0,
                                   tp_group=pg.tp_group, norm_group=norm_group)
        if self.zero3 is not None:
            self.zero3.attach_optimizer(self.optimizer)
            self.sync = None
        else:
            mode = "reduce_scatter" if self.optimizer.zero_stage >= 1 else "allreduce"
            # gradients are summed over every replica of the parameters: DP × CP
            self.sync = GradSyncEngine(self.flat, group=pg.dpcp_group, mode=mode,
                                       shard_view=self.optimizer.shard_view if mode == "reduce_scatter" else None,
                                       tp_group=pg.tp_group, sequence_parallel=pc.sequence_parallel)
        if self.zero3 is None and self.optimizer.zero_stage >= 1 and dp > 1:
            self._install_param_gather_hooks()
        elif (self.zero3 is None and self.optimizer.zero_stage == 0 and self.device.type == "cuda" and pp == 1
              and self.knobs.overlap_optimizer):
            # opt-in: measured neutral on GPT-7B mb 12 (27.7k vs 27.9k tok/s in one A/B,
            # profiles/bench_r1_overlap_opt_ab.jsonl) — the concurrent AdamW slows the GEMMs
            # about as much as it hides
            self._install_param_gather_hooks()
            self.optimizer.overlap_param_gather = False
            self.optimizer.overlap_update = True
        self.eflat = self.eopt = self.esync = None
        if pg.layout.ep > 1:
            experts = [(n, p) for n, p in self.model.named_parameters() if getattr(p, "expert", False)]
            edp = dp // pg.layout.ep
            # expert gradients stay in the parameter dtype: size their buckets by that element
            ebucket = int(c.bucket_mb * 2**20 / torch.tensor([], dtype=c.dtype).element_size())
            self.eflat = FlatParameters(experts, bucket_numel=ebucket, align=64 * edp)
            self.eopt = FlatAdamW(self.eflat, lr=c.learning_rate, betas=tuple(c.betas), eps=c.eps,
                                  weight_decay=c.weight_decay, max_grad_norm=c.gradient_clipping,
                                  dp_group=pg.edp_group, zero_stage=0)
            self.esync = GradSyncEngine(self.eflat, group=pg.edp_group, mode="allreduce")
        total = c.max_steps if c.max_steps > 0 else 1000
        self.scheduler = LRSchedule(c.learning_rate, c.scheduler, c.warmup_steps, total)
        self.pipeline = None
        if pp > 1:
            from llmctl.parallel.pipeline import PipelineSchedule

            self.pipeline = PipelineSchedule(self, num_microbatches=c.num_microbatches or 2 * pp)
        n_local = sum(p.numel() for p in self.model.parameters())
        log.info("rank %d: tp=%d pp=%d dp=%d zero=%d layers[%d:%d] local params %.3fB on %s",
                 self.rank, pg.layout.tp, pp, dp, c.zero_stage, lo, hi, n_local / 1e9, self.device)

    def _main_grad_dtype(self) -> torch.dtype:
        c = self.config
        mode = (c.main_grads or "auto").lower()
        if mode not in ("auto", "fp32", "bf16"):
            raise ValueError(f"main_grads must be auto | fp32 | bf16, got {c.main_grads!r}")
        if c.dtype == torch.float32 or mode == "bf16":
            return c.dtype
        accum = c.gradient_accumulation_steps > 1 or c.pipeline_parallel > 1
        if mode == "auto" and not accum:
            return c.dtype
        if c.zero_stage >= 3:
            if mode == "fp32":
                log.warning("main_grads=fp32 is not implemented for ZeRO-3: gradients stay %s", c.dtype)
            return c.dtype
        return torch.float32

    def _install_param_gather_hooks(self) -> None:
        """ZeRO-1/2: the post-step all-gather of updated parameter shards overlaps the next
        forward — each decoder layer (and the top-level module, for embedding / head / final
        norm) waits only for the buckets holding its own parameters.  ZeRO-0 on one GPU uses
        the same hooks for the side-stream optimizer update (``FlatAdamW.overlap_update``)."""
        flat, opt = self.flat, self.optimizer

        def buckets_of(params):
            return sorted({flat.param_bucket[id(p)].index for p in params if id(p) in flat.param_bucket})

        def hook_for(idx):
            return lambda module, args: opt.wait_params(idx)

        # the embedding buckets are gathered first and the final-norm / LM-head buckets last
        # (flat-offset order): the top-level pre-hook waits only for the former, the head for
        # the latter — waiting for every top-level parameter up front would serialise the
        # whole gather (or side-stream update) before the first layer
        named = [(n, p) for n, p in self.model.named_parameters() if not n.startswith("layers.")]
        front = [p for n, p in named if n in ("embed", "pos_embed")]
        back = [p for n, p in named if n not in ("embed", "pos_embed")]
        self._gather_hooks = [self.model.register_forward_pre_hook(hook_for(buckets_of(front)))]
        for layer in self.model.layers:
            self._gather_hooks.append(layer.register_forward_pre_hook(hook_for(buckets_of(layer.parameters()))))
        back_idx = buckets_of(back)
        self.model.pre_head_hook = lambda: opt.wait_params(back_idx)
        opt.overlap_param_gather = True

    # ------------------------------------------------------------------ data
    def make_data(self):
        from llmctl.io.dataset import build_dataset

        return build_dataset(self.config, self.model_config, dp_rank=self.pg.dp_rank, dp_size=self.pg.layout.dp,
                             device=self.device)

    # ------------------------------------------------------------------ step
    def _late_zero_grad(self) -> None:
        self.optimizer.wait_params()  # every bucket's update has been ordered before this point
        self.flat.zero_grad()

    def _packing(self, input_ids, labels):
        """Packed sequences: the per-row document map and the labels with separator targets
        masked (a separator's next-token label belongs to the next document)."""
        if not self.config.pack_sequences:
            return labels, None
        from llmctl.ops.ref import document_starts

        doc_start = document_starts(input_ids, self.config.doc_separator)
        return labels.masked_fill(input_ids == self.config.doc_separator, -100), doc_start

    def _forward_backward(self, input_ids, labels, denom, before_backward=None):
        labels, doc_start = self._packing(input_ids, labels)
        loss = self.model(input_ids, labels, loss_denom=denom, doc_start=doc_start)
        if self.faults and self.faults.nan_loss(self.global_step + 1):
            loss = loss * float("nan")
        if before_backward is not None:
            before_backward()
        loss.backward()
        return loss.detach()

    def train_step(self, batches: List[Tuple[torch.Tensor, torch.Tensor]]) -> Dict[str, torch.Tensor]:
        """One optimizer step over ``len(batches)`` micro-batches (grad accumulation).  Returns
        device tensors (no host sync): mean loss and grad norm."""
        from llmctl.config.knobs import use

        use(self.knobs)
        self.model.train()
        loss = self.step_graphs.run(self, batches)
        if loss is not None:
            return self._apply(batches, loss)
        # with the side-stream update the previous step may still be reading the gradients:
        # zero them only once the first forward has waited for every bucket (its pre-hooks)
        late_zero = self.optimizer.overlap_update
        if not late_zero:
            self.flat.zero_grad()
        if self.eflat is not None:
            self.eflat.zero_grad()
        if self.zero3 is not None:
            self.zero3.begin_step()
        cpn = self.pg.layout.cp
        if cpn > 1:  # this rank's contiguous chunk of every sequence
            batches = self._cp_split(batches)
        if self.pipeline is not None:
            self.optimizer.wait_params()  # stages call embed/head outside the hooked forward
            loss = self.pipeline.run(batches)
        else:
            n = len(batches)
            tokens = batches[0][1].numel() * cpn  # per replica: the CP ranks share one sequence
            # loss is a per-token mean inside each micro-batch; dividing the denominator
            # by n makes the accumulated gradient the mean over all n micro-batches
            denom = float(tokens * n)
            losses = []
            for i, (x, y) in enumerate(batches):
                last = i == n - 1
                if self.zero3 is not None:
                    ctx = self.zero3.no_sync() if not last else _null()
                else:
                    ctx = self.sync.no_sync() if not last else _null()
                ectx = self.esync.no_sync() if (self.esync is not None and not last) else _null()
                with ctx, ectx:
                    losses.append(self._forward_backward(x, y, denom, before_backward=(
                        self._late_zero_grad if late_zero and i == 0 else None)))
            loss = losses[0] if n == 1 else torch.stack(losses).sum()
        if self.zero3 is not None:
            self.zero3.finish_grad_sync()
        elif self.sync is not None:
            self.sync.finish()
        if self.esync is not None:
            self.esync.finish()
        if self.pipeline is not None:
            self.pipeline.sync_tied_grads()
        return self._apply(batches, loss)

    def _gradients(self, x, y, denom: float) -> torch.Tensor:
        """What a step of one micro-batch on one GPU does before the optimizer (``step_graph`` records it)."""
        self.flat.zero_grad()
        loss = self._forward_backward(x, y, denom)
        self.sync.finish()
        return loss

    def _apply(self, batches, loss) -> Dict[str, torch.Tensor]:
        """The optimizer's part of ``train_step``."""
        lr = self.scheduler(self.global_step)  # 0-based index of the step being applied (HF)
        self.global_step += 1
        if self.eopt is not None:
            # one global clip norm: the expert shards are distinct across the EP group
            enorm = self.eopt.grad_norm_sq().clone()
            dist.all_reduce(enorm, group=self.pg.ep_group)
            gnorm = self.optimizer.step(lr=lr, grad_divisor=float(self.pg.layout.dp), extra_norm_sq=enorm)
            self.eopt.step(lr=lr, grad_divisor=float(self.pg.layout.dp), coef=self.optimizer.last_coef)
        else:
            gnorm = self.optimizer.step(lr=lr, grad_divisor=float(self.pg.layout.dp))
        if self.zero3 is not None:
            self.zero3.after_step()
        self._weights_changed()
        self.consumed_samples += sum(b[0].shape[0] for b in batches) * self.pg.layout.dp
        return {"loss": loss, "grad_norm": gnorm, "lr": torch.tensor(lr)}

    def _cp_zigzag(self) -> bool:
        from llmctl.parallel.context_parallel import zigzag_enabled

        return self.pg.layout.cp > 1 and self.config.context_parallel_mode == "ring" and zigzag_enabled()

    def _cp_split(self, batches):
        from llmctl.parallel.context_parallel import split_sequence

        cpn, r, z = self.pg.layout.cp, self.pg.cp_rank, self._cp_zigzag()
        return [(split_sequence(x, cpn, r, z), split_sequence(y, cpn, r, z)) for x, y in batches]

    @torch.no_grad()
    def evaluate(self, batches) -> float:
        self.optimizer.wait_params()
        self.model.eval()
        tot, n = 0.0, 0
        cpn = self.pg.layout.cp
        root = self.zero3 is not None and self.pipeline is not None
        if root:
            self.zero3.gather_root()
        for x, y in batches:
            denom = float(y.numel())  # whole-sequence token count (CP ranks hold chunks)
            if cpn > 1:
                (x, y), = self._cp_split([(x, y)])
            if self.pipeline is not None:
                l = self.pipeline.eval_loss(x, y, denom)
            else:
                y, doc_start = self._packing(x, y)
                l = self.model(x, y, loss_denom=denom, doc_start=doc_start)
                if cpn > 1:  # partial sums of one mean
                    l = l.detach().float().reshape(1).clone()
                    dist.all_reduce(l, group=self.pg.cp_group)
            tot += float(l)
            n += 1
        if root:
            self.zero3.release_root()
        return tot / max(n, 1)

    # ------------------------------------------------------------------ loop
    def train(self, data_iter: Optional[Iterator] = None) -> Dict[str, float]:
        from llmctl.io.checkpoint import CheckpointManager
        from llmctl.runtime.replay import write_manifest

        from llmctl.config.knobs import use

        use(self.knobs)
        c = self.config
        ckpt = CheckpointManager(self, c.output_dir)
        resume = c.resume_from_checkpoint
        if resume == "auto":  # elastic restarts: newest complete checkpoint of this run, if any
            resume = c.output_dir if (Path(c.output_dir) / "latest").exists() else None
        if resume:
            ckpt.load(resume)
            if self.is_main:
                log.info("resumed from %s at step %d (restart attempt %s)", resume, self.global_step,
                         os.environ.get("TORCHELASTIC_RESTART_COUNT", "0"))
        accum = max(c.gradient_accumulation_steps, 1)
        if self.pipeline is not None:
            accum = self.pipeline.num_microbatches
        if data_iter is not None:
            data = data_iter
        else:
            ds = self.make_data()
            if self.global_step and hasattr(ds, "skip"):
                ds.skip(self.global_step * accum)  # resume: continue the sample stream, not restart it
            data = iter(ds)
        max_steps = c.max_steps if c.max_steps > 0 else None
        if max_steps is None:
            spe = c.samples_per_epoch or 1000 * c.batch_size
            steps_per_epoch = max(spe // (c.batch_size * accum * self.pg.layout.dp), 1)
            max_steps = steps_per_epoch * c.num_epochs
        prof = self._make_profiler()
        tokens_per_step = c.batch_size * c.seq_len * accum * self.pg.layout.dp
        flops_per_token = self.model_config.flops_per_token(c.seq_len)
        t_last = time.time()
        last_loss = float("nan")
        history = []
        while self.global_step < max_steps:
            batches = [next(data) for _ in range(accum)]
            if prof is not None:
                with torch.profiler.record_function("llmctl.train_step"):
                    out = self.train_step(batches)
                prof.step()
            else:
                out = self.train_step(batches)
            s = self.global_step
            if s % c.logging_steps == 0 or s == max_steps:
                if self.device.type == "cuda":
                    torch.cuda.synchronize()
                dt = (time.time() - t_last) / (c.logging_steps if s % c.logging_steps == 0 else 1)
                t_last = time.time()
                last_loss = float(out["loss"])
                if self.pipeline is not None:
                    last_loss = self.pipeline.broadcast_loss(out["loss"])
                gn = float(out["grad_norm"])
                tps = tokens_per_step / max(dt, 1e-9)
                mfu = tps * flops_per_token / (self._peak_flops() * self.pg.layout.world_size)
                rec = dict(step=s, loss=last_loss, grad_norm=gn, lr=float(out["lr"]), step_time=dt,
                           tokens_per_sec=tps, mfu=mfu)
                history.append(rec)
                if self.is_main:
                    log.info("step %d loss %.4f gnorm %.3f lr %.2e %.3fs/step %.0f tok/s MFU %.1f%%", s, last_loss,
                             gn, rec["lr"], dt, tps, 100 * mfu)
                for h in self.metrics_hooks:
                    h(rec)
            if self.faults:
                if self.faults.due(s):
                    ckpt.wait()
                self.faults.after_step(s)
            if c.eval_steps and s % c.eval_steps == 0:
                ev = [next(data) for _ in range(c.eval_batches)]
                vl = self.evaluate(ev)
                if self.is_main:
                    log.info("step %d eval loss %.4f", s, vl)
            if c.save_steps and s % c.save_steps == 0:
                ckpt.save(f"checkpoint-{s}")
                write_manifest(self, history)
        if prof is not None:
            prof.stop()
        ckpt.save("final", final=True)
        ckpt.wait()
        write_manifest(self, history, status="complete")
        return {"final_loss": last_loss, "steps": self.global_step, "history": history}

    # ------------------------------------------------------------------ state (layout-independent)
    def load_full_state_dict(self, full: Dict[str, torch.Tensor]) -> None:
        """Load unsharded tensors (names ``layers.<global>.<p>``) into this rank's shards and
        restart the optimizer masters from them."""
        from llmctl.io.checkpoint import _global_name, _reinit_master_from_params, shard_tp

        named = self.zero3.full_named_parameters() if self.zero3 is not None else list(self.model.named_parameters())
        with torch.no_grad():
            for n, p in named:
                g = self._expert_global(_global_name(n, self.pc.layer_index))
                if g == "lm_head" and g not in full and self.model_config.tie_word_embeddings:
                    g = "embed"  # the last pipeline stage's copy of a tied matrix
                t = shard_tp(g, full[g], self.pg.layout.tp, self.pg.tp_rank, self.model_config)
                p.copy_(t.to(p.dtype))
        if self.zero3 is not None:
            self.zero3.reload_shards_from_full()
        _reinit_master_from_params(self)
        self._weights_changed()
        if self.eopt is not None:
            with torch.no_grad():
                self.eopt.master.copy_(self.eflat.data.float())
                self.eopt.exp_avg.zero_()
                self.eopt.exp_avg_sq.zero_()

    def _weights_changed(self) -> None:
        """Parameters were rewritten (optimizer step, state load): derived copies (the
        transposed dgrad weights) refresh on next use."""
        if self.grad_sink is not None:
            self.grad_sink.epoch += 1

    def _expert_global(self, name: str) -> str:
        """Expert parameter names carry the rank-local expert index; checkpoints use global ids."""
        if self.pg.layout.ep == 1 or (".experts_up." not in name and ".experts_down." not in name):
            return name
        from llmctl.models.moe import expert_param_global_name

        return expert_param_global_name(name, self.pg.ep_rank * (self.model_config.num_experts // self.pg.layout.ep))

    def gather_full_state_dict(self) -> Dict[str, torch.Tensor]:
        """Collective: every rank returns the full unsharded model (CPU tensors)."""
        from llmctl.io.checkpoint import _global_name, consolidate_tp

        self.optimizer.wait_params()
        named = self.zero3.full_named_parameters() if self.zero3 is not None else list(self.model.named_parameters())
        local = {self._expert_global(_global_name(n, self.pc.layer_index)): p.detach().float().cpu() for n, p in named}
        if self.zero3 is not None:
            self.zero3.release_all()
        if not dist.is_initialized():
            return local
        parts: List[Dict[str, torch.Tensor]] = [None] * dist.get_world_size()  # type: ignore
        dist.all_gather_object(parts, (self.pg.tp_rank, self.pg.dp_rank, local))
        by_name: Dict[str, Dict[int, torch.Tensor]] = {}
        ep = self.pg.layout.ep
        for tp_rank, dp_rank, sd in parts:
            for k, v in sd.items():
                # replicated parameters from DP rank 0; expert shards from each rank of EP block 0
                is_expert = ep > 1 and (".experts_up." in k or ".experts_down." in k)
                if dp_rank != 0 and not (is_expert and dp_rank < ep):
                    continue
                by_name.setdefault(k, {})[tp_rank] = v
        if self.model_config.tie_word_embeddings:
            by_name.pop("lm_head", None)  # the pipeline's copy of ``embed``: not a model parameter
        return {k: consolidate_tp(k, [s[i] for i in sorted(s)], self.model_config) for k, s in by_name.items()}

    def _make_profiler(self):
        """``torch.profiler`` over the schedule ``profile_schedule`` (``wait=a,warmup=b,active=c``
        or the reference config's ``step(N)`` = profile step N); one Chrome trace per rank."""
        c = self.config
        if not c.profile_dir:
            return None
        import re

        m = re.fullmatch(r"\s*step\((\d+)\)\s*", c.profile_schedule)
        if m:
            n = max(int(m.group(1)), 1)
            kw = dict(wait=max(n - 2, 0), warmup=1 if n >= 2 else 0, active=1, repeat=1)
        else:
            kw = {k.strip(): int(v) for k, v in (x.split("=") for x in c.profile_schedule.split(",") if x.strip())}
            kw.setdefault("repeat", 1)
        out = Path(c.profile_dir)
        out.mkdir(parents=True, exist_ok=True)
        rank = self.rank

        def ready(p):
            p.export_chrome_trace(str(out / f"trace_rank{rank:05d}_step{self.global_step}.json"))

        acts = [torch.profiler.ProfilerActivity.CPU]
        if self.device.type == "cuda":
            acts.append(torch.profiler.ProfilerActivity.CUDA)  # roctracer on ROCm
        prof = torch.profiler.profile(activities=acts, schedule=torch.profiler.schedule(**kw), on_trace_ready=ready)
        prof.start()
        return prof

    def _peak_flops(self) -> float:
        if self.device.type == "cuda":
            from llmctl.metrics.flops import device_peak_flops

            return device_peak_flops(self.config.dtype)
        return 1e12

    def shutdown(self):
        if dist.is_initialized():
            dist.barrier()
            dist.destroy_process_group()


class _null:
    def __enter__(self):
        return self

    def __exit__(self, *a):
        return False

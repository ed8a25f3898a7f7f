"""Llama-3 dense decoder for MI355X.

The model runner behind engine.generate() — the native replacement for the
reference's remote `chat.completions.create` model execution
(k_llms/resources/completions/completions.py:73). Torch modules orchestrate
the products (ops.linear and the few-row kernels, hipBLASLt/rocBLAS where it is
the faster one) while every other hot op (RMSNorm, RoPE, varlen prefill
attention, paged decode attention, SwiGLU, KV scatter) dispatches to the
hand-written CDNA4 HIP kernels in kllms_amd.ops.

Two forward modes driven by ForwardBatch:
- prefill: packed varlen batch (shared prefill across requests), causal
  attention over the fresh contiguous K/V, K/V scattered into paged cache;
- decode: one token per stream against the paged KV cache (the hipGraph-
  captured hot loop).
"""

from __future__ import annotations

import math
from dataclasses import dataclass, replace
from typing import List, Literal, Optional, Tuple

import torch
import torch.nn as nn

from .. import ops
from ..engine.config import ModelArchConfig
from ..ops.torch_ref import build_cos_sin_cache
from ..parallel.tp import ColumnParallelLinear, ParallelContext, RowParallelLinear


@dataclass
class ForwardBatch:
    mode: Literal["prefill", "decode", "segments"]
    positions: torch.Tensor              # [T] long
    slot_mapping: torch.Tensor           # [T] long — flat KV slots to write
    kv_caches: List[Tuple]  # per layer (k, v, k_scale|None, v_scale|None)
    cu_seqlens: Optional[torch.Tensor] = None   # [n_seq+1] int32 (prefill)
    block_tables: Optional[torch.Tensor] = None  # [B, max_blocks] int32 (decode)
    context_lens: Optional[torch.Tensor] = None  # [B] int32 (decode)
    # segment form, used by models with recurrent state (any mix of prompt
    # portions and single decoded tokens in one step): rows
    # cu_seqlens[b]..cu_seqlens[b+1] continue sequence b at position
    # seg_start[b]; block_tables has one row per SEGMENT; kv_caches holds one
    # engine.kvcache.LayerState per layer
    seg_start: Optional[torch.Tensor] = None     # [B] int32
    state_slots: Optional[torch.Tensor] = None   # [B] int32
    token_seg: Optional[torch.Tensor] = None     # [T] int32 — segment of each row
    # host copy of (first position, row count) per segment, when the step was
    # built on the host (absent for device-resident decode state): lets a
    # layer plan per-piece kernels without a device sync; plans are cached here
    host_segs: Optional[list] = None
    plans: Optional[dict] = None
    # decode-mode batches built from segments of an attention-only model (with
    # host_segs and seg_start): one block table per segment, so that the rows of
    # a long segment can attend together
    seg_tables: Optional[torch.Tensor] = None    # [B, max_blocks] int32


class LlamaAttention(nn.Module):
    def __init__(self, cfg: ModelArchConfig, ctx: ParallelContext, layer_idx: int, dtype):
        super().__init__()
        self.layer_idx = layer_idx
        tp = ctx.world_size
        assert cfg.num_heads % tp == 0 and cfg.num_kv_heads % tp == 0
        self.num_heads = cfg.num_heads // tp
        self.num_kv_heads = cfg.num_kv_heads // tp
        self.head_dim = cfg.head_dim_
        self.scale = 1.0 / math.sqrt(self.head_dim)
        q_size = cfg.num_heads * self.head_dim
        kv_size = cfg.num_kv_heads * self.head_dim
        # Fused QKV, head-sharded across ranks (each rank holds its q, k and
        # v head shards — partition-aware slicing)
        self.qkv_proj = ColumnParallelLinear(
            cfg.hidden_size, q_size + 2 * kv_size, ctx, dtype=dtype,
            partition_sizes=[q_size, kv_size, kv_size],
            bias=cfg.attention_qkv_bias,  # Qwen2-style
        )
        self.o_proj = RowParallelLinear(q_size, cfg.hidden_size, ctx, dtype=dtype)
        self._q = self.num_heads * self.head_dim
        self._kv = self.num_kv_heads * self.head_dim

    def forward(self, hidden: torch.Tensor, batch: ForwardBatch, cos_sin: torch.Tensor) -> torch.Tensor:
        return self.o_proj(self.attend(hidden, batch, cos_sin).reshape(hidden.shape[0], -1))

    def attend(self, hidden: torch.Tensor, batch: ForwardBatch, cos_sin: torch.Tensor) -> torch.Tensor:
        """The heads' results [T, H, D]; keys and values are stored."""
        T = hidden.shape[0]
        qkv = self.qkv_proj(hidden)
        # strided views into the fused QKV row — the HIP kernels take the
        # token stride, so no contiguity copies on the hot path
        q, k, v = qkv.split([self._q, self._kv, self._kv], dim=-1)
        q = q.view(T, self.num_heads, self.head_dim)
        k = k.view(T, self.num_kv_heads, self.head_dim)
        v = v.view(T, self.num_kv_heads, self.head_dim)
        k_cache, v_cache, k_scale, v_scale = batch.kv_caches[self.layer_idx]
        ops.rope_store(q, k, v, batch.positions, cos_sin, k_cache, v_cache, batch.slot_mapping, k_scale, v_scale)

        if batch.mode == "prefill":
            return ops.attn_prefill_varlen(q, k, v, batch.cu_seqlens, self.scale, (batch.plans or {}).get("prefill"))
        return self.attend_cache(q, batch)

    def attend_cache(self, q: torch.Tensor, batch: ForwardBatch, arrived: Optional[torch.Tensor] = None) -> torch.Tensor:
        """Attention of decode-mode rows q [T, H, D] against the paged cache; ``arrived``: zeros of ops.attn_decode_paged."""
        k_cache, v_cache, k_scale, v_scale = batch.kv_caches[self.layer_idx]
        paged = (batch.plans or {}).get("paged")
        if paged is not None and k_scale is None:
            plan, short = paged
            return ops.attn_segments_paged(q, k_cache, v_cache, batch.block_tables, batch.context_lens, self.scale,
                                           plan, short, batch.seg_tables, batch.seg_start)
        return ops.attn_decode_paged(
            q, k_cache, v_cache, batch.block_tables, batch.context_lens, self.scale,
            k_scale, v_scale, arrived,
        )


class LlamaMLP(nn.Module):
    def __init__(self, cfg: ModelArchConfig, ctx: ParallelContext, dtype):
        super().__init__()
        self.gate_up_proj = ColumnParallelLinear(
            cfg.hidden_size, 2 * cfg.intermediate_size, ctx, dtype=dtype,
            partition_sizes=[cfg.intermediate_size, cfg.intermediate_size],
        )
        self.down_proj = RowParallelLinear(cfg.intermediate_size, cfg.hidden_size, ctx, dtype=dtype)
        self._i = cfg.intermediate_size // ctx.world_size

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return self.down_proj(self.activate(x))

    def activate(self, x: torch.Tensor) -> torch.Tensor:
        """silu(gate) * up."""
        p = self.gate_up_proj
        plain = ops.only_weights(p, ColumnParallelLinear) and ops.no_global_hooks()
        act = ops.linear_silu(x, p.weight) if plain and p.bias is None else None
        if act is not None:
            return act
        gate, up = p(x).split([self._i, self._i], dim=-1)
        return ops.silu_mul(gate, up)


class RMSNormModule(nn.Module):
    def __init__(self, hidden_size: int, eps: float, dtype):
        super().__init__()
        self.weight = nn.Parameter(torch.empty(hidden_size, dtype=dtype), requires_grad=False)
        self.eps = eps


class LlamaDecoderLayer(nn.Module):
    def __init__(self, cfg: ModelArchConfig, ctx: ParallelContext, layer_idx: int, dtype):
        super().__init__()
        self.input_layernorm = RMSNormModule(cfg.hidden_size, cfg.rms_norm_eps, dtype)
        self.self_attn = LlamaAttention(cfg, ctx, layer_idx, dtype)
        self.post_attention_layernorm = RMSNormModule(cfg.hidden_size, cfg.rms_norm_eps, dtype)
        self.mlp = self._make_mlp(cfg, ctx, dtype)

    def _make_mlp(self, cfg: ModelArchConfig, ctx: ParallelContext, dtype):
        return LlamaMLP(cfg, ctx, dtype)

    def forward(
        self, hidden: torch.Tensor, residual: Optional[torch.Tensor], batch: ForwardBatch, cos_sin: torch.Tensor
    ) -> Tuple[torch.Tensor, torch.Tensor]:
        if residual is None:
            residual = hidden
            hidden = ops.rmsnorm(hidden, self.input_layernorm.weight, self.input_layernorm.eps)
        else:
            hidden, residual = ops.fused_add_rmsnorm(
                hidden, residual, self.input_layernorm.weight, self.input_layernorm.eps
            )
        hidden = self.self_attn(hidden, batch, cos_sin)
        hidden, residual = ops.fused_add_rmsnorm(
            hidden, residual, self.post_attention_layernorm.weight, self.post_attention_layernorm.eps
        )
        hidden = self.mlp(hidden)
        return hidden, residual


class LlamaForCausalLM(nn.Module):
    layer_cls = LlamaDecoderLayer
    _once = False           # ops.weights_once

    def __init__(self, cfg: ModelArchConfig, ctx: Optional[ParallelContext] = None, dtype=torch.bfloat16):
        super().__init__()
        self.cfg = cfg
        self.ctx = ctx or ParallelContext()
        self.dtype = dtype
        self.embed_tokens = nn.Embedding(cfg.vocab_size, cfg.hidden_size, dtype=dtype)
        self.embed_tokens.weight.requires_grad_(False)
        self.layers = nn.ModuleList(
            [self.layer_cls(cfg, self.ctx, i, dtype) for i in range(cfg.num_layers)]
        )
        self.norm = RMSNormModule(cfg.hidden_size, cfg.rms_norm_eps, dtype)
        # LM head replicated across TP ranks: hidden states are replicated
        # after each layer's all-reduce, so full logits come out identical on
        # every rank — no logits gather needed.
        self.lm_head = nn.Linear(cfg.hidden_size, cfg.vocab_size, bias=False, dtype=dtype)
        self.lm_head.weight.requires_grad_(False)
        self._once = ops.weights_once(self)
        self.register_buffer(
            "cos_sin",
            build_cos_sin_cache(cfg.head_dim_, cfg.max_position_embeddings, cfg.rope_theta, "cpu",
                                rope_scaling=cfg.rope_scaling),
            persistent=False,
        )

    # --- init ---------------------------------------------------------------
    @torch.no_grad()
    def random_init_(self, seed: int = 0) -> None:
        """Deterministic, TP-degree-invariant random init: every parameter is
        generated as its FULL tensor from a per-name seed, then the local
        shard is sliced out — so TP=1/2/4/8 hold numerically identical models.
        """
        import hashlib

        tp = self.ctx.world_size
        rank = self.ctx.rank
        for name, p in self.named_parameters():
            h = int(hashlib.md5(f"{seed}/{name}".encode()).hexdigest()[:15], 16)
            g = torch.Generator(device=p.device)
            g.manual_seed(h)
            shard_dim = None
            full_shape = list(p.shape)
            mod = self._owner_module(name)
            leaf = name.split(".")[-1]
            spec = getattr(mod, "shard_spec", {})
            if isinstance(mod, ColumnParallelLinear):
                shard_dim = 0
                full_shape[0] *= tp
                full = torch.ones(full_shape, dtype=torch.float32, device=p.device) if (
                    "layernorm" in name or name.endswith("norm.weight")
                ) else torch.randn(full_shape, generator=g, dtype=torch.float32, device=p.device) * 0.02
                p.copy_(mod.shard_full_tensor(full).to(p.dtype))
                continue
            elif isinstance(mod, RowParallelLinear):
                shard_dim = 1
                full_shape[1] *= tp
            n_parts = 1
            if leaf in spec:
                entry = spec[leaf]
                # spec value: dim, or (dim, n_parts) for FUSED dims (e.g. the
                # MoE [gate;up] stack) where each equal part shards separately
                shard_dim, n_parts = entry if isinstance(entry, tuple) else (entry, 1)
                full_shape[shard_dim] *= tp
            if "layernorm" in name or name.endswith("norm.weight"):
                full = torch.ones(full_shape, dtype=torch.float32, device=p.device)
            else:
                std = 0.02
                full = torch.randn(full_shape, generator=g, dtype=torch.float32, device=p.device) * std
            if shard_dim is not None and tp > 1:
                size = p.shape[shard_dim]
                if n_parts > 1:
                    # local layout is the concat of this rank's shard of EACH
                    # part — a contiguous narrow would give rank 0 all of the
                    # first part (matches weights.py's per-part sharding)
                    part_full = full.shape[shard_dim] // n_parts
                    part_loc = size // n_parts
                    full = torch.cat(
                        [full.narrow(shard_dim, j * part_full + rank * part_loc, part_loc)
                         for j in range(n_parts)],
                        dim=shard_dim,
                    )
                else:
                    full = full.narrow(shard_dim, rank * size, size)
            p.copy_(full.to(p.dtype))
        if self.cfg.tie_word_embeddings:
            # mirror the weights loader: tied checkpoints share one matrix
            self.lm_head.weight.copy_(self.embed_tokens.weight)

    def _owner_module(self, param_name: str):
        parts = param_name.split(".")[:-1]
        mod = self
        for part in parts:
            mod = getattr(mod, part) if not part.isdigit() else mod[int(part)]
        return mod

    # --- forward ------------------------------------------------------------
    # rows up to which the fused [gate; up] product of any width is the few-row kernel's, which saves the activation's
    # launch. us, library with activation and few-row kernel, at 1 / 32 / 64 / 128 rows:
    #   27648 x 5120  82 55 / 57 59 / 60 62 / 70 85        24576 x 3072  53 31 / 36 37 at 64 / 43 49
    #   37888 x 3584  61 62 / 62 64 at 16 / 71 71 / 73 88
    SILU_ROWS_MAX = 64

    @classmethod
    def _silu_rows(cls, rows: int, weight: torch.Tensor) -> bool:
        n = weight.numel()
        return rows <= (cls.SILU_ROWS_MAX if n < 1 << 27 else 16 if n < 1 << 28 else 0)

    # More, of a width that is a power of two: the others' stages take a third longer at many rows. At 1 / 32 / 64 / 128 / 256
    # rows, 256 beside the better of library and tiles:
    #   28672 x 4096  65 42 / 55 42 / 55 43 / 58 50 / 69 63        16384 x 2048  20 14 / 20 14 / 21 15 / 24 19 / 30 26
    #   22016 x 4096  53 33 / 48 41 / 46 38 / 49 47 / 66 60        57344 x 8192  181 163 / 182 169 / 198 175 / 203 197 / 239 309
    @staticmethod
    def _silu_streams(rows: int, weight: torch.Tensor) -> bool:
        n, width = weight.shape
        return width & (width - 1) == 0 and rows <= (ops.LINEAR_SILU_MAX if n <= 32768 else ops.LINEAR_ROWS_MAX)

    def _takes_rows(self, input_ids: torch.Tensor, batch: ForwardBatch) -> bool:
        """Whether a step runs as _forward_rows: a few decode rows of an unsharded bf16 model on the GPU with the
        sizes that the few-row kernels divide."""
        return batch.mode == "decode" and input_ids.shape[0] <= ops.LINEAR_ROWS_MAX and self._rows_fit(input_ids, batch)

    def _rows_fit(self, input_ids: torch.Tensor, batch: ForwardBatch) -> bool:
        cfg = self.cfg
        at = self.layers[0].self_attn if len(self.layers) else None
        return (batch.mode in ("decode", "prefill") and at is not None and input_ids.is_cuda and input_ids.dim() == 1
                and input_ids.dtype == torch.long and input_ids.shape[0] >= 1 and self.ctx.world_size == 1
                and self.dtype == torch.bfloat16 and not ops._force_torch() and at.head_dim == 128
                and cfg.hidden_size % 128 == 0 and cfg.hidden_size <= 16384 and cfg.intermediate_size % 128 == 0
                and self.cos_sin.is_contiguous() and input_ids.is_contiguous()
                and all(t.is_contiguous() and t.numel() == input_ids.shape[0] for t in (batch.positions, batch.slot_mapping)))

    def _takes_short(self, input_ids: torch.Tensor, batch: ForwardBatch) -> bool:
        """Whether more decode rows than _takes_rows takes, or a short prompt, run as _forward_rows: up to the rows at which
        the few-row products are the faster ones, and where nothing but the modules' own forwards would run. us of the
        library's product and of linear_part with the reading of its sums, at 160 / 256 / 384 rows:
          4096 x 4096    27 19 / 23 23 / 25 29      4096 x 14336  84 43 / 63 53 / 78 66      6144 x 4096   28 24 / 40 31 / 36 40
          2048 x 8192    26 17 / 27 22 / 33 26      8192 x 8192   54 43 / 76 58 / 62 73      10240 x 8192  67 71 / 88 94
          3072 x 8192    32 26 / 38 29 / 47 35      3584 x 18944  111 54 / 130 63 / 89 72    5120 x 5120   42 29 / 55 39 / 44 42
        Whole prompts through four layers in the library and so, us at 24 / 160 / 256 / 320 / 384 tokens:
          1024  228 172 / 275 237 / 290 267 / 314 294 / 323 301      1280  271 210 / 333 311 / 372 363 / 383 385 / 387 394
          2560  397 335 / 591 533 / 672 597 / 675 619 / 701 654      3072  392 337 / 573 526 / 693 650 / 675 653 / 737 693
          3584  927 575 / 1095 822 / 1303 1009 / 1174 1074 / 1219 1145      5120  707 621 / 1123 931 / 1470 1148 / 1281 1282 / 1314 1307"""
        rows = input_ids.shape[0]
        if not (batch.mode == "prefill" or rows > ops.LINEAR_ROWS_MAX) or rows > ops.LINEAR_PART_MAX:
            return False
        if not self._rows_fit(input_ids, batch):
            return False
        at = self.layers[0].self_attn
        widest = max(at.qkv_proj.weight.shape[0], self.cfg.hidden_size)
        most = ops.LINEAR_PART_MAX if widest <= 6144 else 256 if widest <= 8192 else ops.LINEAR_ROWS_MAX
        if 1024 < self.cfg.hidden_size < 1536:
            most = 288
        return rows <= most and self._only_weights(input_ids, batch)

    def _only_weights(self, input_ids: torch.Tensor, batch: ForwardBatch) -> bool:
        """Whether the layers' modules are the plain ones, nothing looks on at their calls, and their weights are such as the
        few-row products read. Other weights are the library's."""
        plain = ops.only_weights
        if not (ops.no_global_hooks() and ops.plain_call(input_ids, batch.positions, batch.slot_mapping)
                and plain(self.embed_tokens, nn.Embedding)    # its result is written to
                and not (torch.is_grad_enabled() and any(p.requires_grad for p in self.parameters()))):
            return False
        read = [self.embed_tokens.weight]
        for layer in self.layers:
            at, mlp = layer.self_attn, layer.mlp
            qkv, o = at.qkv_proj, at.o_proj
            if not (plain(layer, self.layer_cls) and plain(at, LlamaAttention) and plain(qkv, ColumnParallelLinear)
                    and plain(o, RowParallelLinear)):
                return False
            read += (qkv.weight, o.weight) if qkv.bias is None else (qkv.weight, o.weight, qkv.bias)
            if isinstance(mlp, LlamaMLP):
                up, down = mlp.gate_up_proj, mlp.down_proj
                if not (plain(mlp, LlamaMLP) and plain(up, ColumnParallelLinear) and plain(down, RowParallelLinear)
                        and up.bias is None):
                    return False
                read += (up.weight, down.weight)
        return ops.rows_weights_ok(read, input_ids)

    _unknown: Optional[torch.Tensor] = None

    def _unknown_ids(self) -> torch.Tensor:
        """The flag that a step sets for an id outside the vocabulary: pinned, so that the host reads it without a copy
        (a copied model's own is not)."""
        if self._unknown is None or not self._unknown.is_pinned():
            with torch.inference_mode(False):
                self._unknown = torch.zeros(1, dtype=torch.int32, device="cpu", pin_memory=True)
        return self._unknown

    def check_ids(self) -> None:
        """Raises if a step on the paged cache that has run had an id outside the vocabulary (its logits are NaN). It is
        known once the step's results have come to the host, and raised before a later step at the latest."""
        if self._unknown is not None and self._unknown.item():
            self._unknown.zero_()
            raise IndexError(f"a step had a token id outside the vocabulary of {self.embed_tokens.num_embeddings}")

    def _forward_rows(self, input_ids: torch.Tensor, batch: ForwardBatch) -> torch.Tensor:
        """A decode step or a short prompt: weights streamed by the few-row kernel, whose split sums go straight into the
        next row-wise kernel: 8 launches a layer, one more where gate/up is the library's. A prompt's fused projection stays
        whole: its attention reads the keys and values as rows."""
        layers, norm, once = self.layers, self.layers[0].input_layernorm, self._once
        T = input_ids.shape[0]
        if batch.mode == "decode":
            # zeroed by the first launch, and zero again after each layer's attention
            arrived = torch.empty(T * layers[0].self_attn.num_kv_heads * ops.ATTN_COUNTER_GAP, dtype=torch.int32,
                                  device=input_ids.device)
            x, residual = ops.embed_norm_rows(input_ids, self.embed_tokens.weight, norm.weight, norm.eps, self._unknown_ids(),
                                              arrived)
        else:              # a prompt's ids are the caller's: the embedding refuses them in the call
            residual = self.embed_tokens(input_ids)
            x = ops.rmsnorm(residual, norm.weight, norm.eps)
        for i, layer in enumerate(layers):
            at, norm = layer.self_attn, layer.post_attention_layernorm
            k_cache, v_cache, k_scale, v_scale = batch.kv_caches[at.layer_idx]
            if batch.mode == "prefill":
                att = at.attend(x, batch, self.cos_sin)
            else:
                q = ops.rope_store_rows(ops.linear_part(x, at.qkv_proj.weight, once), at.qkv_proj.bias, at.num_heads,
                                        batch.positions, self.cos_sin, k_cache, v_cache, batch.slot_mapping, k_scale, v_scale)
                att = at.attend_cache(q, batch, arrived)
            x = ops.add_norm_rows(ops.linear_part(att.view(T, -1), at.o_proj.weight, once), residual, norm.weight, norm.eps)
            norm = layers[i + 1].input_layernorm if i + 1 < len(layers) else self.norm
            mlp = layer.mlp
            if isinstance(mlp, LlamaMLP):
                w = mlp.gate_up_proj.weight
                act = (ops.linear_silu_rows(x, w, once) if self._silu_rows(T, w) or self._silu_streams(T, w) else mlp.activate(x))
                x = ops.add_norm_rows(ops.linear_part(act, mlp.down_proj.weight, once), residual, norm.weight, norm.eps)
            else:
                x, residual = ops.fused_add_rmsnorm(mlp(x), residual, norm.weight, norm.eps)
        return x

    def _planned(self, input_ids: torch.Tensor, batch: ForwardBatch) -> ForwardBatch:
        """The batch with this pass's attention plans, made once for all layers."""
        if not input_ids.is_cuda or ops._force_torch():
            return batch
        if batch.mode == "prefill":
            plan = ops.prefill_plan(batch.cu_seqlens.to(device=input_ids.device, dtype=torch.int32).contiguous(),
                                    input_ids.shape[0])
            return replace(batch, plans={**(batch.plans or {}), "prefill": plan})
        if (batch.host_segs is not None and batch.seg_tables is not None and self.dtype == torch.bfloat16
                and self.layers and self.layers[0].self_attn.head_dim == 128
                and ops.paged_prefill_pays(batch.host_segs, self.layers[0].self_attn.num_kv_heads)):
            at = self.layers[0].self_attn
            rows = 64 if ops.paged_prefill_few(batch.host_segs, at.num_heads) else 256
            plan, short = ops.paged_prefill_plan(batch.host_segs, input_ids.device, rows)
            if plan is not None:
                return replace(batch, plans={**(batch.plans or {}), "paged": (plan, short)})
        return batch

    def forward_hidden(self, input_ids: torch.Tensor, batch: ForwardBatch) -> torch.Tensor:
        self.check_ids()
        batch = self._planned(input_ids, batch)
        if self._takes_rows(input_ids, batch) or self._takes_short(input_ids, batch):
            return self._forward_rows(input_ids, batch)
        hidden = self.embed_tokens(input_ids)
        residual = None
        cos_sin = self.cos_sin
        for layer in self.layers:
            hidden, residual = layer(hidden, residual, batch, cos_sin)
        hidden, _ = ops.fused_add_rmsnorm(hidden, residual, self.norm.weight, self.norm.eps)
        return hidden

    def compute_logits(self, hidden: torch.Tensor) -> torch.Tensor:
        """fp32 [rows, V]."""
        out = ops.linear_f32(hidden, self.lm_head.weight, self._once) if self.lm_head.bias is None else None
        if out is not None:
            return out
        return self.lm_head(hidden).float()

    def forward_prefill(self, input_ids: torch.Tensor, batch: ForwardBatch) -> torch.Tensor:
        """Returns logits for the LAST token of each packed sequence: [n_seq, V]."""
        hidden = self.forward_hidden(input_ids, batch)
        last_idx = (batch.cu_seqlens[1:] - 1).long()
        return self.compute_logits(hidden[last_idx])

    def forward_decode(self, input_ids: torch.Tensor, batch: ForwardBatch) -> torch.Tensor:
        """One token per stream: [B] ids -> [B, V] logits."""
        hidden = self.forward_hidden(input_ids, batch)
        return self.compute_logits(hidden)

    def to_device(self, device) -> "LlamaForCausalLM":
        self.to(device)
        self.cos_sin = self.cos_sin.to(device)
        return self

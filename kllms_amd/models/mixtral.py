"""Mixtral MoE decoder for MI355X.

Same attention/backbone as Llama (GQA, RoPE, RMSNorm); the MLP is a
top-k-routed mixture of experts. Experts are TP-SHARDED, not
expert-parallel — every rank holds a 1/tp slice of every expert, so routing
needs no all-to-all and the layer keeps the dense model's two all-reduces.

On the GPU the experts run as grouped products over tokens bucketed by expert
(ops/hip/moe.hip), at every row count and without a host round trip, so that a
hipGraph replays them. Few rows that those kernels do not take (other types or
sizes, a gradient) run a DENSE batched GEMM over all experts.

Router semantics match Mixtral: softmax over ALL expert logits (fp32), top-k
(default 2), renormalize the selected weights.
"""

from __future__ import annotations

import torch
import torch.nn as nn

from .. import ops
from ..engine.config import ModelArchConfig
from ..parallel.tp import ParallelContext
from .llama import LlamaDecoderLayer, LlamaForCausalLM


class MixtralMoE(nn.Module):
    # TP sharding of the stacked expert tensors (dim scaled by tp at full
    # size); w_gate_up's dim 1 is the FUSED [gate; up] stack — 2 parts, each
    # sharded separately (matches weights.py's per-part expert sharding)
    shard_spec = {"w_gate_up": (1, 2), "w_down": 2}

    def __init__(self, cfg: ModelArchConfig, ctx: ParallelContext, dtype):
        super().__init__()
        assert cfg.num_experts > 0
        self.ctx = ctx
        tp = ctx.world_size
        assert cfg.intermediate_size % tp == 0
        self.E = cfg.num_experts
        self.k = cfg.num_experts_per_tok
        self.I = cfg.intermediate_size // tp
        H = cfg.hidden_size
        self.gate = nn.Linear(H, self.E, bias=False, dtype=dtype)
        self.gate.weight.requires_grad_(False)
        self.w_gate_up = nn.Parameter(torch.empty(self.E, 2 * self.I, H, dtype=dtype), requires_grad=False)
        self.w_down = nn.Parameter(torch.empty(self.E, H, self.I, dtype=dtype), requires_grad=False)

    def load_expert_(self, e: int, which: str, t: torch.Tensor) -> None:
        if which == "gate_up":
            self.w_gate_up.data[e].copy_(t.to(self.w_gate_up.dtype))
        else:
            self.w_down.data[e].copy_(t.to(self.w_down.dtype))

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        T, H = x.shape
        grouped = x.is_cuda and (T > 8 * self.E or self._takes_grouped(x))
        routed = None
        if self.gate.bias is None and ops.only_weights(self.gate, nn.Linear) and ops.no_global_hooks():
            routed = ops.router_top(x, self.gate.weight, self.k, grouped)
        if routed is not None:
            topw, topi = routed[:2]                                # [T, k]
        else:
            router_logits = self.gate(x).float()                   # [T, E]
            probs = torch.softmax(router_logits, dim=-1)
            topw, topi = torch.topk(probs, self.k, dim=-1)
            topw = topw / topw.sum(dim=-1, keepdim=True)

        if grouped:
            out = self._forward_grouped_hip(x, topw, topi, *(routed[2:] if routed else ()))
        elif T <= 8 * self.E:
            out = self._forward_dense(x, topw, topi)
        else:
            out = self._forward_grouped(x, topw, topi)
        return self.ctx.all_reduce(out)

    def _takes_grouped(self, x: torch.Tensor) -> bool:
        """Whether few rows run as the grouped products. They read the chosen experts alone, where a batched product reads all:
        us of the layer, 8 experts, top 2, and batched, at 1 / 5 / 16 / 64 rows: width 512, experts of 1024 41 124 / 42 141 /
        44 141 / 41 132; 2048, 8192 76 195 / 159 304 / 186 245 / 188 298; 4096, 14336 172 543 / 396 674 / 520 622 / 526 695"""
        gu, down = self.w_gate_up, self.w_down
        return (x.shape[0] >= 1 and self.E <= 4096 and x.dtype == gu.dtype == down.dtype == torch.bfloat16 and not ops._force_torch()
                and x.shape[1] % 64 == 0 and self.I % 64 == 0 and x.shape[1] < 1 << 24 and self.I < 1 << 24
                and x.is_contiguous() and gu.is_contiguous() and down.is_contiguous() and ops.plain_call(x, gu, down)
                and not (torch.is_grad_enabled() and (x.requires_grad or gu.requires_grad or down.requires_grad)))

    def _forward_dense(self, x: torch.Tensor, topw: torch.Tensor, topi: torch.Tensor) -> torch.Tensor:
        """Few tokens in batched GEMMs over all experts: no token bucketing, no
        data-dependent shapes. On the GPU the weights are the left operands: a
        batched bf16 product whose right operand is a transposed view has
        faulted there."""
        T = x.shape[0]
        if x.is_cuda:
            n = max(T, 2)                                       # a single column takes three times two's time
            xt = x.t().unsqueeze(0).expand(self.E, -1, n).contiguous()            # [E, H, n]
            gu2 = torch.bmm(self.w_gate_up, xt).transpose(1, 2).reshape(self.E * n, 2 * self.I)
            act = ops.silu_mul(gu2[:, : self.I], gu2[:, self.I:]).view(self.E, n, self.I)
            ye = torch.bmm(self.w_down, act.transpose(1, 2).contiguous())[:, :, :T].transpose(1, 2)      # [E, T, H]
        else:
            xb = x.unsqueeze(0).expand(self.E, T, -1)                             # [E, T, H]
            gu2 = torch.bmm(xb, self.w_gate_up.transpose(1, 2)).view(self.E * T, 2 * self.I)
            act = ops.silu_mul(gu2[:, : self.I], gu2[:, self.I:]).view(self.E, T, self.I)
            ye = torch.bmm(act, self.w_down.transpose(1, 2))                      # [E, T, H]
        # combine: weight[e, t] = topw where topi == e else 0
        w = torch.zeros(self.E, T, device=x.device, dtype=torch.float32)
        w.scatter_(0, topi.t().long(), topw.t().float())
        return (ye.float() * w.unsqueeze(-1)).sum(dim=0).to(x.dtype)

    def _forward_grouped_hip(self, x: torch.Tensor, topw: torch.Tensor, topi: torch.Tensor, ids=None, pos=None,
                             offsets=None, cleared=None) -> torch.Tensor:
        """The path on the GPU, three launches (ops/hip/moe.hip) behind the router's
        two, without a host round trip: gate/up GEMM with fused silu*mul, down GEMM,
        and the weighted sum of each token's rows. The pairs are sorted here where
        the router's kernel did not take the call."""
        T, H = x.shape
        if ids is None:
            ids, pos, offsets = ops.moe_sort(topi, self.E)
        act = torch.empty(T * self.k, self.I, device=x.device, dtype=x.dtype)
        y = torch.empty(T * self.k, H, device=x.device, dtype=x.dtype)
        ops.moe_gateup(act, x, self.w_gate_up, ids, offsets, x)     # every sorted place has a token: no zero rows
        ops.moe_down(y, act, self.w_down, offsets, cleared)
        return ops.moe_combine_rows(y, topw, pos)

    def _forward_grouped(self, x: torch.Tensor, topw: torch.Tensor, topi: torch.Tensor) -> torch.Tensor:
        """Prefill-shape path: tokens bucketed per expert, one GEMM group per
        expert (rocBLAS); avoids the dense path's E/k x FLOP overhead when
        T is large enough that compute, not weight streaming, dominates."""
        T = x.shape[0]
        out = torch.zeros_like(x)
        flat_exp = topi.reshape(-1)
        flat_tok = torch.arange(T, device=x.device).repeat_interleave(self.k)
        flat_w = topw.reshape(-1)
        for e in range(self.E):
            sel = (flat_exp == e).nonzero(as_tuple=True)[0]
            if sel.numel() == 0:
                continue
            toks = flat_tok[sel]
            xe = x[toks]
            gu = torch.nn.functional.linear(xe, self.w_gate_up[e])
            g, u = gu.split([self.I, self.I], dim=-1)
            ye = torch.nn.functional.linear(ops.silu_mul(g, u), self.w_down[e])
            out.index_add_(0, toks, ye * flat_w[sel].unsqueeze(-1).to(ye.dtype))
        return out


class MixtralDecoderLayer(LlamaDecoderLayer):
    def _make_mlp(self, cfg: ModelArchConfig, ctx: ParallelContext, dtype):
        return MixtralMoE(cfg, ctx, dtype)


class MixtralForCausalLM(LlamaForCausalLM):
    layer_cls = MixtralDecoderLayer

    def load_expert_(self, layer: int, e: int, which: str, t: torch.Tensor) -> None:
        self.layers[layer].mlp.load_expert_(e, which, t)

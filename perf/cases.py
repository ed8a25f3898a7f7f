"""Performance cases of the serving engine on one GPU.

Each case is a piece of work that a program serving requests with this
framework gives the GPU again and again: decode steps of a fanned-out batch,
packed prompt prefills, prompts that continue a cached prefix, sampling, the
routed feed-forward of a mixture-of-experts layer, and the two kinds of step of
a listed-layer hybrid. Models are the package's own 6-layer presets (layer
shapes of full models at reduced depth, random weights), built once per process
and kept, as a server keeps them; inputs come from the seed.

``kind`` of a case:

  decode   DecodeGraphRunner.run: one token for each of requests x fan streams
           whose prompt blocks are shared, replayed as a graph
  prefill  LlamaForCausalLM.forward_prefill: a packed batch of whole prompts
  resume   LLMEngine.step_segments: prompts whose head lies in the cache (a
           shared system prompt), only the tails are computed
  sample   ops.sample: one token per row of logits
  experts  MixtralMoE on a prompt batch's rows
  prompt   LLMEngine.step_segments of a hybrid model: fresh prompts
  step     LLMEngine.step_segments of a hybrid model: one token per stream
"""

from __future__ import annotations

import math
import random
from collections import OrderedDict

import numpy as np
import torch

from kllms_amd import ops
from kllms_amd.engine.config import MODEL_PRESETS, EngineConfig, ModelArchConfig
from kllms_amd.engine.engine import LLMEngine
from kllms_amd.engine.graph_runner import DecodeGraphRunner
from kllms_amd.engine.kvcache import PagedKVCache, SequenceKV
from kllms_amd.models.llama import ForwardBatch
from kllms_amd.models.mixtral import MixtralMoE
from kllms_amd.parallel.tp import ParallelContext

DEVICE = "cuda:0"
BLOCK = 16
F64 = torch.float64


def listed():
    return [
        # the smallest call: one plain chat stream of a small model, where launches and latency count
        dict(name="decode-1", kind="decode", model="llama-1b-l6", requests=1, fan=1, context=150, generated=20, fp8=False),
        # one consensus request alone on the server, n=5 over a 512-token prompt
        dict(name="decode-5", kind="decode", model="llama-8b-l6", requests=1, fan=5, context=512, generated=64, fp8=False),
        # the benchmark's batch: 24 requests of n=5
        dict(name="decode-120", kind="decode", model="llama-8b-l6", requests=24, fan=5, context=512, generated=64, fp8=False),
        # long documents, one answer each, with the fp8 cache
        dict(name="decode-long-fp8", kind="decode", model="llama-8b-l6", requests=16, fan=1, context=6000, generated=64, fp8=True),
        # admission of the benchmark's batch: 24 ragged prompts of about 512 tokens
        dict(name="prefill-24x512", kind="prefill", model="llama-8b-l6", prompts=24, tokens=512, ragged=True),
        # one long document, an odd length
        dict(name="prefill-1x7777", kind="prefill", model="llama-8b-l6", prompts=1, tokens=7777, ragged=False),
        # eight requests behind a system prompt that is already in the cache
        dict(name="resume-8", kind="resume", model="llama-8b-l6", prompts=8, prefix=1536, tokens=150),
        # token choice for the benchmark's batch at the full vocabulary, half of the rows with top-p and top-k
        dict(name="sample-120", kind="sample", rows=120, vocab=128256, truncated=0.5, masked=False),
        # schema-constrained rows (parse, n=16) of one request
        dict(name="sample-16-masked", kind="sample", rows=16, vocab=128256, truncated=0.0, masked=True),
        # one mixture layer (8 experts of 14336, top 2) over four prompts
        dict(name="experts-2048", kind="experts", rows=2048, hidden=4096, ff=14336, experts=8, top=2),
        # hybrid model: eight fresh prompts, and one token for each of 40 streams
        dict(name="hybrid-prompt-8x1000", kind="prompt", model="zutalix-1b-l6", prompts=8, tokens=1000),
        dict(name="hybrid-step-40", kind="step", model="zutalix-1b-l6", streams=40, context=600),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "resume", "sample", "experts", "prompt", "step"])
    model = rng.choice(["llama-1b-l6", "llama-8b-l6"])
    if kind == "decode":
        fan = rng.choice([1, 1, 3, 5, 8, 16])
        context = _log(rng, 24, 7800)
        most = max(1, min(250, 200_000 // (context + 64)) // fan)
        return dict(kind=kind, model=model, requests=_log(rng, 1, most), fan=fan, context=context,
                    generated=rng.randrange(1, 200), fp8=rng.random() < 0.25)
    if kind == "prefill":
        tokens = _log(rng, 20, 7900)
        return dict(kind=kind, model=model, prompts=_log(rng, 1, max(1, min(48, 12000 // tokens))), tokens=tokens,
                    ragged=rng.random() < 0.7)
    if kind == "resume":
        return dict(kind=kind, model=model, prompts=_log(rng, 1, 12), prefix=BLOCK * _log(rng, 8, 300),
                    tokens=_log(rng, 16, 512))
    if kind == "sample":
        return dict(kind=kind, rows=_log(rng, 1, 250), vocab=rng.choice([32000, 128256, 152064, 50257]),
                    truncated=rng.choice([0.0, 0.5, 1.0]), masked=rng.random() < 0.3)
    if kind == "experts":
        hidden, ff = rng.choice([(4096, 14336), (2048, 8192), (4096, 7168)])
        return dict(kind=kind, rows=_log(rng, 80, 6000), hidden=hidden, ff=ff, experts=8, top=2)
    if kind == "prompt":
        tokens = _log(rng, 40, 2000)
        return dict(kind=kind, model="zutalix-1b-l6", prompts=_log(rng, 1, max(1, min(16, 8000 // tokens))), tokens=tokens)
    return dict(kind=kind, model="zutalix-1b-l6", streams=_log(rng, 1, 120), context=_log(rng, 40, 900))


# --- what a server keeps ----------------------------------------------------------

_KEPT: "OrderedDict[tuple, object]" = OrderedDict()


def _keep(key, make):
    if key not in _KEPT:
        while len(_KEPT) >= 2:
            _KEPT.popitem(last=False)
        _KEPT[key] = make()
    _KEPT.move_to_end(key)
    return _KEPT[key]


def _engine(model: str, fp8: bool = False):
    """(engine, graph runner) of one model, weights from seed 0."""
    def make():
        eng = LLMEngine(EngineConfig(
            model=model, device=DEVICE, seed=0, use_hip_graphs=False, enable_prefix_caching=False,
            kv_cache_dtype="fp8_e4m3" if fp8 else "bf16", max_kv_blocks=64000, max_state_slots=640, eos_token_id=-1))
        runner = None if eng.stateful else DecodeGraphRunner(eng, eng.config.hip_graph_batch_sizes)
        return eng, runner
    return _keep(("engine", model, fp8), make)


def _mixture(case):
    def make():
        cfg = ModelArchConfig(arch="mixtral", vocab_size=32000, hidden_size=case["hidden"],
                              intermediate_size=case["ff"], num_layers=1, num_heads=32, num_kv_heads=8,
                              num_experts=case["experts"], num_experts_per_tok=case["top"])
        with torch.device(DEVICE):
            m = MixtralMoE(cfg, ParallelContext(), torch.bfloat16)
        g = torch.Generator(device=DEVICE).manual_seed(0)
        for p in m.parameters():
            for row in p.data.view(p.shape[0], -1):
                row.copy_(torch.randn(row.shape, generator=g, device=DEVICE) * 0.02)
        return m
    return _keep(("experts", case["hidden"], case["ff"], case["experts"], case["top"]), make)


class State:
    """Inputs of one case; gives its cache blocks back when it goes."""

    def __init__(self, **kw):
        self.seqs = []
        self.__dict__.update(kw)

    def __del__(self):
        for s in self.seqs:
            if s.blocks:
                self.engine.kv.free_sequence(s)


def _gen(seed: int, salt: int = 0):
    return torch.Generator(device=DEVICE).manual_seed(int(seed) * 1009 + salt)


def _lengths(n: int, mean: int, ragged: bool):
    """Prompt lengths around ``mean``, a quarter down or a fifth up where ragged (the same for every seed, as the
    outputs' shapes follow from them); room is left below the models' 8192 positions."""
    if not ragged:
        return [mean] * n
    r = random.Random(mean * 31 + n)
    return [max(1, min(7900, int(mean * r.uniform(0.75, 1.2)))) for _ in range(n)]


def _ids(n: int, vocab: int, g):
    return torch.randint(3, vocab, (n,), generator=g, device=DEVICE)


def _fill_cache(kv, blocks, std: float, seed: int):
    """Keys and values of earlier tokens, of the size that random weights give, written as the store writes them."""
    idx = torch.tensor(list(dict.fromkeys(blocks)), device=DEVICE)
    for layer in range(kv.num_layers):
        for which, (cache, scales) in enumerate(((kv.k_all, kv.k_scale_all), (kv.v_all, kv.v_scale_all))):
            g = _gen(seed, 17 + 2 * layer + which)
            x = (torch.randn((idx.numel(),) + tuple(cache.shape[2:]), generator=g, device=DEVICE) * std).bfloat16()
            if kv.fp8:
                s = (x.float().abs().amax(-1) / 448.0).clamp_min(1e-8)
                cache[layer].view(torch.uint8)[idx] = (x.float() / s.unsqueeze(-1)).to(cache.dtype).view(torch.uint8)
                scales[layer][idx] = s
            else:
                cache[layer][idx] = x


def _decode_streams(kv, case, seed):
    """Streams of fan-out over shared prompt blocks, each with some tokens of its own and room for one more."""
    r = random.Random(seed * 131 + 3)
    streams = []
    for n in _lengths(case["requests"], case["context"], True):
        parent = kv.alloc_sequence(n)
        for _ in range(case["fan"]):
            s = kv.fork(parent)
            kv.extend(s, r.randrange(case["generated"] // 2, case["generated"] + 1) + 1)
            streams.append(s)
        kv.free_sequence(parent)
    return streams


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    if kind == "sample":
        B, V = case["rows"], case["vocab"]
        # a peaked head over a flat rest, as a language model's rows look
        logits = torch.randn((B, V), generator=g, device=DEVICE) * 2.0
        hot = torch.randint(0, V, (B, 24), generator=g, device=DEVICE)
        logits.scatter_add_(1, hot, torch.rand((B, 24), generator=g, device=DEVICE) * 8.0)
        cut = torch.arange(B, device=DEVICE) < round(case["truncated"] * B)
        mask = None
        if case["masked"]:
            keep = torch.randint(-2**31, 2**31, (3, B, (V + 31) // 32), generator=g, device=DEVICE)
            mask = (keep[0] & keep[1] & keep[2]).to(torch.int32)
        return State(
            logits=logits, temps=torch.full((B,), 0.8, device=DEVICE),
            top_ps=torch.where(cut, 0.95, 1.0).float(), top_ks=torch.where(cut, 50, 0).int(),
            seeds=torch.randint(0, 2**40, (B,), generator=g, device=DEVICE),
            steps=torch.randint(0, 64, (B,), generator=g, device=DEVICE), mask=mask)
    if kind == "experts":
        return State(moe=_mixture(case), x=torch.randn((case["rows"], case["hidden"]), generator=g, device=DEVICE).bfloat16())
    eng, runner = _engine(case["model"], case.get("fp8", False))
    arch, kv = eng.arch, eng.kv
    std = 0.02 * math.sqrt(arch.hidden_size)
    if kind == "decode":
        seqs = _decode_streams(kv, case, seed)
        ctx = [s.num_tokens for s in seqs]
        width = max(len(s.blocks) for s in seqs) + 5
        bt = torch.zeros((len(seqs), width), dtype=torch.int32)
        for i, s in enumerate(seqs):
            bt[i, :len(s.blocks)] = torch.tensor(s.blocks, dtype=torch.int32)
        _fill_cache(kv, [b for s in seqs for b in s.blocks], std, seed)
        batch = ForwardBatch(
            mode="decode", positions=torch.tensor([c - 1 for c in ctx], device=DEVICE),
            slot_mapping=torch.tensor([s.blocks[(c - 1) // BLOCK] * BLOCK + (c - 1) % BLOCK for s, c in zip(seqs, ctx)],
                                      device=DEVICE),
            kv_caches=kv.layer_caches(), block_tables=bt.to(DEVICE),
            context_lens=torch.tensor(ctx, dtype=torch.int32, device=DEVICE))
        return State(engine=eng, runner=runner, seqs=seqs, batch=batch, ids=_ids(len(seqs), arch.vocab_size, g))
    if kind == "prefill":
        lens = _lengths(case["prompts"], case["tokens"], case["ragged"])
        own = PagedKVCache(arch.num_layers, arch.num_kv_heads, arch.head_dim_, BLOCK,
                           sum(-(-n // BLOCK) for n in lens), DEVICE, torch.bfloat16)
        slots = [x for n in lens for x in own.prefill_slot_mapping(own.alloc_sequence(n))]
        cu = np.concatenate([[0], np.cumsum(lens)])
        batch = ForwardBatch(
            mode="prefill", positions=torch.tensor([p for n in lens for p in range(n)], device=DEVICE),
            slot_mapping=torch.tensor(slots, device=DEVICE), kv_caches=own.layer_caches(),
            cu_seqlens=torch.tensor(cu, dtype=torch.int32, device=DEVICE))
        return State(engine=eng, kv=own, batch=batch, lens=lens, ids=_ids(sum(lens), arch.vocab_size, g))
    if kind == "resume":
        head = kv.alloc_sequence(case["prefix"])
        seqs = [kv.fork(head) for _ in range(case["prompts"])]
        kv.free_sequence(head)
        _fill_cache(kv, seqs[0].blocks, std, seed)
        lens = _lengths(case["prompts"], case["tokens"], True)
        toks = [_ids(n, arch.vocab_size, g).tolist() for n in lens]
        return State(engine=eng, seqs=seqs, toks=toks, start=case["prefix"])
    seqs = [eng.open_sequence() for _ in range(case["prompts"] if kind == "prompt" else case["streams"])]
    if kind == "prompt":
        lens = _lengths(case["prompts"], case["tokens"], True)
        return State(engine=eng, seqs=seqs, toks=[_ids(n, arch.vocab_size, g).tolist() for n in lens], start=0)
    n = case["context"]
    heads = [_ids(n, arch.vocab_size, g).tolist() for _ in seqs]
    for i in range(0, len(seqs), 8):
        eng.step_segments([(s, h, []) for s, h in zip(seqs[i:i + 8], heads[i:i + 8])])
    return State(engine=eng, seqs=seqs, toks=[_ids(1, arch.vocab_size, g).tolist() for _ in seqs], start=n, heads=heads)


@torch.inference_mode()
def run(s):
    if hasattr(s, "logits"):
        tokens, logprobs = ops.sample(s.logits, s.temps, s.top_ps, s.top_ks, s.seeds, s.steps, s.mask)
        return {"tokens": tokens, "logprobs": logprobs}
    if hasattr(s, "moe"):
        return s.moe(s.x)
    if hasattr(s, "runner"):
        return s.runner.run(s.ids, s.batch)
    if hasattr(s, "kv"):
        return {"logits": s.engine.model.forward_prefill(s.ids, s.batch), "k": s.kv.k_all, "v": s.kv.v_all}
    logits = s.engine.step_segments([(q, t, [len(t) - 1]) for q, t in zip(s.seqs, s.toks)])
    for q in s.seqs:
        q.num_tokens = s.start      # the next pass takes the same step again
    return logits


# --- what a pass cannot do without --------------------------------------------------

def _hybrid_weights(arch):
    """Weights of the layers of a hybrid preset (without embedding and head)."""
    W, n = arch.hidden_size, 0
    for layer in arch.layers:
        if layer.parallel is not None:
            le, ri = layer.parallel.left, layer.parallel.right
            n += W * (2 * le.heads * le.dim + le.kv_heads * le.dim + le.heads + 2 * ri.heads * ri.dim + 3 * ri.heads * ri.vdim)
        else:
            d = layer.channel_delta
            n += W * (2 * d.kv_heads * d.dim + 2 * d.heads * d.vdim + d.heads + d.decay_rank + d.gate_rank)
            n += d.heads * d.dim * d.decay_rank + d.heads * d.vdim * d.gate_rank
        if layer.mlp is not None:
            n += 3 * W * layer.mlp.ff
    return n


def work(case):
    kind = case["kind"]
    if kind == "sample":
        return {"bytes": case["rows"] * case["vocab"] * (4 + (1 / 8 if case["masked"] else 0)), "flops": 0}
    if kind == "experts":
        T, H, I, E = case["rows"], case["hidden"], case["ff"], case["experts"]
        return {"bytes": E * 3 * I * H * 2 + 4 * T * H, "flops": 2 * T * case["top"] * 3 * I * H}
    a = MODEL_PRESETS[case["model"]]
    W, V = a.hidden_size, a.vocab_size
    if kind in ("prompt", "step"):
        n = case["prompts"] * case["tokens"] if kind == "prompt" else case["streams"]
        outs = case["prompts"] if kind == "prompt" else n
        weights = _hybrid_weights(a)
        state = kvb = att = 0
        for layer in a.layers:
            for sp in (layer.parallel.right if layer.parallel else layer.channel_delta,):
                state += sp.heads * sp.dim * sp.vdim * 4 * outs * (1 if kind == "prompt" else 2)
                att += 6 * n * sp.heads * sp.dim * sp.vdim
            if layer.parallel:
                le = layer.parallel.left
                span = min(le.mask_size, case["tokens"]) / 2 if kind == "prompt" else min(le.mask_size, case["context"])
                kvb += 4 * le.kv_heads * le.dim * (n if kind == "prompt" else n * span)
                att += 4 * n * span * le.heads * le.dim
        return {"bytes": 2 * weights + 2 * V * W + state + kvb + 4 * outs * V, "flops": 2 * n * weights + 2 * outs * V * W + att}
    L, H, G, D = a.num_layers, a.num_heads, a.num_kv_heads, a.head_dim_
    layer_w = W * (H + 2 * G) * D + H * D * W + 3 * W * a.intermediate_size
    if kind == "decode":
        n = outs = case["requests"] * case["fan"]
        ctx = 0.975 * case["context"] + 0.75 * case["generated"]
        seen = n * ctx
        distinct = case["requests"] * 0.975 * case["context"] + n * 0.75 * case["generated"]
        kvb = distinct * 2 * G * D * ((1 + 4 / D) if case["fp8"] else 2)
    elif kind == "prefill":
        outs = case["prompts"]
        n = outs * case["tokens"] * (0.975 if case["ragged"] else 1)
        seen = n * n / outs / 2
        kvb = n * 4 * G * D
    else:
        outs = case["prompts"]
        n = outs * case["tokens"] * 0.975
        seen = n * (case["prefix"] + case["tokens"] / 2)
        kvb = (case["prefix"] + n) * 4 * G * D
    return {"bytes": L * (2 * layer_w + kvb) + 2 * V * W + 2 * n * W + 4 * outs * V,
            "flops": 2 * n * L * layer_w + 2 * outs * V * W + L * seen * H * D * 4}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        # fp32 logits: another order of the sums moves a log-probability by about 1e-7 of its size; a token changes
        # only where two perturbed logits or a top-p edge tie to fp32 rounding
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}
    if kind == "experts":
        # one layer in bf16 is 0.003 off 64 bits
        return {"rel": 0.012, "max": 0.2}
    if kind in ("prompt", "step"):
        # bf16 activations around an fp32 residual stream: 0.008 off 64 bits
        return {"rel": 0.025, "max": 0.5}
    # a bf16 residual stream through six layers: 0.02 off 64 bits, and 0.011 between two orders of the same keys
    return {"rel": 0.03, "max": 0.5}


# --- the same in 64 bits, in plain torch --------------------------------------------

def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _lin(x, w):
    return x @ w.to(F64).t()


def _causal(q, k, v, scale, first, span=None):
    """Rows ``first``.. of one sequence against its keys from position 0: q [T, H, D], k / v [L, G, D]; ``span``: the
    mask's aligned blocks."""
    T, H, _ = q.shape
    rep = H // k.shape[1]
    out = torch.empty((T, H, v.shape[2]), dtype=F64, device=q.device)
    j = torch.arange(k.shape[0], device=q.device)
    for r in range(0, T, 1024):
        i = torch.arange(first + r, first + min(T, r + 1024), device=q.device).unsqueeze(1)
        hide = j > i
        if span:
            hide = hide | (j // span != i // span)
        for h in range(H):
            s = (q[r:r + 1024, h] @ k[:, h // rep].t()) * scale
            out[r:r + 1024, h] = torch.softmax(s.masked_fill_(hide, -math.inf), -1) @ v[:, h // rep]
    return out


def _llama64(eng, ids, pos, spans, past, want):
    """Logits of the wanted rows, and every layer's new keys and values. spans: (first row, rows) of each sequence in
    ``ids``; past(layer, i): cached keys and values [P, G, D] of sequence i, or None."""
    a, m = eng.arch, eng.model
    H, G, D = a.num_heads, a.num_kv_heads, a.head_dim_
    inv = a.rope_theta ** (-torch.arange(0, D, 2, dtype=F64, device=DEVICE) / D)
    ang = pos.to(F64).unsqueeze(1) * inv
    cos, sin = ang.cos().unsqueeze(1), ang.sin().unsqueeze(1)

    def rope(x):
        u, w = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([u * cos - w * sin, w * cos + u * sin], -1)

    x = m.embed_tokens.weight[ids].to(F64)
    keys, values = [], []
    for li, layer in enumerate(m.layers):
        h = _rms(x, layer.input_layernorm.eps) * layer.input_layernorm.weight.to(F64)
        q, k, v = _lin(h, layer.self_attn.qkv_proj.weight).split([H * D, G * D, G * D], -1)
        q, k, v = rope(q.unflatten(1, (H, D))), rope(k.unflatten(1, (G, D))), v.unflatten(1, (G, D))
        keys.append(k)
        values.append(v)
        att = torch.empty_like(q)
        for i, (r, n) in enumerate(spans):
            kk, vv, old = k[r:r + n], v[r:r + n], past(li, i)
            if old is not None:
                kk, vv = torch.cat([old[0], kk]), torch.cat([old[1], vv])
            att[r:r + n] = _causal(q[r:r + n], kk, vv, 1 / math.sqrt(D), kk.shape[0] - n)
        x = x + _lin(att.flatten(1), layer.self_attn.o_proj.weight)
        h = _rms(x, layer.post_attention_layernorm.eps) * layer.post_attention_layernorm.weight.to(F64)
        gate, up = _lin(h, layer.mlp.gate_up_proj.weight).chunk(2, -1)
        x = x + _lin(torch.nn.functional.silu(gate) * up, layer.mlp.down_proj.weight)
    x = _rms(x[want], m.norm.eps) * m.norm.weight.to(F64)
    return _lin(x, m.lm_head.weight), keys, values


def _cached64(kv, seq, upto):
    def past(layer):
        idx = torch.tensor(seq.blocks[:-(-upto // BLOCK)], device=DEVICE)
        got = []
        for cache, scales in ((kv.k_all, kv.k_scale_all), (kv.v_all, kv.v_scale_all)):
            x = cache[layer][idx].to(F64)
            if kv.fp8:
                x = x * scales[layer][idx].to(F64).unsqueeze(-1)
            got.append(x.transpose(1, 2).flatten(0, 1)[:upto])
        return got
    return past


def _conv64(x, w):
    """Causal convolution of [B, T, C] with taps [C, K], the last one on the current row, then silu."""
    K = w.shape[1]
    x = torch.nn.functional.pad(x, (0, 0, K - 1, 0))
    y = sum(x[:, j:x.shape[1] - (K - 1 - j)] * w[:, j] for j in range(K))
    return torch.nn.functional.silu(y)


def _hybrid64(eng, rows, lens):
    """Logits of the last token of each prompt; rows: [B, T] ids, padded behind ``lens``."""
    a, w = eng.arch, eng.model.checkpoint_map()
    w = {k: v.to(F64) for k, v in w.items()}
    eps = eng.model.eps
    B, T = rows.shape
    silu = torch.nn.functional.silu
    x = _rms(w["embed"][rows], eps) * w["embed.norm"]
    for i, spec in enumerate(a.layers):
        p = f"l{i}."
        h = _rms(x, eps) * w[p + "norm1"]
        lin = lambda t, name: t @ w[p + "mix." + name].t()  # noqa: E731
        if spec.parallel is not None:
            le, ri = spec.parallel.left, spec.parallel.right
            q = (lin(h, "left.q") + w[p + "mix.left.q.b"]).unflatten(2, (le.heads, le.dim))
            k = (lin(h, "left.k") + w[p + "mix.left.k.b"]).unflatten(2, (le.kv_heads, le.dim))
            n = le.rot.dims
            ang = torch.arange(T, dtype=F64, device=DEVICE).unsqueeze(1) * (
                le.rot.base ** (-torch.arange(0, n, 2, dtype=F64, device=DEVICE) / n))
            c, s = ang.cos().unsqueeze(1), ang.sin().unsqueeze(1)

            def rot(t):
                u, v = t[..., 0:n:2], t[..., 1:n:2]
                return torch.cat([torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2), t[..., n:]], -1)

            left = torch.stack([_causal(rot(q)[b], rot(k)[b], k[b], le.scale, 0, le.mask_size) for b in range(B)])
            left = lin((left * torch.sigmoid(lin(h, "left.g")).unsqueeze(-1)).flatten(2), "left.o")
            q, k, v = (silu(lin(h, "right." + m)).unflatten(2, (ri.heads, -1)) for m in "qkv")
            decay = torch.tensor(ri.decay, dtype=F64, device=DEVICE).view(1, -1, 1, 1)
            S = torch.zeros((B, ri.heads, ri.dim, ri.vdim), dtype=F64, device=DEVICE)
            o = torch.empty((B, T, ri.heads, ri.vdim), dtype=F64, device=DEVICE)
            for t in range(T):
                S = S * decay + k[:, t].unsqueeze(-1) * v[:, t].unsqueeze(-2)
                o[:, t] = (q[:, t].unsqueeze(-2) @ S).squeeze(-2)
            right = _rms(o.flatten(2), eps) * w[p + "mix.right.norm"] * torch.sigmoid(lin(h, "right.g"))
            right = lin(right, "right.o")
            y = (_rms(left, eps) * w[p + "mix.left.out"] + _rms(right, eps) * w[p + "mix.right.out"]) / 2
        else:
            d = spec.channel_delta
            rep = d.heads // d.kv_heads
            q, k, v = (_conv64(lin(h, m), w[p + "mix." + m + ".conv"]).unflatten(2, (-1, n))
                       for m, n in (("q", d.dim), ("k", d.dim), ("v", d.vdim)))
            unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
            q, k = unit(q) * d.dim ** -0.5, unit(k)
            q, k = q.repeat_interleave(rep, 2), k.repeat_interleave(rep, 2)
            beta = torch.sigmoid(lin(h, "b"))
            f = (lin(lin(h, "a1"), "a2") + w[p + "mix.dt_bias"]).unflatten(2, (d.heads, d.dim))
            decay = torch.exp(-torch.exp(w[p + "mix.A_log"]).view(1, 1, -1, 1) * torch.nn.functional.softplus(f))
            S = torch.zeros((B, d.heads, d.dim, d.vdim), dtype=F64, device=DEVICE)
            o = torch.empty((B, T, d.heads, d.vdim), dtype=F64, device=DEVICE)
            for t in range(T):
                S = S * decay[:, t].unsqueeze(-1)
                u = beta[:, t].unsqueeze(-1) * (v[:, t] - (k[:, t].unsqueeze(-2) @ S).squeeze(-2))
                S = S + k[:, t].unsqueeze(-1) * u.unsqueeze(-2)
                o[:, t] = (q[:, t].unsqueeze(-2) @ S).squeeze(-2)
            y = lin((_rms(o, eps) * w[p + "mix.norm"]).flatten(2) * torch.sigmoid(lin(lin(h, "g1"), "g2")), "o")
        x = x + _rms(y, eps) * w[p + "norm1b"]
        if spec.mlp is not None:
            h = _rms(x, eps) * w[p + "norm2"]
            g = torch.clamp(h @ w[p + "mlp.gate"].t(), max=spec.mlp.limit)
            u = torch.clamp(h @ w[p + "mlp.up"].t(), -spec.mlp.limit, spec.mlp.limit)
            y = (g * torch.sigmoid(spec.mlp.alpha * g) * (u + 1)) @ w[p + "mlp.down"].t()
            x = x + _rms(y, eps) * w[p + "norm2b"]
    last = x[torch.arange(B, device=DEVICE), torch.tensor(lens, device=DEVICE) - 1]
    return (_rms(last, eps) * w["final.norm"]) @ w["head"].t()


def _splitmix(x):
    with np.errstate(over="ignore"):
        x = x + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return x ^ (x >> np.uint64(31))


def _sample64(s):
    """Log-probabilities of the tokens that the counter-based draw picks, with the draw done in 64 bits."""
    x = s.logits.to(F64)
    B, V = x.shape
    if s.mask is not None:
        at = torch.arange(V, device=DEVICE)
        allowed = (s.mask[:, at // 32] >> (at % 32)) & 1
        x = x.masked_fill(allowed == 0, -math.inf)
    lp = x - torch.logsumexp(x, -1, keepdim=True)
    scaled = x / s.temps.to(F64).unsqueeze(1)
    top, order = scaled.sort(-1, descending=True)
    mass = torch.softmax(top, -1)
    before = mass.cumsum(-1) - mass
    k = torch.where(s.top_ks > 0, s.top_ks, V).unsqueeze(1)
    keep = (before < s.top_ps.to(F64).unsqueeze(1)) & (torch.arange(V, device=DEVICE) < k)
    scaled = scaled.masked_fill(~torch.zeros_like(keep).scatter_(1, order, keep), -math.inf)
    at, got = np.arange(V, dtype=np.uint64), []
    with np.errstate(over="ignore"):
        base = _splitmix(s.seeds.cpu().numpy().astype(np.uint64) * np.uint64(0x9E3779B97F4A7C15)
                         + s.steps.cpu().numpy().astype(np.uint64) * np.uint64(0xBF58476D1CE4E5B9))
    for b in range(B):
        u = ((_splitmix(base[b] ^ at) >> np.uint64(40)) + np.uint64(1)).astype(np.float32) * np.float32(1 / 16777217.0)
        u = torch.from_numpy(u).to(DEVICE).to(F64)
        pick = int((scaled[b] - torch.log(-torch.log(u))).argmax())
        got.append(lp[b, pick])
    return torch.stack(got)


@torch.inference_mode()
def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "sample":
        return {"tokens": None, "logprobs": _sample64(s)}
    if kind == "experts":
        # the choice of experts follows the router's logits as its 16-bit layer gives them
        x, m = s.x.to(F64), s.moe
        probs = torch.softmax(_lin(x, m.gate.weight).bfloat16().to(F64), -1)
        w, e = probs.topk(case["top"], -1)
        w = w / w.sum(-1, keepdim=True)
        out = torch.zeros_like(x)
        for i in range(case["experts"]):
            r, c = (e == i).nonzero(as_tuple=True)
            gate, up = _lin(x[r], m.w_gate_up[i]).chunk(2, -1)
            out[r] += w[r, c].unsqueeze(1) * _lin(torch.nn.functional.silu(gate) * up, m.w_down[i])
        return out
    eng = s.engine
    if kind in ("prompt", "step"):
        full = [(h if kind == "step" else []) + t for h, t in zip(getattr(s, "heads", s.toks), s.toks)]
        lens = [len(t) for t in full]
        rows = torch.tensor([t + [0] * (max(lens) - len(t)) for t in full], device=DEVICE)
        return torch.cat([_hybrid64(eng, rows[i:i + 16], lens[i:i + 16]) for i in range(0, len(lens), 16)])
    if kind == "decode":
        past = [_cached64(eng.kv, q, q.num_tokens - 1) for q in s.seqs]
        n = len(s.seqs)
        return _llama64(eng, s.ids, s.batch.positions, [(i, 1) for i in range(n)], lambda layer, i: past[i](layer),
                        slice(None))[0]
    if kind == "prefill":
        cu = np.cumsum([0] + s.lens)
        logits, keys, values = _llama64(eng, s.ids, s.batch.positions, list(zip(cu, s.lens)), lambda layer, i: None,
                                        torch.tensor(cu[1:] - 1, device=DEVICE))
        slots = s.batch.slot_mapping
        out = {"logits": logits}
        for name, rows in (("k", keys), ("v", values)):
            t = torch.zeros(s.kv.k_all.shape, dtype=F64, device=DEVICE)
            for layer, x in enumerate(rows):
                t[layer, slots // BLOCK, :, slots % BLOCK] = x
            out[name] = t
        return out
    lens = [len(t) for t in s.toks]
    cu = np.cumsum([0] + lens)
    ids = torch.tensor([t for part in s.toks for t in part], device=DEVICE)
    pos = torch.tensor([s.start + i for n in lens for i in range(n)], device=DEVICE)
    past = _cached64(eng.kv, SequenceKV(blocks=s.seqs[0].blocks[:s.start // BLOCK]), s.start)
    return _llama64(eng, ids, pos, list(zip(cu, lens)), lambda layer, i: past(layer),
                    torch.tensor(cu[1:] - 1, device=DEVICE))[0]

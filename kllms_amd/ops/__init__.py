"""Op dispatch: HIP/CDNA4 kernels on GPU, torch reference on CPU.

Policy: on a GPU (`tensor.is_cuda`, which on
PyTorch-ROCm means an AMD GPU) the hand-written gfx950 HIP kernels in
``kllms_amd._C`` are the ONLY path — if the extension is missing the op
RAISES instead of silently falling back to eager PyTorch. On CPU the pure
torch reference implementations (torch_ref.py) run, which is what the
GPU-less CI environment uses.

Set ``KLLMS_AMD_FORCE_TORCH_OPS=1`` to force the torch path on GPU (used only
by numerics tests to produce the oracle on-device).
"""

from __future__ import annotations

import heapq
import os
from typing import NamedTuple, Optional, Sequence, Tuple

import torch

from . import torch_ref

_C = None
_C_err: Optional[str] = None
try:
    from kllms_amd import _C  # type: ignore[no-redef]  # built by setup.py build_ext --inplace
except Exception as e:  # pragma: no cover - import-time probe
    _C = None
    _C_err = str(e)


def hip_available() -> bool:
    return _C is not None


def _force_torch() -> bool:
    return os.environ.get("KLLMS_AMD_FORCE_TORCH_OPS", "0") == "1"


def _hip_or_raise():
    if _C is None:
        raise RuntimeError(
            "kllms_amd HIP extension (kllms_amd/_C*.so) is not built but a GPU "
            "tensor was passed. Build it with `python setup.py build_ext --inplace` "
            f"(PYTORCH_ROCM_ARCH=gfx950). Import error: {_C_err}"
        )
    return _C


def upload(t: torch.Tensor, device) -> torch.Tensor:
    """A host tensor on the device. To a GPU by way of pinned memory, whose copy waits in the stream like a launch: one
    from pageable memory holds the host until all work before it is done (8 prompt tails behind a cached prefix, built
    while the GPU works on the last ones: 3.92 ms with such copies, 3.82 without; a hybrid step of 40 rows 780 us and 699). The pinned block is the caching host
    allocator's, which keeps it until the copy is through."""
    if torch.device(device).type != "cuda" or t.numel() == 0:
        return t.to(device)
    return t.pin_memory().to(device, non_blocking=True)


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    if x.is_cuda and not _force_torch():
        out = torch.empty_like(x)
        _hip_or_raise().rmsnorm(out, x, weight, eps)
        return out
    return torch_ref.rmsnorm(x, weight, eps)


def fused_add_rmsnorm(
    x: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, eps: float
) -> Tuple[torch.Tensor, torch.Tensor]:
    if x.is_cuda and not _force_torch():
        # in-place: residual += x; x_out = rmsnorm(residual)
        out = torch.empty_like(x)
        _hip_or_raise().fused_add_rmsnorm(out, x, residual, weight, eps)
        return out, residual
    return torch_ref.fused_add_rmsnorm(x, residual, weight, eps)


def rope_inplace(q: torch.Tensor, k: torch.Tensor, positions: torch.Tensor, cos_sin: torch.Tensor) -> None:
    if q.is_cuda and not _force_torch():
        _hip_or_raise().rope_inplace(q, k, positions, cos_sin)
        return
    torch_ref.rope_inplace(q, k, positions, cos_sin)


def silu_mul(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    if gate.is_cuda and not _force_torch():
        out = torch.empty(gate.shape, dtype=gate.dtype, device=gate.device)
        _hip_or_raise().silu_mul(out, gate, up)
        return out
    return torch_ref.silu_mul(gate, up)


def store_kv(
    k: torch.Tensor,
    v: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    slot_mapping: torch.Tensor,
    k_scale: Optional[torch.Tensor] = None,
    v_scale: Optional[torch.Tensor] = None,
) -> None:
    """k_scale/v_scale: [NB, KVH, BS] fp32 per-row dequant scales, REQUIRED
    when the caches are fp8 (written here: s = amax(|row|)/448), None for bf16."""
    if k.is_cuda and not _force_torch():
        none = _none(k, torch.float32)
        _hip_or_raise().store_kv(
            k, v, k_cache, v_cache, slot_mapping,
            k_scale if k_scale is not None else none,
            v_scale if v_scale is not None else none)
        return
    torch_ref.store_kv(k, v, k_cache, v_cache, slot_mapping, k_scale, v_scale)


def rope_store(q, k, v, positions, cos_sin, k_cache, v_cache, slot_mapping, k_scale=None, v_scale=None) -> None:
    """rope_inplace(q, k) and store_kv(k, v): one launch for aligned rows of head size 128, else the two."""
    if (q.is_cuda and not _force_torch() and q.dtype == k.dtype == v.dtype == torch.bfloat16
            and q.shape[2] == 128 and k.stride(0) == v.stride(0)
            and all(t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0 and t.stride(2) == 1 and t.stride(1) == 128
                    for t in (q, k, v))
            and all(t.dtype == torch.long and t.is_contiguous() and t.dim() == 1 for t in (positions, slot_mapping))
            and cos_sin.is_contiguous() and k_cache.dtype == v_cache.dtype):
        none = _none(k, torch.float32)
        if positions.shape[0] != q.shape[0] or slot_mapping.shape[0] != q.shape[0]:      # the rows at their head
            positions, slot_mapping = positions[:q.shape[0]], slot_mapping[:q.shape[0]]
        _hip_or_raise().rope_store(q, k, v, positions, cos_sin, k_cache, v_cache, slot_mapping,
                                   k_scale if k_scale is not None else none, v_scale if v_scale is not None else none)
        return
    rope_inplace(q, k, positions, cos_sin)
    store_kv(k, v, k_cache, v_cache, slot_mapping, k_scale, v_scale)


def prefill_plan(cu_seqlens: torch.Tensor, rows: int) -> Optional[torch.Tensor]:
    """Row groups of packed sequences for attn_prefill_varlen, made on the GPU (None on the CPU): one launch serves
    every layer of a forward pass."""
    if cu_seqlens.is_cuda and not _force_torch():
        return _hip_or_raise().attn_prefill_plan(cu_seqlens, rows)
    return None


def attn_prefill_varlen(
    q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cu_seqlens: torch.Tensor, scale: float,
    plan: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    if q.is_cuda and not _force_torch():
        out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        if plan is None:
            plan = prefill_plan(cu_seqlens.to(device=q.device, dtype=torch.int32).contiguous(), q.shape[0])
        _hip_or_raise().attn_prefill(out, q, k, v, plan, scale)
        return out
    return torch_ref.attn_prefill_varlen(q, k, v, cu_seqlens, scale)


# segments shorter than this attend row by row: a workgroup of the paged prefill kernel has eight 32-row tiles. Around
# the line, 12 segments behind 3000 keys (32 heads, 8 kv heads), paged 190 us; row by row 169 for 16 rows each, 248 for 24,
# 327 for 31
PAGED_PREFILL_ROWS = 32
# A group of up to 256 rows is one workgroup a head, so a step of few groups takes as long as its longest group's keys,
# one tile after another: 30 ns a key up to 160 rows, 50 above. Row by row every compute unit is busy, 0.03 to 0.05 ns for
# each row, key and kv head. So the rows have to make 750 row-heads of the longest segment's keys. 32 heads, 8 kv heads, one
# segment behind 6000 keys: 32 rows 184 us paged, 68 row by row; 64 rows 188, 123; 128 rows 189, 227; four of 32 rows
# 181, 239. 4 kv heads: 64 rows 188, 93; 256 rows 299, 282; two of 128 193, 286. 32 kv heads, 32 rows behind 3000: 100, 116.
PAGED_PREFILL_WORK = 750


def paged_prefill_pays(segs, kv_heads: int) -> bool:
    """Whether the long ones of the segments [(start position, rows)] attend together (paged_prefill_plan) or row by
    row like the short ones."""
    long = [(start + n, n) for start, n in segs if n >= PAGED_PREFILL_ROWS]
    return bool(long) and kv_heads * sum(k * n for k, n in long) >= PAGED_PREFILL_WORK * max(k for k, _ in long)


# us of a workgroup that goes over k keys: four waves to a row tile and 64 rows a workgroup; one wave to a row tile and up to
# 128 rows, and up to 256, where a SIMD has two of them. Measured, one segment, at 512 / 1536 / 4000 keys: 20, 36, 76; 26, 55,
# 127; 41, 86, 199.
_PAGED_GROUP = {64: (12, 1 / 63), 128: (11, 1 / 34), 256: (16, 1 / 22)}


def paged_prefill_few(segs, heads: int) -> bool:
    """Whether the long ones of the segments [(start position, rows)] are dealt out in groups of 64 rows, whose four waves
    share each row tile's keys (their sums take 2 us to meet), and not of 256. Few segments leave the chip idle otherwise; with
    many, the keys are staged four times as often. 32 / 8 heads, us, groups of 256 and of 64:
      behind 512    1 segment of 64 rows 24, 19   146 37, 20   512 53, 28     4 of 146 37, 34   300 44, 59     8 of 146 40, 52
      behind 1536   1 of 64 52, 34   146 82, 36   512 98, 47     2 of 300 87, 70     4 of 146 83, 63   256 88, 82     8 of 65 56, 62
        146 88, 99    12 of 64 103, 70   96 106, 95
      behind 4000   1 of 146 190, 76     4 of 256 203, 166     8 of 146 197, 212    12 of 128 259, 240
    One of 33 rows behind 5, whatever the rule says of it: 6.5, 9.4."""
    long = [(start + n, n) for start, n in segs if n >= PAGED_PREFILL_ROWS]
    if max((k for k, _ in long), default=0) < 512:
        return False

    def cost(size):
        """Of all groups, longest first, on as many at a time as compute units have their heads."""
        groups = []
        for k, n in long:
            for r in range(0, n, size):
                rows = min(size, n - r)
                at, key = _PAGED_GROUP[64 if size == 64 else 128 if rows <= 128 else 256]
                groups.append(at + (k - n + r + rows) * key)
        lanes = [0.0] * max(1, 256 // heads)
        for us in sorted(groups, reverse=True):
            heapq.heapreplace(lanes, lanes[0] + us)
        return max(lanes)

    return cost(64) < cost(256)


class PagedGroups(NamedTuple):
    """Groups of up to ``rows`` (64 or 256) rows of segments, [4, G] on the device: the kernel is the one of that size."""
    groups: torch.Tensor
    rows: int


def paged_prefill_plan(segs, device, rows: int = 256) -> tuple:
    """(PagedGroups, [(first row, rows)] left to row-by-row attention) for segments [(start position, rows)] packed in that
    order; None for the groups when every segment is short."""
    groups, short, row = [], [], 0
    for i, (_, n) in enumerate(segs):
        if n >= PAGED_PREFILL_ROWS:
            groups.extend((row, n, r, i) for r in range(0, n, rows))
        elif n and short and short[-1][0] + short[-1][1] == row:
            short[-1] = (short[-1][0], short[-1][1] + n)
        elif n:
            short.append((row, n))
        row += n
    # the groups that see most first
    groups.sort(key=lambda g: -(segs[g[3]][0] + g[2]))
    if not groups:
        return None, short
    return PagedGroups(upload(torch.tensor(groups, dtype=torch.int32).t().contiguous(), device), rows), short


def attn_segments_paged(q, k_cache, v_cache, block_tables, context_lens, scale, plan, short, seg_tables, seg_start):
    """Rows of long segments on the matrix cores against the paged bf16 cache, the others row by row (GPU only)."""
    out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
    _hip_or_raise().attn_prefill_paged(out, q, k_cache, v_cache, plan.groups, seg_tables, seg_start, scale, plan.rows)
    f = _none(q, torch.float32)
    for r, n in short:
        _hip_or_raise().attn_decode_paged(out[r:r + n], q[r:r + n], k_cache, v_cache, block_tables[r:r + n],
                                          context_lens[r:r + n], scale, f, f, f)
    return out


def blocklocal_rows_ok(q, k_cache, v_cache, gate) -> bool:
    """Whether attn_blocklocal_rows takes a step: bf16, head sizes of 128, a group size the decode kernel has."""
    return (_gpu(q) and q.dtype == torch.bfloat16 and k_cache.dtype == torch.bfloat16 and q.shape[2] == 128
            and k_cache.shape[3] == 128 and v_cache.shape[3] == 128 and q.shape[1] // k_cache.shape[1] in (1, 2, 4, 8)
            and q.shape[1] % k_cache.shape[1] == 0 and (gate is None or gate.dtype == torch.bfloat16)
            and q.stride(2) == 1 and q.stride(1) == 128)


def attn_blocklocal_rows(q, k_cache, v_cache, block_tables, context_lens, scale, mask_size, gate=None):
    """Single decoded rows of the block-local mask (0: plain causal), per-head gate: row i against table row i."""
    out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
    f = _none(q, torch.float32)
    _hip_or_raise().attn_decode_paged(out, q, k_cache, v_cache, block_tables, context_lens, scale, f, f,
                                      gate if gate is not None else f, int(mask_size))
    return out


# 32 ints, a line of the L2: workgroups that count in one line wait for each other. One stream of 2000 keys, 32 / 8 heads,
# 128 workgroups: 9.7 us with the eight counters beside each other, 8.9 with this between them; two 11.1, 9.3
ATTN_COUNTER_GAP = 32


def attn_decode_paged(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    block_tables: torch.Tensor,
    context_lens: torch.Tensor,
    scale: float,
    k_scale: Optional[torch.Tensor] = None,
    v_scale: Optional[torch.Tensor] = None,
    arrived: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """``arrived``: an int32 zero for each row and kv head, zero again afterwards; with it, contexts that several workgroups
    share are merged in the same launch. Zeros for ATTN_COUNTER_GAP times as many keep the counters in cache lines of their own."""
    if q.is_cuda and not _force_torch():
        out = torch.empty(q.shape, dtype=q.dtype, device=q.device)
        none = _none(q, torch.float32)
        _hip_or_raise().attn_decode_paged(
            out, q, k_cache, v_cache, block_tables, context_lens, scale,
            k_scale if k_scale is not None else none,
            v_scale if v_scale is not None else none, none, -1, arrived)
        return out
    return torch_ref.attn_decode_paged(q, k_cache, v_cache, block_tables, context_lens, scale,
                                       k_scale, v_scale)


# --- products of a few rows (decode steps) ----------------------------------------
# GPU-only: callers ask linear_rows_ok first and keep F.linear for everything else.

LINEAR_ROWS_MAX = 128
LINEAR_PART_MAX = 384      # of linear_part
LINEAR_SILU_MAX = 256      # of linear_silu_rows


def linear_rows_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether the few-row kernel takes x [M, K] @ w [N, K]^T: bf16 on the GPU, rows and sizes that its 16-byte loads
    and 128-deep chunks divide."""
    return (x.is_cuda and not _force_torch() and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.dim() == 2
            and 1 <= x.shape[0] <= LINEAR_ROWS_MAX and x.shape[1] % 128 == 0 and w.shape[0] % 16 == 0
            and x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0
            and w.is_contiguous() and w.data_ptr() % 16 == 0
            and not (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad)))


def rows_weights_ok(ws: Sequence[torch.Tensor], like: torch.Tensor) -> bool:
    """Whether the few-row kernels read all of these: plain bf16 tensors on ``like``'s device, contiguous, on 16 bytes."""
    return all(type(w) in _PLAIN for w in ws) and _hip_or_raise().rows_weights_ok(ws, like)


WEIGHTS_ONCE_BYTES = 320 << 20


def weights_once(model: torch.nn.Module) -> bool:
    """``once`` of the few-row products in a model's steps: whether the matrices that every step reads are too many to stay in
    the 256 MB last-level cache until the next one. Tables, of which a step reads rows, and stacks of experts, of which it
    reads some, do not count: without them it is a model whose steps hit nothing for certain."""
    return sum(p.numel() * p.element_size() for m in model.modules() if not isinstance(m, torch.nn.Embedding)
               for p in m.parameters(recurse=False) if p.dim() == 2) >= WEIGHTS_ONCE_BYTES


def linear_part(x: torch.Tensor, w: torch.Tensor, once: bool = False) -> torch.Tensor:
    """fp32 sums [S, M, N] of x @ w^T over S shares of K; the consumer adds them up."""
    return _hip_or_raise().linear_rows(x, w, _none(x), 0, 0, once)


def linear_silu_rows(x: torch.Tensor, w: torch.Tensor, once: bool = False) -> torch.Tensor:
    """silu(gate) * up of a fused [gate; up] matrix, bf16."""
    return _hip_or_raise().linear_rows(x, w, _none(x), 3, 1, once)


def linear_f32_rows(x: torch.Tensor, w: torch.Tensor, once: bool = False) -> torch.Tensor:
    """fp32 x @ w^T without a rounding to bf16 (logits)."""
    return _hip_or_raise().linear_rows(x, w, _none(x), 2, 1, once)


def linear_f32(x: torch.Tensor, w: torch.Tensor, once: bool = False) -> Optional[torch.Tensor]:
    """fp32 x @ w^T from the fp32 sums of the bf16 product at every row count (rounded to bf16 at some counts only, near ties
    between tokens would fall differently as a stream's batch grows); None where that is not to be had: not bf16 on the GPU,
    or wanted for a gradient."""
    if not (x.dim() == 2 and x.is_cuda and x.dtype == w.dtype == torch.bfloat16 and not _force_torch()
            and not (torch.is_grad_enabled() and (x.requires_grad or w.requires_grad))):
        return None
    # us, the library and the few-row kernel, weights out of cache, at 1 / 32 / 64 / 96 / 128 rows:
    #   32000 x 4096   61 49 / 60 51 / 61 52 / 62 55 / 64 60        128256 x 2048  114 94 / 122 106 / 127 117 / 137 131 / 139 143
    #   128256 x 4096  188 177 / 209 197 / 223 207 / 239 222 / 250 244
    #   152064 x 3584  230 193 / 263 211 / 224 225 / 240 253 / 255 279
    K = w.shape[1]
    most = 64 if K & (K - 1) else 128 if K >= 4096 else 96
    if x.shape[0] <= most and linear_rows_ok(x, w):
        return linear_f32_rows(x, w, once)
    return torch.mm(x, w.t(), out_dtype=torch.float32)


# --- products of many rows (prompts) ----------------------------------------------

_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _plain_call(*ts: torch.Tensor) -> bool:
    """Whether nothing but the values of these tensors is wanted: no transform, tracer or tensor subclass looks on."""
    return (all(type(t) in _PLAIN for t in ts) and torch.autograd.forward_ad._current_level < 0
            and not torch._C._len_torch_function_stack()
            and not torch._C._are_functorch_transforms_active() and not torch.jit.is_tracing()
            and not torch.compiler.is_compiling() and not torch._C._len_torch_dispatch_stack())


def plain_call(*ts: torch.Tensor) -> bool:
    """_plain_call without autocast, under which the library's products have its type."""
    return _plain_call(*ts) and not torch.is_autocast_enabled("cuda")


def only_weights(module: torch.nn.Module, kind: type) -> bool:
    """Whether a call of ``module`` is ``kind``'s forward and nothing else: the class itself, no hooks on it, no forward of
    the object's own. Asked before a fused call takes a module's weights and passes the module by; hooks on all modules
    are no_global_hooks()."""
    d = module.__dict__
    return type(module) is kind and "forward" not in d and not (
        d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"])


def no_global_hooks() -> bool:
    return not torch.nn.modules.module._has_any_global_hook()


def _try_tiles(x, w, bias, act: int, limit: float = 0.0, alpha: float = 0.0) -> Optional[torch.Tensor]:
    """The product on the tile kernel, where it takes the call (bf16 on the GPU, more than 128 rows, contiguous, sizes that
    its 16-byte accesses and 64-deep stages divide, no gradient or transform to serve) and is the faster one. Subclasses,
    function modes and the compiler see the library's product, as at every other row count."""
    if (x.is_cuda and x.dim() == 2 and x.shape[0] > 128 and not torch.compiler.is_compiling()
            and type(x) in _PLAIN and type(w) in _PLAIN and (bias is None or type(bias) in _PLAIN)
            and not torch._C._len_torch_function_stack() and not _force_torch()):
        return _hip_or_raise().linear_tiles_try(x, w, bias, act, limit, alpha)
    return None


def linear(x: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x @ w^T + bias: prompts on the tile kernel where that is the faster one, everything else in the library."""
    y = _try_tiles(x, w, bias, 0)
    return y if y is not None else torch.nn.functional.linear(x, w, bias)


def linear_silu(x: torch.Tensor, w: torch.Tensor) -> Optional[torch.Tensor]:
    """silu(gate) * up of a fused [gate; up] matrix for prompts, or None where the tile kernel does not take it."""
    return _try_tiles(x, w, None, 1)


def linear_clamped_glu(x: torch.Tensor, w: torch.Tensor, limit: float, alpha: float) -> Optional[torch.Tensor]:
    """clamped_glu of a fused [gate; up] matrix for prompts, or None where the tile kernel does not take it."""
    return _try_tiles(x, w, None, 2, limit, alpha)


def embed_norm_rows(ids, table, weight, eps, unknown=None, clear=None):
    """(rms(table[ids]) * weight, table[ids]). An id outside the table gives a row of NaN and sets ``unknown``, one int32
    of pinned host memory, to 1. ``clear``: int32 values on the GPU that the launch zeroes."""
    return _hip_or_raise().embed_norm_rows(ids, table, weight, eps,
                                           unknown if unknown is not None else torch.empty(0, dtype=torch.int32), clear)


def add_norm_rows(part, residual, weight, eps):
    """residual += the sums of ``part`` (in place); returns rms(residual) * weight."""
    return _hip_or_raise().add_norm_rows(part, residual, weight, eps)


def rope_store_rows(part, bias, num_heads, positions, cos_sin, k_cache, v_cache, slot_mapping, k_scale=None, v_scale=None):
    """Rotates q and k of the fused qkv sums, stores k and v into the paged cache; returns q [M, H, 128]."""
    f = _none(part, torch.float32)
    return _hip_or_raise().rope_store_rows(
        part, bias if bias is not None else _none(part, torch.bfloat16), num_heads,
        positions, cos_sin, k_cache, v_cache, slot_mapping, k_scale if k_scale is not None else f,
        v_scale if v_scale is not None else f)


def decode_inputs(buf: dict, ids, batch, scratch_block: int, block_size: int) -> bool:
    """Fills a captured decode step's fixed buffers in one launch; False where the caller's tensors are not plain
    int64 / int32 rows on the GPU (nothing is written then)."""
    src = (ids, batch.positions, batch.slot_mapping, batch.context_lens, batch.block_tables)
    kinds = (torch.long, torch.long, torch.long, torch.int32, torch.int32)
    if _force_torch() or not all(t.device == buf["ids"].device and t.is_cuda and t.is_contiguous() and t.dtype == d
                                 for t, d in zip(src, kinds)):
        return False
    _hip_or_raise().decode_inputs(buf["ids"], buf["positions"], buf["slots"], buf["context_lens"], buf["block_tables"],
                                  *src, scratch_block, block_size)
    return True


def sample(
    logits: torch.Tensor,
    temperatures: torch.Tensor,
    top_ps: torch.Tensor,
    top_ks: torch.Tensor,
    seeds: torch.Tensor,
    steps: torch.Tensor,
    mask: Optional[torch.Tensor] = None,
    dbg: Optional[torch.Tensor] = None,
) -> Tuple[torch.Tensor, torch.Tensor]:
    if logits.is_cuda and not _force_torch():
        return _hip_or_raise().sample(logits, temperatures, top_ps, top_ks, seeds, steps, mask, dbg)
    return torch_ref.sample(logits, temperatures, top_ps, top_ks, seeds, steps, mask)


def moe_gateup(
    act: torch.Tensor,
    x: torch.Tensor,
    w_gate_up: torch.Tensor,
    sorted_ids: torch.Tensor,
    offsets: torch.Tensor,
    zeros: torch.Tensor,
) -> None:
    """Grouped MoE gate/up GEMM + fused silu*mul into `act` (sorted-by-expert
    row space, expert e at offsets[e]..offsets[e+1]; a sorted id of -1 reads
    `zeros`). GPU-only (Mixtral prefill hot path); the CPU path keeps the
    per-expert torch loop in models/mixtral.py."""
    _hip_or_raise().moe_gateup(act, x, w_gate_up, sorted_ids, offsets, zeros)


def moe_down(
    y: torch.Tensor,
    act: torch.Tensor,
    w_down: torch.Tensor,
    offsets: torch.Tensor,
    cleared: Optional[torch.Tensor] = None,
) -> None:
    """Grouped MoE down GEMM in sorted-row space (see moe_gateup). ``cleared``: the counters that router_top gives, used up
    by the call."""
    _hip_or_raise().moe_down(y, act, w_down, offsets, cleared)


def router_top(x: torch.Tensor, gate: torch.Tensor, k: int, places: bool):
    """Softmax routing of x [T, H] by gate [E, H]: (weights [T, k] fp32 that sum to one, experts [T, k] int32), and with
    ``places`` the (ids, pos, offsets) of moe_sort and counters for moe_down behind them. None where the kernel does not
    take the call (up to 32 experts and 8 choices, bf16 on the GPU, H a multiple of 64) or where a subclass, a function
    mode, a transform, a gradient or the compiler looks on."""
    if (x.is_cuda and not torch.compiler.is_compiling() and type(x) in _PLAIN and type(gate) in _PLAIN
            and not torch._C._len_torch_function_stack() and not _force_torch()):
        return _hip_or_raise().moe_route_try(x, gate, k, places)
    return None


def moe_sort(topi: torch.Tensor, experts: int):
    """(token of each sorted place, place of each (token, choice), expert offsets), without a host round trip."""
    return _hip_or_raise().moe_sort(topi.long().contiguous(), experts)


def moe_combine_rows(y: torch.Tensor, weights: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
    """sum over choices of weights[t, j] * y[pos[t, j]], fp32 sums, bf16 result."""
    return _hip_or_raise().moe_combine(y, weights.float().contiguous(), pos)


def levenshtein_pairs(
    chars: torch.Tensor,
    lens: torch.Tensor,
    pair_i: torch.Tensor,
    pair_j: torch.Tensor,
) -> torch.Tensor:
    """Batched Myers bit-parallel edit distance over packed [N, 64] uint8
    normalized strings; returns int32 distances per (i, j) pair. GPU-only —
    the CPU consensus path keeps the pure-python DP (utils/text.py)."""
    return _hip_or_raise().levenshtein_pairs(chars, lens, pair_i, pair_j)


# --- sequence-mixer family (kllms_amd._C_seq) -----------------------------------
# fp32 residual stream, block-local paged attention, recurrent mixers. The
# extension is separate from _C so that a model of this family compiles only
# its own kernels in a checkout where nothing is built yet.

_SEQ = None


def _seq():
    global _SEQ
    if _SEQ is None:
        from . import jit

        _SEQ = jit.load("_C_seq")
    return _SEQ


def seq_hip_loaded() -> bool:
    return _SEQ is not None


def _gpu(t: torch.Tensor) -> bool:
    return t.is_cuda and not _force_torch()


_NONE: dict = {}   # (dtype, device) -> an empty tensor standing for "not given"; it holds nothing, so sharing is safe


def _none(ref: torch.Tensor, dtype=None) -> torch.Tensor:
    key = (dtype or ref.dtype, ref.device)
    t = _NONE.get(key)
    if t is None:
        with torch.inference_mode(False):
            t = _NONE[key] = torch.empty(0, dtype=key[0], device=key[1])
    return t


def embed_rmsnorm(ids, table, weight, eps, pos_table=None, positions=None, w_next=None):
    """fp32 x = rms(table[ids] (+ pos_table[positions])) * weight; with w_next also rms(x) * w_next in the table's dtype."""
    if _gpu(table):
        out = torch.empty((ids.numel(), table.shape[1]), dtype=torch.float32, device=table.device)
        nxt = torch.empty(out.shape, dtype=table.dtype, device=table.device) if w_next is not None else _none(table)
        has = pos_table is not None
        _seq().embed_rmsnorm(out, ids, table, weight, eps, pos_table if has else _none(table),
                             positions if has else _none(table, torch.long),
                             w_next if w_next is not None else _none(table, torch.float32), nxt)
        return (out, nxt) if w_next is not None else out
    out = torch_ref.embed_rmsnorm(ids, table, weight, eps, pos_table, positions)
    return (out, torch_ref.rmsnorm_cast(out, w_next, eps, table.dtype)) if w_next is not None else out


def rmsnorm_cast(x, weight, eps, out_dtype):
    if _gpu(x):
        out = torch.empty(x.shape, dtype=out_dtype, device=x.device)
        _seq().rmsnorm_cast(out, x, weight, eps)
        return out
    return torch_ref.rmsnorm_cast(x, weight, eps, out_dtype)


def sandwich_residual(x, a, w_post, eps, b=None, wa=None, wb=None, w_next=None, out_dtype=None, cast=False):
    """x (fp32 residual, in place) += rms(y) * w_post with y = a, or
    y = (rms(a) wa + rms(b) wb) / 2; returns rms(x) * w_next in a's dtype.
    With w_next None: the new x in a's dtype if ``cast`` (the input of a
    sublayer that reads the stream itself), else None."""
    if _gpu(x):
        want = w_next is not None or cast
        out = torch.empty(a.shape, dtype=a.dtype, device=a.device) if want else _none(a)
        f = _none(x, torch.float32)
        _seq().sandwich_residual(
            x, a, b if b is not None else _none(a), wa if b is not None else f, wb if b is not None else f,
            w_post, w_next if w_next is not None else f, out, eps)
        return out if want else None
    return torch_ref.sandwich_residual(x, a, w_post, eps, b, wa, wb, w_next, out_dtype or a.dtype, cast)


def rope_pairs_store(q, k, v, positions, inv_freq, k_cache, v_cache, slot_mapping, kv_fresh=None) -> None:
    """kv_fresh (GPU only, optional): [T, 2, G, D] buffer that also receives
    this step's rotated keys ([:, 0]) and values ([:, 1]) packed, for the
    dense prefill kernel."""
    if _gpu(q):
        _seq().rope_pairs_store(q, k, v if v is not None else _none(q), positions, inv_freq,
                                k_cache, v_cache, slot_mapping,
                                kv_fresh if kv_fresh is not None else _none(q))
        return
    torch_ref.rope_pairs_store(q, k, v, positions, inv_freq, k_cache, v_cache, slot_mapping)


def attn_masked_paged(q, k_cache, v_cache, block_tables, token_seg, positions, scale, mask_kind, mask_size,
                      keep_first=0, sink=False, gate=None, row_map=None, out=None):
    """Paged softmax attention with a block-local (mask_kind 0) or sliding
    window + kept first tokens (mask_kind 1) causal mask, optional sink term,
    gate per head [T, H] or per element [T, H*Dv]. row_map / out (GPU only):
    serve just the listed rows, writing into an existing [T, H, Dv] tensor
    whose other rows another kernel fills."""
    if _gpu(q):
        if out is None:
            out = torch.empty((q.shape[0], q.shape[1], v_cache.shape[3]), dtype=q.dtype, device=q.device)
        _seq().attn_masked_paged(out, q, k_cache, v_cache, block_tables, token_seg, positions,
                                 gate if gate is not None else _none(q), scale, int(mask_kind), int(mask_size),
                                 int(keep_first), bool(sink),
                                 row_map if row_map is not None else _none(q, torch.int32),
                                 _none(q, torch.float32), _none(q, torch.float32), 0, 0.0,
                                 _none(q, torch.float32), _none(q, torch.float32))
        return out
    assert row_map is None and out is None
    return torch_ref.attn_masked_paged(q, k_cache, v_cache, block_tables, token_seg, positions, scale,
                                       mask_kind, mask_size, keep_first, sink, gate)


def attn_blocklocal_paged(q, k_cache, v_cache, block_tables, token_seg, positions, scale, mask_size,
                          gate=None, row_map=None, out=None):
    """Block-local mask, no sink, per-head gate: a case of attn_masked_paged."""
    if _gpu(q):
        return attn_masked_paged(q, k_cache, v_cache, block_tables, token_seg, positions, scale, 0, mask_size,
                                 0, False, gate, row_map, out)
    assert row_map is None and out is None
    return torch_ref.attn_blocklocal_paged(q, k_cache, v_cache, block_tables, token_seg, positions,
                                           scale, mask_size, gate)


def attn_varlen_mfma(out, q, k, v, grp_start, grp_qpos0, grp_len, scale) -> None:
    """Dense causal MFMA attention over packed pieces (bf16, head size 128;
    GPU only): each piece attends within itself. Tile groups come from
    dense_tile_groups()."""
    _seq().attn_varlen_mfma(out, q, k, v, grp_start, grp_qpos0, grp_len, scale)


def dense_tile_groups(pieces, device):
    """Host metadata for attn_varlen_mfma: pieces = [(first row, length)];
    32-row q-tiles of each piece, 8 per workgroup (idle wave slots = -1)."""
    NW = 8
    gs, gl, gq = [], [], []
    for row0, L in pieces:
        tiles = list(range(0, L, 32))
        for g0 in range(0, len(tiles), NW):
            grp = tiles[g0:g0 + NW]
            gs.append(row0)
            gl.append(L)
            gq.extend(grp + [-1] * (NW - len(grp)))
    return tuple(upload(torch.tensor([*gs, *gq, *gl], dtype=torch.int32), device).split([len(gs), len(gq), len(gl)]))


def head_gate(out, gate) -> None:
    """out[t, h, :] *= sigmoid(gate[t, h]) in place."""
    if _gpu(out):
        _seq().head_gate(out, gate)
        return
    out.mul_(torch.sigmoid(gate.float()).unsqueeze(-1).to(out.dtype))


def linear_attn_decay(q, k, v, decay, state, state_slots, cu_seqlens, seg_start, chunks=None):
    """S <- decay_h S + silu(k) silu(v)^T, o = S^T silu(q) over segments; o [T,
    H, V] fp32. ``chunks`` (GPU, from retention_chunks): the chunk-parallel form;
    None: token by token."""
    if _gpu(q):
        o = torch.empty((q.shape[0], q.shape[1], v.shape[2]), dtype=torch.float32, device=q.device)
        e = _none(q, torch.int32)
        ch, c0 = chunks if chunks is not None else (e, e)
        _seq().linear_attn_decay(o, q, k, v, decay, state, state_slots, cu_seqlens, seg_start, ch, c0)
        return o
    return torch_ref.linear_attn_decay(q, k, v, decay, state, state_slots, cu_seqlens, seg_start)


def gated_rmsnorm(o, weight, gate, eps, out_dtype, gate_act="sigmoid"):
    """Grouped RMS norm of o [T, groups, S] fp32 (weight [S] or None) times
    the activated gate (sigmoid or silu)."""
    if _gpu(o):
        out = torch.empty((o.shape[0], o.shape[1] * o.shape[2]), dtype=out_dtype, device=o.device)
        _seq().gated_rmsnorm(out, o, weight if weight is not None else _none(o), gate, eps,
                             0 if gate_act == "sigmoid" else 2)
        return out
    return torch_ref.gated_rmsnorm(o, weight, gate, eps, out_dtype, gate_act)


def causal_conv_silu(x, w, conv_state, state_slots, cu_seqlens, seg_start, token_seg, bias=None):
    if _gpu(x):
        y = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _seq().causal_conv_silu(y, x, w, conv_state, state_slots, cu_seqlens, seg_start, token_seg,
                                bias if bias is not None else _none(x, torch.float32))
        return y
    return torch_ref.causal_conv_silu(x, w, conv_state, state_slots, cu_seqlens, seg_start, bias)


def gated_delta_rule(q, k, v, beta_logit, a, dt_bias, a_log, state, state_slots, cu_seqlens, seg_start):
    if _gpu(q):
        o = torch.empty((v.shape[0], v.shape[1], v.shape[2]), dtype=torch.float32, device=q.device)
        _seq().gated_delta_rule(o, q, k, v, beta_logit, a, dt_bias, a_log, state, state_slots,
                                cu_seqlens, seg_start)
        return o
    return torch_ref.gated_delta_rule(q, k, v, beta_logit, a, dt_bias, a_log, state, state_slots,
                                      cu_seqlens, seg_start)


def gated_act(gate, up, limit: float, alpha: float, up_bias: float):
    """min(g, limit) sigmoid(alpha min(g, limit)) (clamp(u, +-limit) + up_bias)."""
    if _gpu(gate):
        out = torch.empty(gate.shape, dtype=gate.dtype, device=gate.device)
        _seq().gated_act(out, gate, up, limit, alpha, up_bias)
        return out
    return torch_ref.gated_act(gate, up, limit, alpha, up_bias)


def clamped_glu(gate, up, limit: float, alpha: float):
    if _gpu(gate):
        return gated_act(gate, up, limit, alpha, 1.0)
    return torch_ref.clamped_glu(gate, up, limit, alpha)


def silu_glu(gate, up):
    """silu(gate) * up in the activation dtype (bf16 or fp32)."""
    return gated_act(gate, up, float("inf"), 1.0, 0.0)


# --- a hybrid model's step of single decoded rows ----------------------------------
# GPU-only (ops/hip/seq/seq_steps.hip): callers ask hybrid_rows_ok first.

def hybrid_rows_ok(x, h, batch) -> bool:
    """Whether a step's sublayers can run as hybrid_*_rows: up to 128 rows, each its own sequence, bf16 on the GPU."""
    T = h.shape[0]
    return (_gpu(h) and h.dtype == torch.bfloat16 and x.dtype == torch.float32 and 1 <= T <= LINEAR_ROWS_MAX
            and batch.context_lens is not None and batch.block_tables is not None and batch.token_seg is not None
            and batch.block_tables.shape[0] == T and batch.block_tables.is_contiguous()
            and batch.positions.dtype == torch.long
            and all(t is not None and t.is_contiguous() and t.numel() == n and t.dtype == torch.int32 for t, n in (
                (batch.context_lens, T), (batch.state_slots, T), (batch.seg_start, T), (batch.token_seg, T),
                (batch.cu_seqlens, T + 1), (batch.block_tables, batch.block_tables.numel())))
            and all(t.is_contiguous() and t.numel() == T and t.dtype == torch.long
                    for t in (batch.positions, batch.slot_mapping))
            and not (torch.is_grad_enabled() and (x.requires_grad or h.requires_grad)) and _plain_call(x, h)
            and no_global_hooks())


def hybrid_parallel_rows(x, h, w_in, bias, at, inv_freq, k_cache, v_cache, o_left, decay, state, norm_right, o_right, wa,
                         wb, w_post, w_next, batch, heads, scale, mask_size, eps, once=False):
    """x (fp32 stream) += the parallel sublayer of h in place, with cache and state; returns the next normed input. at:
    columns of left q, k, head gates and right q, k, v, gate in h @ w_in^T + bias. None, and nothing done, where the
    weights do not lie as the kernels read them (contiguous, from 16 bytes on)."""
    return _seq().hybrid_parallel_rows(
        x, h, w_in, bias if bias is not None else _none(h), at, inv_freq, k_cache, v_cache, o_left, decay, state,
        norm_right, o_right, wa, wb, w_post, w_next, batch.positions, batch.slot_mapping, batch.block_tables,
        batch.context_lens, batch.state_slots, batch.cu_seqlens, batch.seg_start, heads, scale, mask_size, eps, once)


def hybrid_delta_rows(x, h, w_in, at, conv, conv_state, a2, g2, dt_bias, a_log, state, norm, w_out, w_post, w_next, batch,
                      kv_heads, eps, once=False):
    """The same of a gated-delta-rule sublayer; at: columns of q, k, v, the low-rank inputs and the write strengths."""
    return _seq().hybrid_delta_rows(x, h, w_in, at, conv, conv_state, a2, g2, dt_bias, a_log, state, norm, w_out, w_post,
                                    w_next, batch.state_slots, batch.cu_seqlens, batch.seg_start, batch.token_seg,
                                    kv_heads, eps, once)


def hybrid_glu_rows(x, h, w_in, w_down, w_post, w_next, limit, alpha, eps, once=False):
    """The same of a clamped gated-linear-unit sublayer."""
    return _seq().hybrid_glu_rows(x, h, w_in, w_down, w_post, w_next, limit, alpha, eps, once)


def embed_bigram(ids, table, bigram, scale, mul_prev, mul_cur, buckets, tok_state, state_slots, cu_seqlens,
                 seg_start, token_seg, out=None):
    """fp32 rows table[id] * scale (+ the hashed bigram row); ``out``: an
    existing contiguous [T, W] fp32 tensor to fill."""
    if _gpu(table):
        if out is None:
            out = torch.empty((ids.numel(), table.shape[1]), dtype=torch.float32, device=table.device)
        has = bigram is not None
        _seq().embed_bigram(out, ids, table, bigram if has else _none(table), float(scale), int(mul_prev),
                            int(mul_cur), int(buckets), tok_state if has else _none(table, torch.int32),
                            state_slots, cu_seqlens, seg_start, token_seg)
        return out
    x = torch_ref.embed_bigram(ids, table, bigram, scale, mul_prev, mul_cur, buckets, tok_state,
                               state_slots, cu_seqlens, seg_start)
    return x if out is None else out.copy_(x)


def group_norm_pair(x, a, b, w1, w2, groups, eps, out_dtype):
    """x (fp32 residual, in place) += a + b; returns the grouped RMS norm of x
    under two weights (the second may be None)."""
    if _gpu(x):
        h1 = torch.empty(x.shape, dtype=out_dtype, device=x.device)
        h2 = torch.empty(x.shape, dtype=out_dtype, device=x.device) if w2 is not None else None
        f = _none(x, torch.float32)
        e = _none(x, out_dtype)
        _seq().group_norm_pair(x, a if a is not None else e, b if b is not None else e, w1,
                               w2 if w2 is not None else f, h1, h2 if h2 is not None else e, int(groups), eps)
        return h1, h2
    return torch_ref.group_norm_pair(x, a, b, w1, w2, groups, eps, out_dtype)


def cast_concat(x, x0, a, b, out_dtype):
    """x (fp32 residual, in place) += a + b; returns [x | x0] in out_dtype."""
    if _gpu(x):
        out = torch.empty((x.shape[0], 2 * x.shape[1]), dtype=out_dtype, device=x.device)
        e = _none(x, out_dtype)
        _seq().cast_concat(out, x, x0, a if a is not None else e, b if b is not None else e)
        return out
    return torch_ref.cast_concat(x, x0, a, b, out_dtype)


def qk_norm_store(q, k, v, wq, wk, eps, k_cache, v_cache, slot_mapping) -> None:
    if _gpu(q):
        _seq().qk_norm_store(q, k, v, wq, wk, eps, k_cache, v_cache, slot_mapping)
        return
    torch_ref.qk_norm_store(q, k, v, wq, wk, eps, k_cache, v_cache, slot_mapping)


def token_shift_mix(h, mu, shift_state, state_slots, cu_seqlens, seg_start, token_seg, n_act):
    """([n_act, T, W] in h's dtype, [n - n_act, T, W] fp32) mixes of each row
    with its predecessor; carries the last row in shift_state."""
    if _gpu(h):
        T, W = h.shape
        n = mu.shape[0]
        act = torch.empty((n_act, T, W), dtype=h.dtype, device=h.device)
        f32 = torch.empty((n - n_act, T, W), dtype=torch.float32, device=h.device)
        _seq().token_shift_mix(act, f32, h, mu, shift_state, state_slots, cu_seqlens, seg_start, token_seg)
        return act, f32
    return torch_ref.token_shift_mix(h, mu, shift_state, state_slots, cu_seqlens, seg_start, n_act, h.dtype)


def wkv_recurrence(r, k, v, d, w0, u, state, state_slots, cu_seqlens, seg_start):
    if _gpu(r):
        o = torch.empty((r.shape[0], r.shape[1], v.shape[2]), dtype=torch.float32, device=r.device)
        _seq().wkv_recurrence(o, r, k, v, d, w0, u, state, state_slots, cu_seqlens, seg_start)
        return o
    return torch_ref.wkv_recurrence(r, k, v, d, w0, u, state, state_slots, cu_seqlens, seg_start)


def mlstm_recurrence(q, k, v, gates, gate_bias, cap, state, state_slots, cu_seqlens, seg_start):
    if _gpu(q):
        o = torch.empty((q.shape[0], q.shape[1], v.shape[2]), dtype=torch.float32, device=q.device)
        e = _none(q, torch.float32)
        _seq().mlstm_recurrence(o, q, k, v, gates, gate_bias, float(cap), state, state_slots, cu_seqlens,
                                seg_start, e, e)
        return o
    return torch_ref.mlstm_recurrence(q, k, v, gates, gate_bias, cap, state, state_slots, cu_seqlens,
                                      seg_start)


def mlstm_mix_out(q, k, v, gates, gate_bias, cap, state, state_slots, cu_seqlens, seg_start, weight, gate, eps,
                  out_dtype):
    """mlstm_recurrence followed by head_rmsnorm_gate(sigmoid); on the GPU the
    read-out's division happens inside the norm kernel."""
    if _gpu(q):
        T, H, V = q.shape[0], q.shape[1], v.shape[2]
        oe = torch.empty((T, H, V + 1), dtype=torch.float32, device=q.device)
        mt = torch.empty((T, H), dtype=torch.float32, device=q.device)
        _seq().mlstm_recurrence(_none(q, torch.float32), q, k, v, gates, gate_bias, float(cap), state, state_slots,
                                cu_seqlens, seg_start, oe, mt)
        out = torch.empty((T, H * V), dtype=out_dtype, device=q.device)
        _seq().head_rmsnorm_gate(out, oe, weight, gate, eps, 0, mt)
        return out
    o = torch_ref.mlstm_recurrence(q, k, v, gates, gate_bias, cap, state, state_slots, cu_seqlens, seg_start)
    return torch_ref.head_rmsnorm_gate(o, weight, gate, eps, "sigmoid", out_dtype)


def head_rmsnorm_gate(o, weight, gate, eps, gate_act, out_dtype):
    if _gpu(o):
        out = torch.empty((o.shape[0], o.shape[1] * o.shape[2]), dtype=out_dtype, device=o.device)
        _seq().head_rmsnorm_gate(out, o, weight, gate, eps,
                                 0 if gate_act == "sigmoid" else 1, _none(o, torch.float32))
        return out
    return torch_ref.head_rmsnorm_gate(o, weight, gate, eps, gate_act, out_dtype)


_SCORE_KINDS = {"softmax": 0, "sigmoid": 1, "top_softmax": 2}


def moe_route(z, correction, top, group_count, group_keep, score="softmax", renormalize=True, scale=1.0):
    """Routing from fp32 logits z [T, N]: (idx [T, top] int32, w [T, top] fp32)."""
    if _gpu(z):
        idx = torch.empty((z.shape[0], top), dtype=torch.int32, device=z.device)
        w = torch.empty((z.shape[0], top), dtype=torch.float32, device=z.device)
        _seq().moe_route(idx, w, _none(z, torch.int32), z, _none(z),
                         correction if correction is not None else _none(z), int(top), int(group_count),
                         int(group_keep), 0, _SCORE_KINDS[score], bool(renormalize), float(scale))
        return idx, w
    return torch_ref.moe_route(z, correction, top, group_count, group_keep, score, renormalize, scale)


def moe_route_rows(h, router, correction, top, group_count, group_keep, experts, all_experts_form,
                   score="softmax", renormalize=True, scale=1.0):
    """Router GEMV in fp32 + routing in one kernel. Returns (idx, w, rowidx);
    rowidx [T, top] (only when all_experts_form) addresses rows of the
    all-experts output [experts * T, W]: choice * T + row, -1 = identity."""
    T = h.shape[0]
    if _gpu(h):
        idx = torch.empty((T, top), dtype=torch.int32, device=h.device)
        w = torch.empty((T, top), dtype=torch.float32, device=h.device)
        rowidx = torch.empty((T, top), dtype=torch.int32, device=h.device) if all_experts_form else None
        _seq().moe_route(idx, w, rowidx if rowidx is not None else _none(h, torch.int32), h, router,
                         correction if correction is not None else _none(router),
                         int(top), int(group_count), int(group_keep), int(experts),
                         _SCORE_KINDS[score], bool(renormalize), float(scale))
        return idx, w, rowidx
    z = torch.nn.functional.linear(h.float(), router)
    idx, w = torch_ref.moe_route(z, correction, top, group_count, group_keep, score, renormalize, scale)
    rowidx = None
    if all_experts_form:
        t_idx = torch.arange(T, dtype=torch.int32, device=h.device).unsqueeze(1)
        rowidx = torch.where(idx < experts, idx * T + t_idx, torch.full_like(idx, -1))
    return idx, w, rowidx


def moe_combine(rows, h, rowidx, w, out_dtype, extra=None, extra_gate=None):
    """Fixed-order sum of each row's chosen expert rows, weighted by w (None =
    unweighted), plus sigmoid(extra_gate[t]) * extra[t] when given
    (extra_gate: a [T] view, any stride; None: plus extra[t])."""
    if _gpu(h):
        out = torch.empty(h.shape, dtype=out_dtype, device=h.device)
        _seq().moe_combine(out, rows, h, rowidx, w if w is not None else _none(h, torch.float32),
                           extra if extra is not None else _none(h),
                           extra_gate if extra_gate is not None else _none(h))
        return out
    return torch_ref.moe_combine(rows, h, rowidx, w, out_dtype, extra, extra_gate)


def scale_rows(h, src_row, scale):
    """out[i] = h[src_row[i]] * scale[i]: expert inputs that carry their
    routing weight. src_row int32 [n], scale fp32 [n]."""
    if _gpu(h):
        out = torch.empty((src_row.numel(), h.shape[1]), dtype=h.dtype, device=h.device)
        _seq().scale_rows(out, h, src_row, scale)
        return out
    return torch_ref.scale_rows(h, src_row, scale)


def moe_spread_rows(h, idx, w, experts: int):
    """[experts, T, W] inputs of the all-experts form when the routing weight
    sits on the expert's input: w[t, j] * h[t] for row t's j-th choice, zero
    rows for the experts a row did not choose."""
    if _gpu(h):
        out = torch.empty((experts, h.shape[0], h.shape[1]), dtype=h.dtype, device=h.device)
        _seq().moe_spread_rows(out, h, idx, w)
        return out
    return torch_ref.moe_spread_rows(h, idx, w, experts)


def gelu_tanh(x):
    """Tanh-form gelu of a [T, C] row view, in x's dtype."""
    if _gpu(x):
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _seq().gelu_tanh(out, x)
        return out
    return torch_ref.gelu_tanh(x)


def scale_softcap_(z, scale: float, cap: float) -> None:
    """fp32 logits in place: z * scale, then cap * tanh(. / cap) if cap > 0."""
    if _gpu(z):
        _seq().scale_softcap(z, float(scale), float(cap))
        return
    torch_ref.scale_softcap_(z, scale, cap)


def latent_kv_store(q, dkv, w_norm, eps, positions, inv_freq, cache, slot_mapping, nope_dim) -> None:
    """Rotates the rotated part of every query head in place; norms the
    latent, rotates the shared key part and stores [latent | key part] into
    the paged latent cache."""
    if _gpu(q):
        _seq().latent_kv_store(q, dkv, w_norm, eps, positions, inv_freq, cache, slot_mapping, int(nope_dim))
        return
    torch_ref.latent_kv_store(q, dkv, w_norm, eps, positions, inv_freq, cache, slot_mapping, nope_dim)


def attn_latent_paged(q_abs, q, cache, block_tables, token_seg, positions, scale, mask_size, gate, nope_dim,
                      tile_rows: int = 0, use_mfma: bool = True, key_splits: int = 0, sink=None):
    """Sliding-window softmax attention over the paged latent cache in the
    absorbed form (one shared key/value row per token for all heads):
    returns the heads' weighted latent sums [T, H, C], gated per head. sink
    [H] fp32: one more term exp(sink_h) in the softmax denominator.
    GPU: bf16 rows go through the matrix-unit kernel when the sizes fit it
    (``tile_rows`` = query rows per workgroup, 0 = as many as fit 32 (row,
    head) columns; 1 suits steps of single decoded tokens), fp32 rows and
    other sizes through the plain kernel. ``key_splits`` (with tile_rows 1):
    workgroups that share one row's keys, merged by a second kernel; 0 = as
    many as fill the chip for this step (few rows, long windows), -1 = none."""
    if _gpu(q):
        T, H, C = q.shape[0], q.shape[1], q_abs.shape[2]
        out = torch.empty((T, H, C), dtype=q.dtype, device=q.device)
        ns = 1
        if tile_rows == 1 and use_mfma and q.dtype == torch.bfloat16 and key_splits >= 0:
            # an upper bound of a row's 32-key tiles, from the window or the block table's width
            reach = mask_size if mask_size > 0 else block_tables.shape[1] * cache.shape[2]
            reach = min(reach, block_tables.shape[1] * cache.shape[2])
            tiles = max(1, (reach + 31) // 32)
            groups = T * ((H + 31) // 32)
            # about four tiles per workgroup, and no more workgroups than two per compute unit
            ns = key_splits or max(1, min((tiles + 3) // 4, 512 // max(1, groups)))
            ns = max(1, min(ns, tiles, 64))
        f = torch.float32
        f_none = _none(q, f)
        part_o = torch.empty((T, H, ns, C), dtype=f, device=q.device) if ns > 1 else f_none
        part_ml = torch.empty((T, H, ns, 2), dtype=f, device=q.device) if ns > 1 else f_none
        _seq().attn_latent_paged(out, q_abs, q, cache, block_tables, token_seg, positions,
                                 gate if gate is not None else _none(q), float(scale), int(mask_size),
                                 int(nope_dim), int(tile_rows), bool(use_mfma), part_o, part_ml,
                                 sink if sink is not None else f_none)
        return out
    return torch_ref.attn_latent_paged(q_abs, q, cache, block_tables, token_seg, positions, scale, mask_size,
                                       gate, nope_dim, sink)


def sigmoid_gate_(x, gate) -> None:
    """x [T, C] *= sigmoid(gate) element by element; gate a row view."""
    if _gpu(x):
        _seq().sigmoid_gate(x, gate)
        return
    torch_ref.sigmoid_gate_(x, gate)


def attn_window_sink(q, st, batch, spec, gate):
    """Windowed attention with kept first tokens and a sink for one step's
    rows, keys through the block table (prompt portions, decoded tokens and
    mixes alike)."""
    return attn_masked_paged(q, st.k, st.v, batch.block_tables, batch.token_seg, batch.positions, spec.scale,
                             1, spec.mask_size, spec.keep_first, spec.sink, gate)


def ln_residual_mix(x_in, a, w_post, eps, x_out, streams=None, n_prev=0, dwa=None):
    """x_out = x_in + layernorm(a) * w_post (a None: x_in itself); with
    ``streams`` [L, T, W] the sum is kept as streams[n_prev] and x_out becomes
    sum_{j <= n_prev} dwa[j] * streams[j]. Returns the (mean, rstd) of every
    row of x_out, [T, 2] fp32 — what the next layer norm of the stream needs."""
    if _gpu(x_in):
        stats = torch.empty((x_in.shape[0], 2), dtype=torch.float32, device=x_in.device)
        f = _none(x_in, torch.float32)
        has = streams is not None
        _seq().ln_residual_mix(x_out, x_in, a if a is not None else f, w_post if a is not None else f, stats,
                               streams if has else f, dwa if has else f, int(n_prev), eps)
        return stats
    return torch_ref.ln_residual_mix(x_in, a, w_post, eps, x_out, streams, n_prev, dwa)


def ln_canon(x, stats, w_norm, canon_w, hist, state_slots, cu_seqlens, seg_start, token_seg, out_dtype):
    """Layer norm of the fp32 stream from its row statistics, times w_norm,
    plus the short causal convolution of that normed row with its
    predecessors (canon_w [K, W] taps-major; None = norm only); the
    sequence's last K-1 normed rows are carried in hist [slots, K-1, W] fp32."""
    if _gpu(x):
        out = torch.empty(x.shape, dtype=out_dtype, device=x.device)
        f = _none(x, torch.float32)
        has = canon_w is not None
        i = _none(x, torch.int32)
        _seq().ln_canon(out, x, stats, w_norm, canon_w if has else f, hist if has else f,
                        state_slots if has else i, cu_seqlens if has else i, seg_start if has else i,
                        token_seg if has else i)
        return out
    return torch_ref.ln_canon(x, stats, w_norm, canon_w, hist, state_slots, cu_seqlens, seg_start, out_dtype)


def qk_fullnorm_rope_store(q, k, v, wq, wk, eps, positions, inv_freq, k_cache, v_cache, slot_mapping) -> None:
    """Whole-projection RMS norm of q (in place) and k, half-split rotation of
    the first 2 * len(inv_freq) entries of every head, normed rotated k and v
    into the paged caches. k None: q only."""
    if _gpu(q):
        e = _none(q)
        has = k is not None
        _seq().qk_fullnorm_rope_store(q, k if has else e, v if has else e, wq,
                                      wk if has else _none(q, torch.float32), eps, positions, inv_freq,
                                      k_cache if has else e, v_cache if has else e,
                                      slot_mapping if has else _none(q, torch.long))
        return
    torch_ref.qk_fullnorm_rope_store(q, k, v, wq, wk, eps, positions, inv_freq, k_cache, v_cache, slot_mapping)


def pool_kv_update(k_cache, v_cache, pool_k, pool_v, block_tables, token_seg, positions, run: int,
                   row_map=None) -> None:
    """Means of the cached keys / values of every aligned run of ``run``
    positions that one of this step's rows completes, into the fp32 pooled
    caches. ``row_map`` (int32): the rows to look at, when the caller knows
    which rows end a run; None = every row."""
    if _gpu(k_cache):
        _seq().pool_kv_update(k_cache, v_cache, pool_k, pool_v, block_tables, token_seg, positions, int(run),
                              row_map if row_map is not None else _none(k_cache, torch.int32))
        return
    torch_ref.pool_kv_update(k_cache, v_cache, pool_k, pool_v, block_tables, token_seg, positions, run, row_map)


def attn_window_pool_paged(q, k_cache, v_cache, pool_k, pool_v, block_tables, token_seg, positions, scale,
                           softcap, mask_size, run, key_splits: int = 0):
    """Sliding-window attention over the paged cache with the pooled entries
    of the runs that lie wholly before the window, soft-capped scores; prompt
    portions, decoded tokens and mixes alike. ``key_splits`` (GPU): workgroups
    that share one (row, head)'s keys, merged by a second kernel; 0 = as many
    as fill the chip for this step (few rows, long windows), 1 = none."""
    if _gpu(q):
        out = torch.empty((q.shape[0], q.shape[1], v_cache.shape[3]), dtype=q.dtype, device=q.device)
        f = _none(q, torch.float32)
        has = run > 0
        # steps of few rows: a (row, head)'s key tiles are shared out over several workgroups.
        # An upper bound of the visible keys, from the mask or the block table's width
        T, H = q.shape[0], q.shape[1]
        ctx = block_tables.shape[1] * k_cache.shape[2]
        reach = min(ctx, mask_size + (ctx // run if has else 0)) if mask_size > 0 else ctx
        tiles = (reach + 63) // 64
        ns = key_splits or max(1, min((tiles + 3) // 4, 512 // max(1, T * H), 64))
        part_o = torch.empty((T, H, ns, v_cache.shape[3]), dtype=torch.float32, device=q.device) if ns > 1 else f
        part_ml = torch.empty((T, H, ns, 2), dtype=torch.float32, device=q.device) if ns > 1 else f
        _seq().attn_masked_paged(out, q, k_cache, v_cache, block_tables, token_seg, positions, _none(q),
                                 scale, 2, int(mask_size), 0, False, _none(q, torch.int32),
                                 pool_k if has else f, pool_v if has else f, int(run), float(softcap),
                                 part_o, part_ml)
        return out
    return torch_ref.attn_window_pool_paged(q, k_cache, v_cache, pool_k, pool_v, block_tables, token_seg,
                                            positions, scale, softcap, mask_size, run)


def ssd_recurrence(x, B, C, dt, dt_bias, a_log, skip, state, state_slots, cu_seqlens, seg_start):
    """S <- exp(-exp(a_log) d) S + d B x^T, o = S^T C + skip x with
    d = softplus(dt + dt_bias) per head and token; o [T, H, V] fp32."""
    if _gpu(x):
        o = torch.empty((x.shape[0], x.shape[1], x.shape[2]), dtype=torch.float32, device=x.device)
        _seq().ssd_recurrence(o, x, B, C, dt, dt_bias, a_log, skip, state, state_slots, cu_seqlens, seg_start)
        return o
    return torch_ref.ssd_recurrence(x, B, C, dt, dt_bias, a_log, skip, state, state_slots, cu_seqlens, seg_start)


def gate_group_rmsnorm(o, weight, gate, eps, out_dtype):
    """(o * silu(gate)) RMS-normed in groups, times weight: o [T, groups, S] fp32."""
    if _gpu(o):
        out = torch.empty((o.shape[0], o.shape[1] * o.shape[2]), dtype=out_dtype, device=o.device)
        _seq().gated_rmsnorm(out, o, weight, gate, eps, 1)
        return out
    return torch_ref.gate_group_rmsnorm(o, weight, gate, eps, out_dtype)


RETENTION_CHUNK = 64          # rows per chunk of the chunk-parallel form
RETENTION_MAX_DIM = 128       # largest key size of the chunk-parallel form


def retention_chunks(segs, device):
    """Host metadata of the chunk-parallel form: segs = [(start position,
    rows)] of a step in row order -> (chunks [NC, 4] int32: first row, rows,
    segment, 0; seg_c0 [B + 1] int32: a segment's range of chunks)."""
    chunks, c0, row0 = [], [0], 0
    for b, (_, n) in enumerate(segs):
        chunks += [(row0 + i, min(RETENTION_CHUNK, n - i), b, 0) for i in range(0, n, RETENTION_CHUNK)]
        c0.append(len(chunks))
        row0 += n
    return (upload(torch.tensor(chunks, dtype=torch.int32).reshape(-1, 4), device),
            upload(torch.tensor(c0, dtype=torch.int32), device))


def retention(q, k, v, decay, positions, inv_freq, state, state_slots, cu_seqlens, seg_start, chunks=None):
    """Half-split rotation of q and k, k scaled by D^-1/2, then
    S <- decay_h S + k v^T, o = S^T q over segments; o [T, H, V] fp32.
    ``chunks`` (GPU, from retention_chunks): the chunk-parallel form; None:
    token by token."""
    if _gpu(q):
        o = torch.empty((q.shape[0], q.shape[1], v.shape[2]), dtype=torch.float32, device=q.device)
        e = _none(q, torch.int32)
        ch, c0 = chunks if chunks is not None else (e, e)
        _seq().retention(o, q, k, v, decay, positions, inv_freq, state, state_slots, cu_seqlens, seg_start, ch, c0)
        return o
    return torch_ref.retention(q, k, v, decay, positions, inv_freq, state, state_slots, cu_seqlens, seg_start)


def retention_mix_out(q, k, v, gate, decay, positions, inv_freq, state, state_slots, cu_seqlens, seg_start, eps,
                      out_dtype, chunks=None, single=False):
    """retention followed by the heads' RMS norm (no weight) and silu gate
    ([T, H*V] logits). ``single`` (GPU): every segment is one row (decode),
    the whole of it runs as one kernel."""
    V = v.shape[2]
    if single and _gpu(q) and q.shape[2] <= 1024 and (V <= 256 or (V % 4 == 0 and V <= 1024)):
        out = torch.empty((q.shape[0], q.shape[1] * V), dtype=out_dtype, device=q.device)
        _seq().retention_step(out, q, k, v, gate, decay, positions, inv_freq, state, state_slots, seg_start, eps)
        return out
    o = retention(q, k, v, decay, positions, inv_freq, state, state_slots, cu_seqlens, seg_start, chunks)
    return gated_rmsnorm(o, None, gate, eps, out_dtype, "silu")


def gelu_glu(gate, up):
    """gelu(gate) * up (tanh form) of two row views, in gate's dtype."""
    if _gpu(gate):
        out = torch.empty(gate.shape, dtype=gate.dtype, device=gate.device)
        _seq().gelu_glu(out, gate, up)
        return out
    return torch_ref.gelu_glu(gate, up)


def relu2(x):
    """max(x, 0)^2 of a [T, C] row view, in x's dtype."""
    if _gpu(x):
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _seq().relu2(out, x)
        return out
    return torch_ref.relu2(x)


def gelu_mul_rows(z, table, ids, col0: int):
    """gelu(z [T, C]) * table[ids, col0 : col0 + C] in z's dtype."""
    if _gpu(z):
        out = torch.empty(z.shape, dtype=z.dtype, device=z.device)
        _seq().gelu_mul_rows(out, z, table, ids, int(col0))
        return out
    return torch_ref.gelu_mul_rows(z, table, ids, col0)


def add_cast(x, a, b, out_dtype):
    """x (fp32 residual, in place) += a + b (b may be None); returns x in
    out_dtype (fp32: x itself)."""
    if _gpu(x):
        out = x if out_dtype == torch.float32 else torch.empty(x.shape, dtype=out_dtype, device=x.device)
        _seq().add_cast(_none(x, out_dtype) if out is x else out, x, a, b if b is not None else _none(a))
        return out
    return torch_ref.add_cast(x, a, b, out_dtype)


def dyt_residual(x, a, post, nxt, out_dtype):
    """x (fp32 stream, in place) += tanh(alpha a) w + b with post = (alpha, w,
    b); returns tanh(alpha x) w + b with nxt, the next reader's input."""
    if _gpu(x):
        out = torch.empty(x.shape, dtype=out_dtype, device=x.device)
        _seq().dyt_residual(out, x, a, *post, *nxt)
        return out
    return torch_ref.dyt_residual(x, a, post, nxt, out_dtype)


def embed_dyt(ids, table, scale: float, nxt):
    """The stream's start: (x, h) with x = table[ids] * scale in fp32 and h =
    tanh(alpha x) w + b with nxt in the table's dtype."""
    if _gpu(table):
        x = torch.empty((ids.numel(), table.shape[1]), dtype=torch.float32, device=table.device)
        h = torch.empty(x.shape, dtype=table.dtype, device=table.device)
        _seq().embed_dyt(h, x, ids, table, float(scale), *nxt)
        return x, h
    return torch_ref.embed_dyt(ids, table, scale, nxt)


def rmsnorm_rows(x, weight, eps):
    """RMS norm of a [T, C] row view, packed result in x's dtype."""
    if _gpu(x):
        out = torch.empty(x.shape, dtype=x.dtype, device=x.device)
        _seq().rmsnorm_rows(out, x, weight, eps)
        return out
    return torch_ref.rmsnorm_rows(x, weight, eps)


def conv_qkv_store(y, w, conv_state, state_slots, cu_seqlens, seg_start, token_seg, positions, q_cols, temp_coef,
                   temp_every, k_cols=None, v_cols=None, k_cache=None, v_cache=None, slot_mapping=None, single=False):
    """Short causal convolution of a fused projection's rows; k and v columns
    into the paged caches, the q columns times the query temperature returned
    packed [T, width]. ``single``: every segment is one row (the history is
    updated by the same launch)."""
    if _gpu(y):
        q = torch.empty((y.shape[0], q_cols[1]), dtype=y.dtype, device=y.device)
        has = k_cols is not None
        e = _none(y)
        ko, vo = (k_cols[0], v_cols[0]) if has else (0, 0)
        _seq().conv_qkv_store(q, y, w, conv_state, state_slots, cu_seqlens, seg_start, token_seg, positions,
                              int(q_cols[0]), float(temp_coef), int(temp_every), int(ko), int(vo),
                              k_cache if has else e, v_cache if has else e,
                              slot_mapping if has else _none(y, torch.long), bool(single))
        return q
    return torch_ref.conv_qkv_store(y, w, conv_state, state_slots, cu_seqlens, seg_start, positions, q_cols, temp_coef,
                                    temp_every, k_cols, v_cols, k_cache, v_cache, slot_mapping)


def diff_tile_rows(heads: int, kv_heads: int) -> int:
    """Query rows per workgroup of the matrix-unit kernel: four tiles of 32
    columns, of one head each, shared between consecutive rows and up to four
    heads of a key/value head."""
    r = heads // kv_heads
    return 32 if r >= 3 else 128 // r


def diff_tiles(segs, rows: int, device):
    """Host metadata of attn_diff_paged for a step of segments
    [(start position, rows)] in row order: (tiles [NT, 2] int32: first row,
    row count — pieces of at most ``rows`` rows of a segment with two rows or
    more, longest key ranges first; single [NS] int32: the rows of one-row
    segments). Either may be empty."""
    tiles, single, row0 = [], [], 0
    for start, n in segs:
        if n == 1:
            single.append(row0)
        else:
            tiles += [(start + min(n, i + rows), row0 + i, min(rows, n - i)) for i in range(0, n, rows)]
        row0 += n
    tiles = [(r, n) for _, r, n in sorted(tiles, reverse=True)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=device)
    return i32(tiles).reshape(-1, 2), i32(single)


def diff_key_splits(rows: int, groups: int, reach: int) -> int:
    """Workgroups that share one row's keys in the decode form: as many as
    fill the chip, at most one per 64-key tile."""
    tiles = max(1, (reach + 63) // 64)
    return max(1, min(tiles, (512 + rows * groups - 1) // max(1, rows * groups), 64))


def attn_diff_paged(q, k_cache, v_cache, block_tables, token_seg, positions, scale, lam, out_scale, eps, plan=None,
                    use_mfma: bool = True, key_splits: int = 0):
    """Differential attention over the paged cache (plain causal):
    rms(softmax_1 v - lam softmax_2 v) * out_scale per head, [T, H, V].
    GPU: bf16 goes through the matrix-unit kernels when the sizes fit them —
    ``plan`` = diff_tiles() of the step, None = every row on its own (decode) —
    and fp32 and other sizes through the plain kernel. ``key_splits``: see
    diff_key_splits (0 = by that rule)."""
    if _gpu(q):
        T, H, V = q.shape[0], q.shape[1], v_cache.shape[3]
        out = torch.empty((T, H, V), dtype=q.dtype, device=q.device)
        f, i = _none(q, torch.float32), _none(q, torch.int32)
        mfma = use_mfma and q.dtype == torch.bfloat16 and _seq().attn_diff_mfma_fits(q.shape[2] // 2, V)
        args = (out, q, k_cache, v_cache, block_tables, token_seg, positions, float(scale), float(lam),
                float(out_scale), float(eps))
        if not mfma:
            _seq().attn_diff_paged(*args, 0, i, f, f)
            return out
        tiles, single = plan if plan is not None else (i, i)
        if tiles.numel():
            _seq().attn_diff_paged(*args, 1, tiles, f, f)
        n = T if plan is None else single.numel()
        if n:
            reach = block_tables.shape[1] * k_cache.shape[2]
            ns = key_splits or diff_key_splits(n, k_cache.shape[1], reach)
            part_o = torch.empty((n, H, 2, ns, V), dtype=torch.float32, device=q.device)
            part_ml = torch.empty((n, H, 2, ns, 2), dtype=torch.float32, device=q.device)
            _seq().attn_diff_paged(*args, 2, single, part_o, part_ml)
        return out
    return torch_ref.attn_diff_paged(q, k_cache, v_cache, block_tables, token_seg, positions, scale, lam, out_scale,
                                     eps)

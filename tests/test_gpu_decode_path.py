"""Kernels of the decode step against float64 at the sizes where their tiling changes."""

import pytest
import torch

from kllms_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = 128


def paged_case(B, KVH, gqa, BS, ctx, fp8, seed=0, width=None):
    """q, caches, scales, block tables, lengths; blocks shuffled, streams 0 and 1 share their full blocks."""
    g = torch.Generator().manual_seed(seed)
    need = [max(1, (c + BS - 1) // BS) for c in ctx]
    NB = sum(need) + 3
    perm = torch.randperm(NB, generator=g).tolist()
    bt = torch.zeros((B, width or max(need)), dtype=torch.int32)
    for b in range(B):
        own = [perm.pop() for _ in range(need[b])]
        if b == 1:
            own[:min(ctx[0], ctx[1]) // BS] = bt[0, :min(ctx[0], ctx[1]) // BS].tolist()
        bt[b, :need[b]] = torch.tensor(own, dtype=torch.int32)
    k, v = ((torch.randn(NB, KVH, BS, D, generator=g) * s).bfloat16() for s in (1.0, 1.0))
    q = torch.randn(B, KVH * gqa, D, generator=g).bfloat16()
    ks = vs = None
    if fp8:
        ks, vs = ((t.float().abs().amax(-1) / 448).clamp_min(1e-8) for t in (k, v))
        k, v = ((t.float() / s.unsqueeze(-1)).to(torch.float8_e4m3fn) for t, s in ((k, ks), (v, vs)))
    return q, k, v, ks, vs, bt, torch.tensor(ctx, dtype=torch.int32)


def attention64(q, k, v, ks, vs, bt, ctx, scale):
    B, H, _ = q.shape
    KVH, BS = k.shape[1], k.shape[2]
    k, v = k.to(torch.float32).double(), v.to(torch.float32).double()
    if ks is not None:
        k, v = k * ks.double().unsqueeze(-1), v * vs.double().unsqueeze(-1)
    out = torch.zeros(B, H, D, dtype=torch.float64)
    for b in range(B):
        L = int(ctx[b])
        rows = torch.arange(L)
        blk = bt[b].long()[rows // BS]
        kk, vv = k[blk, :, rows % BS], v[blk, :, rows % BS]     # [L, KVH, D]
        for h in range(H):
            g = h // (H // KVH)
            out[b, h] = torch.softmax(kk[:, g] @ q[b, h].double() * scale, 0) @ vv[:, g]
    return out


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("gqa,KVH,BS", [(1, 2, 16), (2, 1, 8), (4, 8, 16), (8, 2, 32), (4, 3, 5)])
@pytest.mark.parametrize("ctx,width", [
    ([1], None), ([63, 64], None), ([65, 255, 256, 257], None),
    ([1, 1000, 300, 17], 256),                 # a table much wider than the contexts: shares without keys
    ([700 - 13 * i for i in range(40)], None),  # several tiles for a wave
])
def test_paged_decode_tiles(gqa, KVH, BS, ctx, width, fp8):
    q, k, v, ks, vs, bt, n = paged_case(len(ctx), KVH, gqa, BS, ctx, fp8, seed=gqa * 31 + len(ctx), width=width)
    scale = D ** -0.5
    dev = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    # q as the fused projection's view: a token stride wider than its heads
    wide = torch.zeros(q.shape[0], q.shape[1] + 3, D, dtype=q.dtype, device=DEV)
    wide[:, :q.shape[1]] = q.to(DEV)
    out = ops.attn_decode_paged(wide[:, :q.shape[1]], dev(k), dev(v), dev(bt), dev(n), scale, dev(ks), dev(vs))
    ref = attention64(q, k, v, ks, vs, bt, n, scale)
    err = (out.double().cpu() - ref).abs()
    # one bf16 rounding of the result (2^-9), fp32 sums before it
    assert (err <= 2 ** -8 * ref.abs() + 2e-5).all(), err.max()

"""Kernels of the decode step against float64 at the sizes where their tiling changes."""

import pytest
import torch

from kllms_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = 128


def paged_case(B, KVH, gqa, BS, ctx, fp8, seed=0, width=None, shared=True):
    """q, caches, scales, block tables, lengths; blocks shuffled, streams 0 and 1 share their full blocks unless not ``shared``."""
    g = torch.Generator().manual_seed(seed)
    need = [max(1, (c + BS - 1) // BS) for c in ctx]
    NB = sum(need) + 3
    perm = torch.randperm(NB, generator=g).tolist()
    bt = torch.zeros((B, width or max(need)), dtype=torch.int32)
    for b in range(B):
        own = [perm.pop() for _ in range(need[b])]
        if b == 1 and shared:
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


# lengths at the edges of tiles, of rounds of four and of the lines where more workgroups share a context (3, 8 and 16 rounds);
# in one launch with counters, and with the merge in a second
@pytest.mark.parametrize("joined", [True, False])
# and, with 8 kv heads and 8 streams, the line from which the cache is streamed (512 keys, in fp8 1024), unless blocks are shared
@pytest.mark.parametrize("gqa,KVH,BS,fp8", [(1, 3, 16, False), (2, 2, 1, True), (4, 4, 16, False), (4, 8, 4, True), (4, 2, 6, True),
                                            (8, 1, 16, False), (8, 2, 32, True), (4, 8, 16, False), (1, 8, 16, True), (1, 16, 8, False)])
@pytest.mark.parametrize("ctx", [[384], [385, 1, 33], [1024, 1025, 31, 32], [2048, 2049, 640, 641, 5], [4200, 90],
                                 [513 + 17 * i for i in range(70)], [600, 512, 511, 512, 1024, 1023, 513, 1200]])
def test_shared_contexts(ctx, gqa, KVH, BS, fp8, joined):
    q, k, v, ks, vs, bt, n = paged_case(len(ctx), KVH, gqa, BS, ctx, fp8, seed=gqa + len(ctx) + BS, width=-(-8192 // BS))
    dev = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    arrived = torch.zeros(len(ctx) * KVH, dtype=torch.int32, device=DEV) if joined else None
    args = (dev(q), dev(k), dev(v), dev(bt), dev(n), D ** -0.5, dev(ks), dev(vs), arrived)
    out = ops.attn_decode_paged(*args)
    ref = attention64(q, k, v, ks, vs, bt, n, D ** -0.5)
    err = (out.double().cpu() - ref).abs()
    # one bf16 rounding of the result (2^-9), fp32 sums before it
    assert (err <= 2 ** -8 * ref.abs() + 2e-5).all(), err.max()
    assert torch.equal(ops.attn_decode_paged(*args), out)
    assert arrived is None or not arrived.any()


# shares that a thread merges one after the other, and counters in lines of their own
@pytest.mark.parametrize("gap", [0, 1, 32])
@pytest.mark.parametrize("gqa,KVH,BS,fp8", [(1, 1, 16, False), (1, 2, 16, True), (1, 2, 5, True), (2, 2, 8, True), (4, 1, 16, False),
                                            (8, 1, 16, False), (8, 1, 16, True)])
@pytest.mark.parametrize("ctx", [[6300], [17000, 40, 900], [140000]])
def test_few_long_contexts(ctx, gqa, KVH, BS, fp8, gap):
    q, k, v, ks, vs, bt, n = paged_case(len(ctx), KVH, gqa, BS, ctx, fp8, seed=gqa + len(ctx) + BS, shared=False)
    dev = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    arrived = torch.zeros(len(ctx) * KVH * gap, dtype=torch.int32, device=DEV) if gap else None
    args = (dev(q), dev(k), dev(v), dev(bt), dev(n), D ** -0.5, dev(ks), dev(vs), arrived)
    out = ops.attn_decode_paged(*args)
    ref = attention64(q, k, v, ks, vs, bt, n, D ** -0.5)
    err = (out.double().cpu() - ref).abs()
    # one bf16 rounding of the result (2^-9), fp32 sums before it
    assert (err <= 2 ** -8 * ref.abs() + 2e-5).all(), err.max()
    assert torch.equal(ops.attn_decode_paged(*args), out)
    assert arrived is None or not arrived.any()


@pytest.mark.parametrize("left", [float("inf"), float("nan")])
@pytest.mark.parametrize("gqa,KVH,BS,fp8", [(4, 2, 16, True), (1, 2, 4, True), (8, 1, 32, True), (2, 2, 6, True), (4, 2, 16, False)])
@pytest.mark.parametrize("ctx", [[1, 2, 3, 5], [33, 62, 127, 130], [385, 514, 1027, 2049]])
def test_what_lies_behind_the_context_is_not_read(ctx, gqa, KVH, BS, fp8, left):
    """Blocks are given to the next sequence as they are: keys, values and scales of the one before, which may have overflowed."""
    q, k, v, ks, vs, bt, n = paged_case(len(ctx), KVH, gqa, BS, ctx, fp8, seed=sum(ctx) + BS, shared=False)
    ref = attention64(q, k, v, ks, vs, bt, n, D ** -0.5)
    for b, c in enumerate(ctx):
        blk, at = int(bt[b, (c - 1) // BS]), (c - 1) % BS + 1
        for t in (k, v):
            (t.view(torch.uint8) if fp8 else t)[blk, :, at:] = 0x7f if fp8 else left
        for t in (ks, vs) if fp8 else ():
            t[blk, :, at:] = left
    dev = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    out = ops.attn_decode_paged(dev(q), dev(k), dev(v), dev(bt), dev(n), D ** -0.5, dev(ks), dev(vs))
    err = (out.double().cpu() - ref).abs()
    # one bf16 rounding of the result (2^-9), fp32 sums before it
    assert (err <= 2 ** -8 * ref.abs() + 2e-5).all(), err.max()


def test_empty_tables():
    """Rows without a context, and a table without a column: zeros."""
    q, k, v, _, _, bt, n = (t if t is None else t.to(DEV) for t in paged_case(3, 2, 4, 16, [40, 5, 17], False))
    out = ops.attn_decode_paged(q, k, v, bt[:, :0].contiguous(), n * 0, 0.1)
    assert not out.any()
    assert torch.equal(ops.attn_decode_paged(q, k, v, bt, n * 0, 0.1), out)


@pytest.mark.parametrize("joined", [True, False])
def test_a_table_of_more_positions_than_32_bits(joined):
    """As many columns as make 2^31 positions: the shares of a context are those of a table that is just wide enough."""
    q, k, v, _, _, bt, n = (t if t is None else t.to(DEV) for t in paged_case(1, 2, 4, 16, [5000], False))
    arrived = torch.zeros(2, dtype=torch.int32, device=DEV) if joined else None
    wide = torch.zeros((1, 2 ** 27), dtype=torch.int32, device=DEV)
    wide[:, :bt.shape[1]] = bt
    want = ops.attn_decode_paged(q, k, v, bt, n, 0.1, None, None, arrived)
    assert torch.equal(ops.attn_decode_paged(q, k, v, wide, n, 0.1, None, None, arrived), want)


@pytest.mark.parametrize("joined", [True, False])
@pytest.mark.parametrize("gqa,KVH,BS,fp8", [(1, 2, 16, False), (2, 3, 16, False), (4, 2, 16, False), (8, 1, 16, False), (4, 2, 16, True)])
@pytest.mark.parametrize("ctx", [[5, 40], [700, 1300]])
def test_infinite_values_give_infinities(ctx, gqa, KVH, BS, fp8, joined):
    """One key with an infinite value in some dims (in fp8 an infinite scale): those of the result are infinite, the others as ever."""
    q, k, v, ks, vs, bt, n = paged_case(len(ctx), KVH, gqa, BS, ctx, fp8, seed=sum(ctx), shared=False)
    q = q * 0.1                                                   # no weight near the smallest numbers
    for b, c in enumerate(ctx):
        blk, at = int(bt[b, (c // 2) // BS]), (c // 2) % BS
        if fp8:
            v.view(torch.uint8)[blk, :, at] &= 0x80               # signed zeros, which stay: 0 * inf
            v.view(torch.uint8)[blk, :, at, 1::3] |= 0x31
            vs[blk, :, at] = float("inf")
        else:
            v[blk, :, at, 1::6], v[blk, :, at, 4::6] = float("inf"), -float("inf")
    dev = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    arrived = torch.zeros(len(ctx) * KVH, dtype=torch.int32, device=DEV) if joined else None
    out = ops.attn_decode_paged(dev(q), dev(k), dev(v), dev(bt), dev(n), D ** -0.5, dev(ks), dev(vs), arrived).double().cpu()
    ref = attention64(q, k, v, ks, vs, bt, n, D ** -0.5)
    assert torch.equal(out[..., 1::3], ref[..., 1::3]) and ref[..., 1::3].isinf().all()
    if not fp8:
        rest = torch.arange(D) % 3 != 1
        err = (out - ref)[..., rest].abs()
        # one bf16 rounding of the result (2^-9), fp32 sums before it
        assert (err <= 2 ** -8 * ref[..., rest].abs() + 2e-5).all(), err.max()


@pytest.mark.parametrize("M", [1, 15, 16, 17, 33, 64, 65, 128])
@pytest.mark.parametrize("N,K", [(16, 128), (48, 256), (64, 384), (192, 1280), (2048, 2048)])
def test_linear_rows(M, N, K):
    g = torch.Generator().manual_seed(M * 13 + N + K)
    x = torch.randn(M, K + 8, generator=g).bfloat16().to(DEV)[:, :K]      # a row view
    w = (torch.randn(N, K, generator=g) * 0.05).bfloat16().to(DEV)
    assert ops.linear_rows_ok(x, w)
    ref = x.double() @ w.double().t()
    # fp32 sums of K products: K * 2^-24 of the terms' size
    tol = K * 2 ** -24 * (x.double().abs() @ w.double().abs().t())
    for s in (0, 1, 2, 5):
        got = ops._hip_or_raise().linear_rows(x, w, ops._none(x), 0, min(s, K // 128)).double().sum(0)
        assert ((got - ref).abs() <= tol).all()
    assert ((ops.linear_f32_rows(x, w).double() - ref).abs() <= tol).all()
    b = torch.randn(N, generator=g).bfloat16().to(DEV)
    got = ops._hip_or_raise().linear_rows(x, w, b, 1, 1).double()
    full = ref + b.double()
    assert ((got - full).abs() <= tol + 2 ** -8 * full.abs()).all()
    if N % 64 == 0:
        gate, up = ref.chunk(2, -1)
        full = torch.nn.functional.silu(gate) * up
        got = ops.linear_silu_rows(x, w).double()
        # the sums' and their bf16 rounding's error through silu(g) * u (slope below 1.1 in g), a fast exponential, the
        # result's rounding
        tg, tu = (tol + 2 ** -9 * ref.abs()).chunk(2, -1)
        assert ((got - full).abs() <= 1.1 * tg * (up.abs() + tu) + tu * gate.abs() + 2 ** -8 * full.abs() + 1e-6).all()


@pytest.mark.parametrize("S,M,n", [(1, 1, 128), (3, 5, 4096), (8, 128, 512), (2, 2, 16384), (5, 7, 4100)])
def test_add_and_embed_norm_rows(S, M, n):
    g = torch.Generator().manual_seed(S + M + n)
    part = torch.randn(S, M, n, generator=g).to(DEV)
    res = torch.randn(M, n, generator=g).bfloat16().to(DEV)
    w = torch.rand(n, generator=g).bfloat16().to(DEV)
    want = (res.double() + part.double().sum(0))
    out = ops.add_norm_rows(part, res, w, 1e-5)
    # the sum's rounding to bf16, then the residual's
    assert ((res.double() - want).abs() <= 2 ** -8 * (want.abs() + part.double().sum(0).abs()) + 1e-5).all()
    r = res.double()
    ref = r / torch.sqrt((r * r).mean(-1, keepdim=True) + 1e-5) * w.double()
    assert ((out.double() - ref).abs() <= 2 ** -8 * ref.abs() + 1e-5).all()
    table = torch.randn(11, n, generator=g).bfloat16().to(DEV)
    ids = torch.randint(0, 11, (M,), generator=g).to(DEV)
    clear = torch.ones(1500, dtype=torch.int32, device=DEV)
    out, row = ops.embed_norm_rows(ids, table, w, 1e-5, None, clear)
    assert torch.equal(row, table[ids]) and not clear.any()
    r = row.double()
    ref = r / torch.sqrt((r * r).mean(-1, keepdim=True) + 1e-5) * w.double()
    assert ((out.double() - ref).abs() <= 2 ** -8 * ref.abs() + 1e-5).all()


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("S,M,H,G,BS,bias", [(1, 1, 4, 4, 16, False), (3, 5, 8, 2, 16, True), (8, 128, 32, 8, 8, False)])
def test_rope_store_rows(S, M, H, G, BS, bias, fp8):
    g = torch.Generator().manual_seed(S * M + H)
    N = (H + 2 * G) * D
    # sums that are bf16 values already, so that the separate kernels start from the same numbers
    part = torch.zeros(S, M, N)
    part[-1] = torch.randn(M, N, generator=g).bfloat16().float()
    part = part.to(DEV)
    b = torch.randn(N, generator=g).bfloat16().to(DEV) if bias else None
    NB = (M + BS - 1) // BS + 1
    slots = torch.randperm(NB * BS, generator=g)[:M].to(DEV)
    pos = torch.randint(0, 500, (M,), generator=g).to(DEV)
    ang = torch.arange(512).unsqueeze(1) * 10000.0 ** (-torch.arange(0, D, 2) / D)
    cs = torch.cat([ang.cos(), ang.sin()], 1).to(DEV)
    kind = torch.float8_e4m3fn if fp8 else torch.bfloat16
    new = lambda: (torch.zeros(NB, G, BS, D, device=DEV, dtype=kind), torch.zeros(NB, G, BS, D, device=DEV, dtype=kind),  # noqa: E731
                   torch.ones(NB, G, BS, device=DEV) if fp8 else None, torch.ones(NB, G, BS, device=DEV) if fp8 else None)
    kc, vc, ks, vs = new()
    q = ops.rope_store_rows(part, b, H, pos, cs, kc, vc, slots, ks, vs)
    full = (part[-1].double() + (b.double() if bias else 0)).bfloat16().double()
    c, s = cs[pos].double()[:, None, :64], cs[pos].double()[:, None, 64:]
    rows = full.view(M, H + 2 * G, D)
    lo, hi = rows[..., :64], rows[..., 64:]
    rot = torch.cat([lo * c - hi * s, hi * c + lo * s], -1)
    want = torch.cat([rot[:, :H + G], rows[:, H + G:]], 1)
    size = 2 ** -8 * torch.maximum(want.abs(), want.roll(64, -1).abs()) + 1e-6
    assert ((q.double() - want[:, :H]).abs() <= size[:, :H]).all()
    for cache, sc, part64, tol in ((kc, ks, want[:, H:H + G], size[:, H:H + G]), (vc, vs, want[:, H + G:], size[:, H + G:])):
        got = cache[slots // BS, :, slots % BS].float().double()
        if fp8:
            sc = sc[slots // BS, :, slots % BS].double().unsqueeze(-1)
            assert torch.allclose(sc.squeeze(-1), part64.abs().amax(-1) / 448, rtol=2 ** -7)
            got, tol = got * sc, tol + part64.abs() * 2 ** -4 + sc * 2 ** -9    # e4m3: 3 bits, subnormals of 2^-9
        assert ((got - part64).abs() <= tol).all()
    assert int((kc.view(torch.uint8) != 0).any(-1).sum()) <= M * G      # nothing beside the slots


@pytest.mark.parametrize("preset", ["mid-llama", "mid-qwen", "mid-mixtral"])
@pytest.mark.parametrize("rows", [1, 16, 65, 128, 129])
def test_decode_rows_match_general_path(preset, rows):
    """A whole decode step through the few-row kernels against the same model's general kernels (the path of any other
    row count), both within bf16 rounding of each other."""
    from kllms_amd.engine.config import EngineConfig
    from kllms_amd.engine.engine import LLMEngine
    from kllms_amd.models.llama import ForwardBatch

    eng = LLMEngine(EngineConfig(model=preset, max_kv_blocks=1024, use_hip_graphs=False, seed=3))
    g = torch.Generator().manual_seed(rows)
    ctx = torch.randint(1, 60, (rows,), generator=g)
    seqs = [eng.kv.alloc_sequence(int(c)) for c in ctx]
    bt = torch.zeros(rows, 4, dtype=torch.int32)
    for i, s in enumerate(seqs):
        bt[i, :len(s.blocks)] = torch.tensor(s.blocks, dtype=torch.int32)
    eng.kv.k_all.normal_()
    eng.kv.v_all.normal_()
    slots = torch.tensor([s.blocks[(int(c) - 1) // 16] * 16 + (int(c) - 1) % 16 for s, c in zip(seqs, ctx)])
    batch = ForwardBatch(mode="decode", positions=(ctx - 1).to(DEV), slot_mapping=slots.to(DEV),
                         kv_caches=eng.kv.layer_caches(), block_tables=bt.to(DEV),
                         context_lens=ctx.to(torch.int32).to(DEV))
    ids = torch.randint(0, 2000, (rows,), generator=g).to(DEV)
    with torch.inference_mode():
        assert eng.model._takes_rows(ids, batch) == (rows <= 128)
        assert eng.model._takes_rows(ids, batch) != eng.model._takes_short(ids, batch)     # the latter: more rows
        got = eng.model.forward_decode(ids, batch)
        eng.model._takes_rows = eng.model._takes_short = lambda *a: False
        want = eng.model.forward_decode(ids, batch)
    # bf16 activations through two layers; a routed row may change its experts
    off = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert float(off.median()) < 0.02 and (preset == "mid-mixtral" or float(off.max()) < 0.05)


@pytest.mark.parametrize("gqa,KVH,BS", [(4, 4, 16), (1, 2, 8), (8, 1, 16)])
@pytest.mark.parametrize("mask", [24, 256, 1024])
def test_blocklocal_rows(gqa, KVH, BS, mask):
    ctx = [1, 23, 24, 25, 48, 256, 257, 1000, 1024, 1025]
    q, k, v, _, _, bt, n = paged_case(len(ctx), KVH, gqa, BS, ctx, False, seed=mask)
    gate = torch.randn(len(ctx), KVH * gqa + 8, generator=torch.Generator().manual_seed(1)).bfloat16().to(DEV)[:, :KVH * gqa]
    scale = D ** -0.5
    out = ops.attn_blocklocal_rows(q.to(DEV), k.to(DEV), v.to(DEV), bt.to(DEV), n.to(DEV), scale, mask, gate)
    for b, L in enumerate(ctx):
        lo = (L - 1) // mask * mask
        at = torch.arange(lo, L)
        blk = bt[b].long()[at // BS]
        kk, vv = k[blk, :, at % BS].double(), v[blk, :, at % BS].double()
        for h in range(KVH * gqa):
            ref = torch.softmax(kk[:, h // gqa] @ q[b, h].double() * scale, 0) @ vv[:, h // gqa]
            ref = ref * torch.sigmoid(gate[b, h].double().cpu())
            assert ((out[b, h].double().cpu() - ref).abs() <= 2 ** -8 * ref.abs() + 2e-5).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,Dk,V", [(2, 64, 128), (3, 128, 96), (2, 24, 40), (1, 5, 7)])
def test_linear_attention_chunks(H, Dk, V, dtype):
    """Chunk-parallel decayed linear attention against the recurrence in float64; segments fresh and continued, with
    lengths around the chunk size and single rows among them."""
    segs = [(0, 64), (5, 1), (0, 200), (9, 65), (3, 17)]
    T = sum(n for _, n in segs)
    g = torch.Generator().manual_seed(H + Dk)
    wide = torch.randn(T, H * (2 * Dk + V) + 8, generator=g).to(dtype)
    q, k, v = (wide[:, a:b].unflatten(1, (H, -1)) for a, b in
               ((0, H * Dk), (H * Dk, 2 * H * Dk), (2 * H * Dk, H * (2 * Dk + V))))
    decay = torch.exp(-1.0 / 2.0 ** (1 + 3 * torch.arange(H))).float()
    state = torch.randn(7, H, Dk, V, generator=g)
    slots = torch.tensor([4, 0, 6, 2, 3], dtype=torch.int32)
    cu = torch.tensor([0] + [n for _, n in segs]).cumsum(0).to(torch.int32)
    start = torch.tensor([s for s, _ in segs], dtype=torch.int32)
    dev = wide.to(DEV)
    qd, kd, vd = (dev[:, a:b].unflatten(1, (H, -1)) for a, b in
                  ((0, H * Dk), (H * Dk, 2 * H * Dk), (2 * H * Dk, H * (2 * Dk + V))))
    got_state = state.to(DEV)
    o = ops.linear_attn_decay(qd, kd, vd, decay.to(DEV), got_state, slots.to(DEV), cu.to(DEV), start.to(DEV),
                              ops.retention_chunks(segs, DEV))
    silu = torch.nn.functional.silu
    r = 0
    for b, (s, n) in enumerate(segs):
        S = torch.zeros(H, Dk, V, dtype=torch.float64) if s == 0 else state[slots[b]].double()
        size = S.abs()
        for t in range(r, r + n):
            kk, vv, qq = silu(k[t].double()), silu(v[t].double()), silu(q[t].double())
            S = S * decay.double().view(H, 1, 1) + kk.unsqueeze(-1) * vv.unsqueeze(-2)
            size = size * decay.double().view(H, 1, 1) + (kk.unsqueeze(-1) * vv.unsqueeze(-2)).abs()
            ref = (qq.unsqueeze(-2) @ S).squeeze(-2)
            bound = (qq.abs().unsqueeze(-2) @ size).squeeze(-2)
            # fp32 sums of at most Dk + 64 products of the terms' size, a few roundings each (fast silu included)
            assert ((o[t].double().cpu() - ref).abs() <= (Dk + 64) * 2 ** -23 * bound + 1e-6).all()
        assert ((got_state[slots[b]].double().cpu() - S).abs() <= 300 * 2 ** -23 * size + 1e-6).all()
        r += n
    assert torch.equal(got_state[1].cpu(), state[1])


@pytest.mark.parametrize("gated,fp8", [(False, False), (False, True), (True, False)])
def test_more_decode_rows_than_a_grid_has_in_y(gated, fp8):
    """65536 rows and more (a row per token of long prompt portions), against the same rows in two calls."""
    g = torch.Generator(device=DEV).manual_seed(5)
    B, H, KVH, BS, NB = 65539, 2, 1, 16, 64
    q = torch.randn(B, H, D, generator=g, device=DEV).bfloat16()
    k, v = (torch.randn(NB, KVH, BS, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    sc = [None, None]
    if fp8:
        sc = [torch.rand(NB, KVH, BS, generator=g, device=DEV) + 0.5 for _ in range(2)]
        k, v = k.to(torch.float8_e4m3fn), v.to(torch.float8_e4m3fn)
    bt = torch.randint(0, NB, (B, 2), generator=g, device=DEV, dtype=torch.int32)
    ctx = torch.randint(1, 33, (B,), generator=g, device=DEV, dtype=torch.int32)
    gate = torch.randn(B, H, generator=g, device=DEV).bfloat16()

    def rows(a, b):
        if gated:
            return ops.attn_blocklocal_rows(q[a:b], k, v, bt[a:b], ctx[a:b], 0.1, 24, gate[a:b])
        return ops.attn_decode_paged(q[a:b], k, v, bt[a:b], ctx[a:b], 0.1, *sc)

    assert torch.equal(rows(0, B), torch.cat([rows(0, 40000), rows(40000, B)]))


@pytest.mark.parametrize("gqa", [1, 2, 4, 8])
@pytest.mark.parametrize("L", [2, 33, 1024])         # both keys in a tile, in two waves' tiles, in two shares of the context
def test_blocklocal_rows_keep_32_bit_exponentials(L, gqa):
    """A context whose last key dominates and has V = 0, so that the result is the first key's exp(-50..-70) alone, and
    gates down to exp(-10): their relative error is the result's, which stays a normal number."""
    B, BS = 200, 16
    nb = (L + BS - 1) // BS
    g = torch.Generator().manual_seed(L + gqa)
    k, v = (torch.zeros(B * nb, 1, BS, D) for _ in range(2))
    k[..., 0] = -300.0
    bt = torch.arange(B * nb, dtype=torch.int32).view(B, nb)
    top, low = torch.arange(B) % 6 + 2.0, -48.0 - torch.arange(B) % 60 / 4
    for b in range(B):
        k[b * nb, 0, 0, 0] = low[b]
        v[b * nb, 0, 0] = torch.rand(D, generator=g).bfloat16().float() + 0.5
        k[bt[b, (L - 1) // BS], 0, (L - 1) % BS, 0] = top[b]
    v = v.bfloat16()
    q = torch.zeros(B, gqa, D)
    q[..., 0] = 1.0
    gate = (-10 * torch.rand(B, gqa, generator=g)).bfloat16()
    dev = lambda t: t.to(DEV)  # noqa: E731
    out = ops.attn_blocklocal_rows(dev(q.bfloat16()), dev(k.bfloat16()), dev(v), dev(bt),
                                   torch.full((B,), L, dtype=torch.int32, device=DEV), 1.0, 1024, dev(gate))
    p = torch.exp((low - top).double()).view(B, 1, 1)
    ref = p / (1 + p) * v[bt[:, 0].long(), 0, 0].double().view(B, 1, D) * torch.sigmoid(gate.double()).unsqueeze(-1)
    # the rounding to bf16, and about ten 32-bit ones of 2^-24 before it (exponentials, fold, divisions, gate)
    half = 2.0 ** (torch.floor(torch.log2(ref.abs())) - 8)
    assert ((out.double().cpu() - ref).abs() <= half + 10 * 2 ** -24 * ref.abs()).all()


def test_logits_keep_the_heads_gradient_and_bias():
    """A trainable LM head, or one with a bias, is not the few-row kernel's: it has neither."""
    from kllms_amd.engine.config import MODEL_PRESETS
    from kllms_amd.models.llama import LlamaForCausalLM

    with torch.device(DEV):
        model = LlamaForCausalLM(MODEL_PRESETS["mid-llama"])
    g = torch.Generator(device=DEV).manual_seed(0)
    w = model.lm_head.weight
    w.data.normal_(0, 0.02, generator=g)
    h = torch.randn(5, w.shape[1], generator=g, device=DEV).bfloat16()
    want = h.double() @ w.double().t()
    tol = 2 ** -8 * want.abs() + 1e-3                  # the library rounds to bf16
    w.requires_grad_(True)
    out = model.compute_logits(h)
    out.sum().backward()
    assert ((out.double() - want).abs() <= tol).all()
    # the gradient of every row is the sum of h, summed in 32 bits or more and rounded to bf16
    assert torch.allclose(w.grad.double(), h.double().sum(0).expand_as(w), rtol=2 ** -8, atol=1e-4)
    with torch.no_grad():
        assert not model.compute_logits(h).requires_grad
        model.lm_head.bias = torch.nn.Parameter(torch.randn(w.shape[0], generator=g, device=DEV).bfloat16())
        full = want + model.lm_head.bias.double()
        assert ((model.compute_logits(h).double() - full).abs() <= 2 ** -8 * full.abs() + 1e-3).all()


@pytest.mark.parametrize("rows", [3, 70])
def test_decode_step_takes_the_head_of_longer_rows(rows):
    """A decode step whose positions and slots lie in larger buffers gives what their heads give."""
    from dataclasses import replace

    from kllms_amd.engine.config import EngineConfig
    from kllms_amd.engine.engine import LLMEngine
    from kllms_amd.models.llama import ForwardBatch

    eng = LLMEngine(EngineConfig(model="mid-llama", max_kv_blocks=512, use_hip_graphs=False, seed=3))
    eng.kv.k_all.normal_(), eng.kv.v_all.normal_()
    ctx = torch.arange(rows) % 15 + 1
    bt = torch.arange(1, rows + 1, dtype=torch.int32).view(rows, 1)
    pad = torch.zeros(5, dtype=torch.long)
    batch = ForwardBatch(mode="decode", positions=torch.cat([ctx - 1, pad]).to(DEV),
                         slot_mapping=torch.cat([bt[:, 0] * 16 + ctx - 1, pad]).to(DEV), kv_caches=eng.kv.layer_caches(),
                         block_tables=bt.to(DEV), context_lens=ctx.to(torch.int32).to(DEV))
    exact = replace(batch, positions=batch.positions[:rows].clone(), slot_mapping=batch.slot_mapping[:rows].clone())
    ids = torch.arange(rows, device=DEV)
    with torch.inference_mode():
        a, b = (eng.model.forward_decode(ids, x) for x in (batch, exact))
    assert float(((a - b).norm(dim=-1) / b.norm(dim=-1)).max()) < 0.03     # bf16 through two layers, two sets of kernels


@pytest.mark.parametrize("rows", [1, 5, 64, 65, 128, 300])
def test_logits_are_32_bit_sums_at_every_row_count(rows):
    from kllms_amd.engine.config import MODEL_PRESETS
    from kllms_amd.models.llama import LlamaForCausalLM

    with torch.device(DEV):
        model = LlamaForCausalLM(MODEL_PRESETS["mid-llama"])
    g = torch.Generator(device=DEV).manual_seed(rows)
    w = model.lm_head.weight
    w.data.normal_(0, 0.02, generator=g)
    h = torch.randn(rows, w.shape[1], generator=g, device=DEV).bfloat16()
    out = model.compute_logits(h)
    assert out.dtype == torch.float32
    # sums of K products in 32 bits
    tol = w.shape[1] * 2 ** -24 * (h.double().abs() @ w.double().abs().t().contiguous())
    assert ((out.double() - h.double() @ w.double().t().contiguous()).abs() <= tol).all()


@pytest.mark.parametrize("captured", [False, True])
@pytest.mark.parametrize("bad", [-1, 2000, 1 << 40])
def test_an_id_outside_the_vocabulary_is_reported(bad, captured):
    """The step reads no foreign memory and its logits are NaN; the model raises once it has run, and goes on after that."""
    import copy

    from kllms_amd.engine.config import EngineConfig
    from kllms_amd.engine.engine import LLMEngine
    from kllms_amd.engine.graph_runner import DecodeGraphRunner
    from kllms_amd.models.llama import ForwardBatch

    eng = LLMEngine(EngineConfig(model="mid-llama", max_kv_blocks=64, use_hip_graphs=False, seed=3))
    bad = eng.model.cfg.vocab_size if bad == 2000 else bad
    rows = torch.arange(3, device=DEV)
    batch = ForwardBatch(mode="decode", positions=torch.zeros_like(rows), slot_mapping=(rows + 8) * eng.kv.block_size,
                         kv_caches=eng.kv.layer_caches(), block_tables=(rows + 8).to(torch.int32).view(3, 1),
                         context_lens=torch.ones(3, dtype=torch.int32, device=DEV))
    run = DecodeGraphRunner(eng, [4]).run if captured else eng.model.forward_decode
    good, wrong = rows + 5, torch.tensor([5, bad, 7], device=DEV)
    with torch.inference_mode():
        want = run(good, batch).cpu()
        for _ in range(2):
            got = run(wrong, batch).cpu()
            assert got[1].isnan().all() and torch.equal(got[::2], want[::2])
            with pytest.raises(IndexError, match="outside the vocabulary"):
                eng._check_ids()
            assert torch.equal(run(good, batch).cpu(), want)
        run(wrong, batch).cpu()
        with pytest.raises(IndexError):     # whoever does not ask is told at the next step
            run(good, batch)
        assert torch.equal(run(good, batch).cpu(), want)
        twin = copy.deepcopy(eng.model)     # its flag is its own
        twin.forward_decode(wrong, batch).cpu()
        eng.model.check_ids()
        with pytest.raises(IndexError):
            twin.check_ids()


def test_decode_step_takes_32_bit_ids():
    """Ids of 32 bits, which an embedding takes as well, go to the general path."""
    from kllms_amd.engine.config import EngineConfig
    from kllms_amd.engine.engine import LLMEngine
    from kllms_amd.models.llama import ForwardBatch

    eng = LLMEngine(EngineConfig(model="mid-llama", max_kv_blocks=64, use_hip_graphs=False, seed=3))
    rows = torch.arange(3, device=DEV)
    batch = ForwardBatch(mode="decode", positions=torch.zeros_like(rows), slot_mapping=(rows + 8) * eng.kv.block_size,
                         kv_caches=eng.kv.layer_caches(), block_tables=(rows + 8).to(torch.int32).view(3, 1),
                         context_lens=torch.ones(3, dtype=torch.int32, device=DEV))
    with torch.inference_mode():
        want, got = (eng.model.forward_decode((rows + 5).to(t), batch) for t in (torch.long, torch.int32))
    assert float(((got - want).norm(dim=-1) / want.norm(dim=-1)).max()) < 0.03     # bf16 through two layers, two sets of kernels


@pytest.mark.parametrize("M", [1, 31, 32, 33, 96, 97, 129, 192, 193, 256, 257, 384])
@pytest.mark.parametrize("N,K,splits", [(16, 128, 1), (80, 128, 2), (4112, 640, 5), (5136, 1152, 17), (2064, 4224, 3), (4096, 8192, 0)])
def test_linear_rows_tiles_and_splits(M, N, K, splits):
    """Tiles of 64 and 128 rows of W with a ragged last one, parts of x of uneven length, fewer stages than buffers, splits
    of uneven length, one stage each at most."""
    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) * 0.05).bfloat16().to(DEV)
    ref = x.double() @ w.double().t()
    tol = K * 2 ** -24 * (x.double().abs() @ w.double().abs().t())
    part = ops._hip_or_raise().linear_rows(x, w, ops._none(x), 0, splits)
    assert splits == 0 or part.shape[0] == min(splits, K // 64)
    assert ((part.double().sum(0) - ref).abs() <= tol).all()
    if M <= 256 and N % 64 == 0:
        gate, up = ref.chunk(2, -1)
        tg, tu = tol.chunk(2, -1)
        full = torch.nn.functional.silu(gate) * up
        # the sums' error through silu(g) * u (slope below 1.1 in g), a fast exponential, the result's rounding
        assert ((ops.linear_silu_rows(x, w).double() - full).abs()
                <= 1.1 * tg * (up.abs() + tu) + tu * gate.abs() + 2 ** -8 * full.abs() + 1e-6).all()


@pytest.mark.parametrize("M,N,K", [(m, n, 512) for m in (1, 32, 33, 128) for n in (5104, 5120, 5632, 5648, 7664, 7680, 8448, 8464)]
                         + [(m, n, k) for m in (129, 130, 193, 289, 384) for n, k in ((3056, 640), (3072, 640), (2048, 8064), (2048, 8192))]
                         + [(97, 5120, 8192), (97, 5120, 8320), (96, 5120, 8320)])
def test_linear_rows_at_the_lines_of_their_tiles(M, N, K):
    """Where the split sums go from tiles of 64 rows of W to 128 and back, and from four parts of x to three and two."""
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.05).bfloat16()
    xd, wt = x.double(), w.double().t().contiguous()
    assert ((ops.linear_part(x, w).double().sum(0) - xd @ wt).abs() <= K * 2 ** -24 * (xd.abs() @ wt.abs())).all()


@pytest.mark.parametrize("N,K", [(2032, 2048), (2064, 2048), (1984, 2048), (2112, 2048), (32768, 128), (32704, 128)])
@pytest.mark.parametrize("M", [1, 33, 128, 160])
def test_linear_rows_around_the_streaming_line(M, N, K):
    """A little below 8 MB of weights, and from there on, where they pass the caches by if the caller says so: each form, with
    ragged tiles, and the same bits either way."""
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.05).bfloat16()
    xd, wt = x.double(), w.double().t().contiguous()
    ref, tol = xd @ wt, K * 2 ** -24 * (xd.abs() @ wt.abs())     # fp32 sums of K products
    C, none = ops._hip_or_raise(), ops._none(x)
    for form in range(4):
        if M <= (384, 128, 128, 256)[form] and (form != 3 or N % 64 == 0):
            assert torch.equal(C.linear_rows(x, w, none, form, 0, True), C.linear_rows(x, w, none, form, 0))
    assert ((ops.linear_part(x, w).double().sum(0) - ref).abs() <= tol).all()
    if M <= 128:
        got = ops._hip_or_raise().linear_rows(x, w, ops._none(x), 1, 1).double()
        assert ((got - ref).abs() <= tol + 2 ** -8 * ref.abs()).all()
        assert ((ops.linear_f32_rows(x, w).double() - ref).abs() <= tol).all()
    if N % 64 == 0:
        gate, up = ref.chunk(2, -1)
        tg, tu = tol.chunk(2, -1)
        full = torch.nn.functional.silu(gate) * up
        assert ((ops.linear_silu_rows(x, w).double() - full).abs()
                <= 1.1 * tg * (up.abs() + tu) + tu * gate.abs() + 2 ** -8 * full.abs() + 1e-6).all()


@pytest.mark.parametrize("N", [128, 192, 16320, 16448, 20544, 32896])
@pytest.mark.parametrize("M", [5, 40, 128, 129, 256])
def test_gated_rows_at_the_lines_of_their_tiles(M, N):
    K = 256
    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(N, K, generator=g) * 0.05).bfloat16().to(DEV)
    ref = x.double() @ w.double().t()
    gate, up = ref.chunk(2, -1)
    tg, tu = (K * 2 ** -24 * (x.double().abs() @ w.double().abs().t())).chunk(2, -1)
    full = torch.nn.functional.silu(gate) * up
    assert ((ops.linear_silu_rows(x, w).double() - full).abs()
            <= 1.1 * tg * (up.abs() + tu) + tu * gate.abs() + 2 ** -8 * full.abs() + 1e-6).all()


@pytest.mark.parametrize("preset", ["mid-llama", "mid-qwen", "mid-mixtral"])
@pytest.mark.parametrize("lens", [[1], [7, 20], [128], [100, 29], [384], [200, 185]])
def test_short_prompts_match_general_path(preset, lens, monkeypatch):
    """A short prompt through the few-row products against the same model's general kernels, which a hook on any of its
    modules brings back, both within bf16 rounding of each other at every row (of a mixture: every row whose experts are the
    same); the cache rows of the first layer are the same."""
    from kllms_amd.engine.config import EngineConfig
    from kllms_amd.engine.engine import LLMEngine
    from kllms_amd.models.llama import ForwardBatch

    eng = LLMEngine(EngineConfig(model=preset, max_kv_blocks=256, use_hip_graphs=False, seed=3))
    seqs = [eng.kv.alloc_sequence(n) for n in lens]
    slots = torch.tensor([x for s in seqs for x in eng.kv.prefill_slot_mapping(s)])
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    batch = ForwardBatch(mode="prefill", positions=torch.tensor([p for n in lens for p in range(n)]).to(DEV),
                         slot_mapping=slots.to(DEV), kv_caches=eng.kv.layer_caches(), cu_seqlens=cu.to(DEV))
    ids = torch.randint(0, 2000, (sum(lens),), generator=torch.Generator().manual_seed(sum(lens))).to(DEV)
    m = eng.model
    route, experts = ops.router_top, []
    monkeypatch.setattr(ops, "router_top", lambda *a: (lambda r: (experts.append(r[1].sort(-1)[0]), r)[1])(route(*a)))

    def hidden():
        experts.clear()
        return m.forward_hidden(ids, batch).float(), list(experts)

    with torch.inference_mode():
        assert m._takes_short(ids, batch) == (sum(lens) <= 384)
        rows, chosen = hidden()
        got, kv = m.forward_prefill(ids, batch), eng.kv.k_all.clone()
        for owner in (m.embed_tokens, m.layers[0], m.layers[0].self_attn, m.layers[0].self_attn.qkv_proj, m.layers[1].self_attn.o_proj):
            seen = []
            h = owner.register_forward_hook(lambda *a: seen.append(1))
            want = m.forward_prefill(ids, batch)
            h.remove()
            assert seen
        with torch.autocast("cuda", torch.bfloat16):
            assert not m._takes_short(ids, batch)
        h = m.embed_tokens.register_forward_hook(lambda *a: None)
        general, chosen_too = hidden()
        h.remove()
    off = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert float(off.max()) < (0.5 if preset == "mid-mixtral" else 0.05)      # a routed row may change its experts
    same = torch.ones(sum(lens), dtype=torch.bool, device=DEV)
    assert len(chosen) == len(chosen_too) == (m.cfg.num_layers if preset == "mid-mixtral" else 0)
    for a, b in zip(chosen, chosen_too):
        same &= (a == b).all(-1)
    off = ((rows - general).norm(dim=-1) / general.norm(dim=-1))[same]
    # two layers, each some six roundings to bf16 (2^-9) apart
    assert float(same.float().mean()) >= 0.9 and float(off.max()) < 0.02
    assert torch.equal(kv[0], eng.kv.k_all[0])


@pytest.mark.parametrize("S,M,n", [(4, 3, 4096), (9, 2, 2048), (17, 5, 4100), (16, 1, 16384)])
def test_add_norm_rows_at_the_batches_of_splits(S, M, n):
    test_add_and_embed_norm_rows(S, M, n)


@pytest.mark.parametrize("S,M", [(2, 3), (4, 1), (5, 7), (9, 2), (17, 5)])
def test_rope_store_rows_at_the_batches_of_splits(S, M):
    test_rope_store_rows(S, M, 8, 2, 16, True, False)


@pytest.mark.parametrize("M", [1, 2, 5, 64, 128, 129, 384])
@pytest.mark.parametrize("stride", [0, 8, 120, 512, 648, (1 << 25) - 8, 1 << 25])
@pytest.mark.parametrize("N,K", [(64, 640), (5184, 640)])
def test_linear_rows_of_repeated_and_overlapping_rows(M, stride, N, K):
    """Rows that are one and the same, that overlap, and that lie further apart than 32 bits of offsets reach over a tile."""
    if stride > K + 8 and M > 5:
        M = 65 if stride < 1 << 25 and M == 128 and N == 64 else 5       # 4 GiB of rows once
    g = torch.Generator(device=DEV).manual_seed(M + stride + N)
    x = torch.empty((M - 1) * stride + K, dtype=torch.bfloat16, device=DEV).as_strided((M, K), (stride, 1))
    for m in range(M):
        x[m].normal_(generator=g)
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.05).bfloat16()
    xd, wt = x.double().contiguous(), w.double().t().contiguous()
    ref = xd @ wt
    tol = K * 2 ** -24 * (xd.abs() @ wt.abs())
    C, none = ops._hip_or_raise(), ops._none(x)
    for splits in (0, 1, 5):
        assert ((C.linear_rows(x, w, none, 0, splits).double().sum(0) - ref).abs() <= tol).all()
    if M <= 256:
        gate, up = ref.chunk(2, -1)
        tg, tu = tol.chunk(2, -1)
        full = torch.nn.functional.silu(gate) * up
        assert ((ops.linear_silu_rows(x, w).double() - full).abs()
                <= 1.1 * tg * (up.abs() + tu) + tu * gate.abs() + 2 ** -8 * full.abs() + 1e-6).all()
    if M <= 128:
        assert ops.linear_rows_ok(x, w)
        assert ((ops.linear_f32(x, w).double() - ref).abs() <= tol).all()
        assert ((C.linear_rows(x, w, none, 1, 1).double() - ref).abs() <= tol + 2 ** -8 * ref.abs()).all()


@pytest.mark.parametrize("preset", ["mid-llama", "mid-zutalix"])
def test_steps_of_weights_that_pass_the_caches_by(preset):
    """The word of a model of many weights reaches each product of a step and changes none of its bits."""
    from kllms_amd.engine.config import EngineConfig
    from kllms_amd.engine.engine import LLMEngine

    out, said = [], []
    for once in (False, True):
        eng = LLMEngine(EngineConfig(model=preset, max_kv_blocks=64, use_hip_graphs=False, seed=3))
        m = eng.model
        assert not m._once
        for part in m.modules():
            for name in ("_once", "once"):
                if name in part.__dict__:
                    setattr(part, name, once)
        saved, rows = ops.linear_part, []
        ops.linear_part = lambda x, w, o=False: rows.append(o) or saved(x, w, o)
        try:
            s = eng.open_sequence()
            eng.step_segments([(s, list(range(5, 40)), [34])])
            out.append([eng.step_segments([(s, [7 + i], [0])]) for i in range(2)])
        finally:
            ops.linear_part = saved
        said.append(set(rows))
    assert all(torch.equal(a, b) for a, b in zip(*out))
    assert said == ([set(), set()] if preset == "mid-zutalix" else [{False}, {True}])


@pytest.mark.parametrize("preset", ["mid-llama", "mid-zutalix"])
@pytest.mark.parametrize("rows", [1, 5, 64, 128])
def test_logits_of_one_row_repeated(preset, rows):
    from kllms_amd.engine.config import EngineConfig
    from kllms_amd.engine.engine import LLMEngine

    m = LLMEngine(EngineConfig(model=preset, max_kv_blocks=64, use_hip_graphs=False, seed=3)).model
    w = m.lm_head.weight
    h = torch.randn(1, w.shape[1], generator=torch.Generator().manual_seed(rows)).bfloat16().to(DEV)
    with torch.inference_mode():
        out = m.compute_logits(h.expand(rows, -1))
    tol = w.shape[1] * 2 ** -24 * (h.double().abs() @ w.double().abs().t().contiguous())
    assert ((out.double() - h.double() @ w.double().t().contiguous()).abs() <= tol).all()


class _Tagged(torch.Tensor):
    pass


@pytest.mark.parametrize("which", ["qkv_proj", "o_proj", "gate_up_proj", "down_proj", "embed_tokens", "bias"])
@pytest.mark.parametrize("how", ["transposed", "off 16 bytes", "subclass"])
def test_short_prompts_with_weights_that_lie_otherwise(which, how):
    """What the few-row products do not read the library does, in whole prompts and in portions of more than 128 rows."""
    from kllms_amd.engine.config import EngineConfig
    from kllms_amd.engine.engine import LLMEngine

    eng = LLMEngine(EngineConfig(model="mid-qwen", max_kv_blocks=64, use_hip_graphs=False, enable_prefix_caching=False, seed=3))
    ids = torch.randint(0, 2000, (200,), generator=torch.Generator().manual_seed(1))

    def run():
        out = []
        for n in (100, 200):
            if n > 128:
                s = eng.open_sequence()
                out.append(eng.step_segments([(s, ids[:n].tolist(), [n - 1])]).double())
                eng.kv.free_sequence(s)
            s = eng.kv.alloc_sequence(n)
            batch = ForwardBatch(mode="prefill", positions=torch.arange(n, device=DEV), kv_caches=eng.kv.layer_caches(),
                                 slot_mapping=torch.tensor(eng.kv.prefill_slot_mapping(s), device=DEV),
                                 cu_seqlens=torch.tensor([0, n], dtype=torch.int32, device=DEV))
            taken = eng.model._takes_short(ids[:n].to(DEV), batch)
            out.append(eng.model.forward_prefill(ids[:n].to(DEV), batch).double())
            eng.kv.free_sequence(s)
        return out, taken

    from kllms_amd.models.llama import ForwardBatch
    with torch.inference_mode():
        want, taken = run()
        assert taken
        for layer in eng.model.layers:
            m = {"embed_tokens": eng.model.embed_tokens, "bias": layer.self_attn.qkv_proj}.get(which)
            m = m if m is not None else getattr(layer.self_attn if which[:2] in ("qk", "o_") else layer.mlp, which)
            name = "bias" if which == "bias" else "weight"
            w = getattr(m, name).data
            if how == "transposed":
                w = torch.stack((w, w), -1)[..., 0] if w.dim() == 1 else w.t().contiguous().t()
            elif how == "off 16 bytes":
                w = w.new_empty(w.numel() + 1)[1:].view_as(w).copy_(w)
            else:
                w = w.as_subclass(_Tagged)
            setattr(m, name, torch.nn.Parameter(w, requires_grad=False))
        got, taken = run()
    assert not taken
    for a, b in zip(got, want):
        assert (a - b).norm() <= 0.05 * b.norm()      # bf16 through two layers, two sets of kernels


@pytest.mark.parametrize("tokens", [40, 200])
def test_a_prompt_with_an_id_outside_the_vocabulary_is_refused(tokens):
    """In the call, each time, and nothing of it is kept for other prompts."""
    from kllms_amd.engine.config import EngineConfig
    from kllms_amd.engine.engine import GenRequest, LLMEngine
    from kllms_amd.engine.sampling import SamplingParams

    eng = LLMEngine(EngineConfig(model="mid-llama", max_kv_blocks=128, use_hip_graphs=False, seed=3, prefix_cache_min_tokens=16))
    ids = torch.randint(0, 2000, (tokens,), generator=torch.Generator().manual_seed(1)).tolist()
    good = [GenRequest(prompt_ids=ids, n=1, sampling=SamplingParams(temperature=0.0, max_tokens=4))]
    bad = [GenRequest(prompt_ids=ids[:5] + [eng.arch.vocab_size] + ids[6:], n=1,
                      sampling=SamplingParams(temperature=0.0, max_tokens=4))]
    for _ in range(2):
        with pytest.raises(IndexError, match="outside the vocabulary"):
            eng.generate(bad)
        assert not eng.prefix_cache.match(bad[0].prompt_ids, 16)
        assert len(eng.generate(good)[0].streams[0].token_ids) == 4


@pytest.mark.parametrize("tokens", [1, 100, 300])
def test_prompts_look_their_ids_up_in_the_embedding(tokens, monkeypatch):
    """Which refuses an id without a row in the call; steps on the paged cache report it."""
    from kllms_amd.engine.config import EngineConfig
    from kllms_amd.engine.engine import LLMEngine
    from kllms_amd.models.llama import ForwardBatch

    eng = LLMEngine(EngineConfig(model="mid-llama", max_kv_blocks=128, use_hip_graphs=False, seed=3))
    seen = []
    looked_up = torch.nn.functional.embedding
    monkeypatch.setattr(torch.nn.functional, "embedding", lambda i, *a: (seen.append(i.numel()), looked_up(i, *a))[1])
    s = eng.kv.alloc_sequence(tokens)
    batch = ForwardBatch(mode="prefill", positions=torch.arange(tokens, device=DEV), kv_caches=eng.kv.layer_caches(),
                         slot_mapping=torch.tensor(eng.kv.prefill_slot_mapping(s), device=DEV),
                         cu_seqlens=torch.tensor([0, tokens], dtype=torch.int32, device=DEV))
    ids = torch.arange(tokens, device=DEV)
    with torch.inference_mode():
        assert eng.model._takes_short(ids, batch)
        eng.model.forward_prefill(ids, batch)
        assert seen == [tokens]

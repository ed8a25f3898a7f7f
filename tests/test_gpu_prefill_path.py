"""Causal prefill attention, packed and against the paged cache, against float64 at the edges of its tiles."""

import math

import pytest
import torch

from kllms_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = 128


def causal64(q, k, v, scale, first):
    """Rows first.. of one sequence; also the bound sum p |v| of what rounding P to bf16 can move."""
    T, H, _ = q.shape
    rep = H // k.shape[1]
    k, v, q = (t.double().to(DEV) for t in (k, v, q))
    hide = torch.arange(k.shape[0], device=DEV) > torch.arange(first, first + T, device=DEV).unsqueeze(1)
    out, size = [], []
    for h in range(H):
        p = torch.softmax((q[:, h] @ k[:, h // rep].t() * scale).masked_fill(hide, -torch.inf), -1)
        out.append(p @ v[:, h // rep])
        size.append(p @ v[:, h // rep].abs())
    return torch.stack(out, 1), torch.stack(size, 1)


def check(got, ref, size, p=2 ** -8):
    # P in bf16 (2^-9 of each term) with a fast exponential, the result rounded to bf16. Against the cache P is fp32 or
    # two bf16 parts (2^-17 of each term), and scores are sums of 128 products in 32 bits
    err = (got.double() - ref).abs()
    assert (err <= p * size + 2 ** -8 * ref.abs() + 1e-6).all(), float((err - p * size - 2 ** -8 * ref.abs()).max())


@pytest.mark.parametrize("H,G", [(4, 4), (8, 2), (32, 8), (7, 1)])
@pytest.mark.parametrize("lens", [[1], [31, 32, 33], [63, 64, 65, 0, 1], [255, 256, 257], [700, 5, 513]])
@pytest.mark.parametrize("scale", [D ** -0.5, -0.3])
def test_packed(H, G, lens, scale):
    g = torch.Generator().manual_seed(sum(lens) + H)
    T = sum(lens)
    qkv = torch.randn(T, H + 2 * G, D, generator=g).bfloat16().to(DEV)      # the fused projection's layout
    q, k, v = qkv.split([H, G, G], 1)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(DEV)
    out = ops.attn_prefill_varlen(q, k, v, cu, scale)
    plan = ops.prefill_plan(cu, T)
    assert torch.equal(out, ops.attn_prefill_varlen(q, k, v, cu, scale, plan))
    r = 0
    for n in lens:
        if n:
            check(out[r:r + n], *causal64(q[r:r + n].cpu(), k[r:r + n].cpu(), v[r:r + n].cpu(), scale, 0))
        r += n


def test_plan_covers_many_sequences():
    g = torch.Generator().manual_seed(1)
    lens = torch.randint(0, 700, (1500,), generator=g)
    cu = torch.cat([torch.zeros(1, dtype=torch.long), lens.cumsum(0)]).to(torch.int32).to(DEV)
    start, length, first = ops.prefill_plan(cu, int(lens.sum())).cpu().long()
    live = length > 0
    got = sorted(zip(start[live].tolist(), length[live].tolist(), first[live].tolist()))
    want = sorted((int(s), int(n), f) for s, n in zip(cu.cpu()[:-1], lens) for f in range(0, int(n), 256))
    assert got == want


# few: four waves to a row tile, at the edges of their tiles and stages of keys, of the row tiles and of the groups
@pytest.mark.parametrize("few", [False, True])
@pytest.mark.parametrize("H,G,BS", [(8, 2, 16), (32, 8, 16), (4, 4, 5), (4, 2, 1)])
@pytest.mark.parametrize("segs", [[(0, 40)], [(17, 32), (1000, 300), (3, 1), (5, 2)], [(255, 1), (64, 257), (0, 31), (700, 33)],
                                  [(576, 32), (95, 64), (0, 33), (1151, 1), (1, 63)], [(480, 32), (2000, 47)],
                                  [(600, 65), (31, 128), (1, 129), (128, 192), (97, 95)]])
def test_segments_against_cache(H, G, BS, segs, few):
    g = torch.Generator().manual_seed(sum(n for _, n in segs) + H)
    NB = sum((s + n + BS - 1) // BS for s, n in segs) + 2
    perm = torch.randperm(NB, generator=g).tolist()
    kc, vc = (torch.randn(NB, G, BS, D, generator=g).bfloat16() for _ in range(2))
    width = max((s + n + BS - 1) // BS for s, n in segs)
    bt = torch.zeros(len(segs), width, dtype=torch.int32)
    for i, (s, n) in enumerate(segs):
        m = (s + n + BS - 1) // BS
        bt[i, :m] = torch.tensor([perm.pop() for _ in range(m)], dtype=torch.int32)
    T = sum(n for _, n in segs)
    q = torch.randn(T, H + 1, D, generator=g).bfloat16().to(DEV)[:, :H]
    plan, short = ops.paged_prefill_plan(segs, DEV, *([64] if few else []))
    row_seg = torch.tensor([i for i, (_, n) in enumerate(segs) for _ in range(n)])
    ctx = torch.tensor([s + j + 1 for s, n in segs for j in range(n)], dtype=torch.int32)
    if plan is None:
        return
    out = ops.attn_segments_paged(q, kc.to(DEV), vc.to(DEV), bt[row_seg].to(DEV), ctx.to(DEV), D ** -0.5, plan, short,
                                  bt.to(DEV), torch.tensor([s for s, _ in segs], dtype=torch.int32).to(DEV))
    r = 0
    for i, (s, n) in enumerate(segs):
        at = torch.arange(s + n)
        blk = bt[i].long()[at // BS]
        check(out[r:r + n], *causal64(q[r:r + n].cpu(), kc[blk, :, at % BS], vc[blk, :, at % BS], D ** -0.5, s), 2 ** -14)
        r += n


@pytest.mark.parametrize("rows", [[40, 20], [150, 1, 33], [300]])
def test_step_segments_matches_row_by_row(rows, cached=37):
    """Portions behind a cached head through LLMEngine.step_segments, every row's logits, against the same step with
    each row attending alone."""
    from kllms_amd.engine.config import EngineConfig
    from kllms_amd.engine.engine import LLMEngine

    eng = LLMEngine(EngineConfig(model="mid-llama", max_kv_blocks=512, use_hip_graphs=False, seed=3))
    g = torch.Generator().manual_seed(sum(rows))

    def step(alone):
        eng.model._planned = (lambda ids, batch: batch) if alone else type(eng.model)._planned.__get__(eng.model)
        seqs = [eng.open_sequence() for _ in rows]
        heads = [torch.randint(0, 2000, (cached + 11 * i,), generator=torch.Generator().manual_seed(i)).tolist()
                 for i in range(len(rows))]
        eng.step_segments([(s, h, []) for s, h in zip(seqs, heads)])
        out = eng.step_segments([(s, t, list(range(len(t)))) for s, t in zip(seqs, toks)])
        for s in seqs:
            eng.kv.free_sequence(s)
        return out

    toks = [torch.randint(0, 2000, (n,), generator=g).tolist() for n in rows]
    a, b = step(False), step(True)
    assert float(((a - b).norm(dim=-1) / b.norm(dim=-1)).max()) < 0.03     # bf16 through two layers


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("T,H,G,BS", [(1, 4, 2, 16), (33, 7, 1, 5), (257, 32, 8, 16)])
def test_rope_store_matches_the_two_kernels(T, H, G, BS, fp8):
    g = torch.Generator().manual_seed(T)
    qkv = torch.randn(T, H + 2 * G, D, generator=g).bfloat16().to(DEV)
    NB = (T + BS - 1) // BS + 1
    slots = torch.randperm(NB * BS, generator=g)[:T].to(DEV)
    pos = torch.randint(0, 300, (T,), generator=g).to(DEV)
    ang = torch.arange(300).unsqueeze(1) * 10000.0 ** (-torch.arange(0, D, 2) / D)
    cs = torch.cat([ang.cos(), ang.sin()], 1).to(DEV)
    kind = torch.float8_e4m3fn if fp8 else torch.bfloat16
    got = []
    for fused in (True, False):
        rows = qkv.clone()
        q, k, v = rows.split([H, G, G], 1)
        kc, vc = (torch.zeros(NB, G, BS, D, device=DEV, dtype=kind) for _ in range(2))
        ks, vs = (torch.ones(NB, G, BS, device=DEV) for _ in range(2)) if fp8 else (None, None)
        if fused:
            ops.rope_store(q, k, v, pos, cs, kc, vc, slots, ks, vs)
        else:
            ops.rope_inplace(q, k, pos, cs)
            ops.store_kv(k, v, kc, vc, slots, ks, vs)
        got.append((rows, kc.view(torch.uint8), vc.view(torch.uint8), ks, vs))
    a, b = got
    # the same products, which one of the two may contract into a fused multiply-add: a last place of bf16 in the rows
    # (2^-8 of the larger term), the same bytes of V
    big = torch.maximum(qkv.float().abs(), qkv.float().abs().roll(64, -1))
    assert ((a[0].float() - b[0].float()).abs() <= 2 ** -7 * big).all()
    assert float((a[0] != b[0]).float().mean()) < 0.01
    assert torch.equal(a[2], b[2])
    assert float((a[1] != b[1]).float().mean()) < 0.02
    if fp8:
        assert torch.equal(a[4], b[4]) and torch.allclose(a[3], b[3], rtol=2 ** -7)


@pytest.mark.parametrize("H,I,counts", [(64, 64, [1, 0, 2]), (320, 192, [0, 255, 256, 257, 1]), (512, 448, [31, 512, 0, 0, 33])])
def test_mixture_products_against_float64(H, I, counts):
    E, k = len(counts), 2
    g = torch.Generator().manual_seed(H)
    T = sum(counts)
    first = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])[torch.randperm(T, generator=g)]
    topi = torch.stack([first, (first + 1) % E], 1).to(DEV)
    topw = torch.rand(T, k, generator=g).to(DEV)
    x = torch.randn(T, H, generator=g).bfloat16().to(DEV)
    wg = (torch.randn(E, 2 * I, H, generator=g) * H ** -0.5).bfloat16().to(DEV)
    wd = (torch.randn(E, H, I, generator=g) * I ** -0.5).bfloat16().to(DEV)
    ids, pos, offsets = ops.moe_sort(topi, E)
    assert offsets.tolist() == [0] + torch.bincount(topi.flatten(), minlength=E).cumsum(0).tolist()
    assert torch.equal(ids[pos.view(T, k).long()], torch.arange(T, device=DEV, dtype=ids.dtype).unsqueeze(1).expand(T, k))
    act = torch.empty(T * k, I, device=DEV, dtype=x.dtype)
    y = torch.empty(T * k, H, device=DEV, dtype=x.dtype)
    ops.moe_gateup(act, x, wg, ids, offsets, x)
    ops.moe_down(y, act, wd, offsets)
    got = ops.moe_combine_rows(y, topw, pos)
    # act, y and the result are each rounded to bf16 (2^-9); the sums and silu in 32 bits stay far below that
    ref, lim = torch.zeros(T, H, device=DEV, dtype=torch.float64), torch.zeros(T, H, device=DEV, dtype=torch.float64)
    for j in range(k):
        for e in range(E):
            rows = (topi[:, j] == e).nonzero()[:, 0]
            gate, up = (x[rows].double() @ wg[e].double().t().contiguous()).split([I, I], 1)
            a = torch.nn.functional.silu(gate) * up
            ye = a @ wd[e].double().t().contiguous()
            w = topw[rows, j].double().unsqueeze(1)
            ref[rows] += w * ye
            lim[rows] += w * 2 ** -8 * (a.abs() @ wd[e].double().abs().t().contiguous() + ye.abs())
    assert ((got.double() - ref).abs() <= lim + 2 ** -8 * ref.abs() + 1e-5).all()


@pytest.mark.parametrize("H,I,counts", [
    (256, 1088, [32, 33, 64, 65, 80, 81, 96, 97, 128, 129]),      # one column tile, 17 stages
    (1088, 2112, [20, 130, 0, 150, 260, 385, 1]),                 # five column tiles, the last of 64; 33 stages
    (256, 2624, [32, 33, 64, 65, 80, 81, 96, 97, 128, 129]),      # the same with shares: 41 stages in four
    (1088, 2624, [20, 130, 0, 150, 260, 385, 1]),
    (2048, 2624, [700, 600, 600, 600, 600, 600, 600, 600]),       # 42 tiles an XCD: a whole round, and ten in three shares
    (320, 64, [1] * 60 + [0] * 3 + [2, 300, 0, 1] + [3] * 63),    # experts of more than one walk of a wave's lanes
    (64, 2624, [5] * 64 + [0] * 64 + [9]),
    (320, 320, [96, 96, 97, 112, 112, 113, 224, 224, 225]),      # tiles of 224 rows, and their edges in one and two parts
    (64, 2624, [96, 96, 97, 112, 112, 113, 224, 224, 225]),
])
def test_mixture_products_at_the_edges_of_row_tiles(H, I, counts):
    # expert e gets counts[e] + counts[e - 1] rows: 64, 128, 160, 192, 224 and 256 a tile, and parts of two and three tiles
    test_mixture_products_against_float64(H, I, counts)


@pytest.mark.parametrize("counts", [[1, 64, 0], [65, 130, 200], [225, 0, 600], [0, 9000, 3000]])
def test_mixture_products_of_weights_beyond_the_cache(counts):
    """How W is loaded, which its size and the rows of an expert decide, is not to be seen in the results: the first experts
    alone give the same bits as with all others behind them, whose products have more than 320 MB of W to read. The last one's
    experts have too many rows for the difference."""
    E, H, I, few = 21, 4096, 2048, len(counts)
    g = torch.Generator(device=DEV).manual_seed(sum(counts))
    wg = torch.empty(E, 2 * I, H, device=DEV, dtype=torch.bfloat16).normal_(0, H ** -0.5, generator=g)
    wd = torch.empty(E, H, I, device=DEV, dtype=torch.bfloat16).normal_(0, I ** -0.5, generator=g)
    S = sum(counts)
    x = torch.randn(S, H, device=DEV, generator=g).bfloat16()
    ids = torch.randperm(S, device=DEV, generator=g).to(torch.int32)
    ends = torch.tensor([0] + counts).cumsum(0)
    got = []
    for n in (few, E):
        offsets = torch.cat([ends, ends[-1:].expand(n - few)]).to(device=DEV, dtype=torch.int32)
        act, y = torch.empty(S, I, device=DEV, dtype=x.dtype), torch.empty(S, H, device=DEV, dtype=x.dtype)
        ops.moe_gateup(act, x, wg[:n], ids, offsets, x)
        ops.moe_down(y, act, wd[:n], offsets)
        got.append((act, y))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert torch.isfinite(got[0][1]).all() and got[0][1].abs().amax(1).gt(0).all()


@pytest.mark.parametrize("E", [1, 8, 128, 1024, 1025, 4096])
@pytest.mark.parametrize("T,k", [(1, 1), (63, 2), (65, 3), (1025, 2), (9001, 2)])
def test_sort_of_the_mixture_keeps_the_order_of_the_pairs(T, k, E):
    """Places of one expert in the order of the pairs, so that a row is in the same tile, with the same order of its sums,
    in every call; an expert out of range has no place."""
    topi = torch.randint(-1, E + 1, (T, k), generator=torch.Generator().manual_seed(T + E))
    ids, pos, offsets = ops.moe_sort(topi.to(DEV), E)
    flat = topi.flatten()
    order = torch.sort(torch.where((flat >= 0) & (flat < E), flat, E), stable=True).indices
    n = int(((flat >= 0) & (flat < E)).sum())
    assert offsets.tolist() == [0] + torch.bincount(flat[order[:n]], minlength=E).cumsum(0).tolist()
    assert torch.equal(ids[:n].cpu().long(), order[:n] // k)
    want = torch.full((T * k,), -1)
    want[order[:n]] = torch.arange(n)
    assert torch.equal(pos.flatten().cpu().long(), want)


def test_mixture_products_of_views_off_16_bytes():
    def off(*shape):
        n = torch.Size(shape).numel()
        return torch.randn(n + 1, device=DEV).bfloat16()[1:].view(shape)

    T, H, I, E = 70, 128, 192, 2
    x, wg, wd = off(T, H), off(E, 2 * I, H), off(E, H, I)
    ids = torch.arange(T, device=DEV, dtype=torch.int32)
    offsets = torch.tensor([0, 30, T], device=DEV, dtype=torch.int32)
    act, y = off(T, I), off(T, H)
    ops.moe_gateup(act, x, wg, ids, offsets, x)
    ops.moe_down(y, act, wd, offsets)
    act2, y2 = torch.empty(T, I, device=DEV, dtype=x.dtype), torch.empty(T, H, device=DEV, dtype=x.dtype)
    ops.moe_gateup(act2, x.clone(), wg.clone(), ids, offsets, x.clone())
    ops.moe_down(y2, act2, wd.clone(), offsets)
    assert torch.equal(act, act2) and torch.equal(y, y2)


@pytest.mark.parametrize("which", ["q", "kv", "all"])
@pytest.mark.parametrize("stride,at", [(0, 1), (0, 4), (4, 0), (12, 8), (2, 3)])      # elements between rows' ends, and before the first
def test_prompt_attention_of_rows_off_16_bytes(which, stride, at):
    """Contiguous rows that begin off 16 bytes, and rows whose stride takes them off: the copies' results, bit by bit, in whole
    prompts, in tables of pieces and against a paged cache."""
    T, H, G, BS = 300, 4, 2, 16
    g = torch.Generator(device=DEV).manual_seed(stride + at)
    q, k, v = (torch.randn(T, h, D, generator=g, device=DEV).bfloat16() for h in (H, G, G))

    def off(t):
        row = t[0].numel() + stride
        flat = torch.zeros(T * row + at, device=DEV, dtype=t.dtype)[at:]
        return flat.as_strided((T, t.shape[1], D), (row, D, 1)).copy_(t)

    moved = [off(t) if which == "all" or (which == "q") == (t is q) else t for t in (q, k, v)]
    cu = torch.tensor([0, 41, T], dtype=torch.int32, device=DEV)
    pieces = ops.dense_tile_groups([(0, 41), (41, T - 41)], torch.device(DEV))
    got = []
    for a, b, c in ((q, k, v), moved):
        out = torch.zeros_like(q)
        ops.attn_varlen_mfma(out, a, b, c, *pieces, 0.1)
        got.append((ops.attn_prefill_varlen(a, b, c, cu, 0.1), out))
    assert all(torch.equal(a, b) for a, b in zip(*got)) and torch.isfinite(got[0][1]).all()
    NB = (T + BS - 1) // BS
    cache = [torch.randn(NB, G, BS, D, generator=g, device=DEV).bfloat16() for _ in range(2)]
    other = [torch.zeros(t.numel() + at, device=DEV, dtype=t.dtype)[at:].view_as(t).copy_(t) for t in cache]
    plan, _ = ops.paged_prefill_plan([(0, T)], DEV)
    tables, pos = torch.arange(NB, dtype=torch.int32, device=DEV).view(1, NB), torch.zeros(1, dtype=torch.int32, device=DEV)
    a = ops.attn_segments_paged(q, *cache, None, None, 0.1, plan, [], tables, pos)
    b = ops.attn_segments_paged(moved[0], *(cache if which == "q" else other), None, None, 0.1, plan, [], tables, pos)
    assert torch.equal(a, b)


@pytest.mark.parametrize("T,H", [(65535, 8), (65536, 64), (70001, 2056)])
def test_mixture_of_more_rows_than_a_grid_has_in_y(T, H):
    g = torch.Generator(device=DEV).manual_seed(T)
    E, k = 8, 2
    topi = torch.rand(T, E, generator=g, device=DEV).topk(k, -1).indices
    topw = torch.rand(T, k, generator=g, device=DEV)
    ids, pos, offsets = ops.moe_sort(topi, E)
    assert torch.equal(ids[pos.long()], torch.arange(T, device=DEV, dtype=ids.dtype).unsqueeze(1).expand(T, k))
    y = torch.randn(T * k, H, generator=g, device=DEV).bfloat16()
    got = ops.moe_combine_rows(y, topw, pos)
    rows = y[pos.long()].float()
    ref = (rows * topw.unsqueeze(-1)).sum(1)
    # two products and a sum in fp32, one rounding to bf16 (2^-9)
    lim = 2 ** -8 * ref.abs() + 2 ** -22 * (rows.abs() * topw.unsqueeze(-1)).sum(1)
    assert ((got.float() - ref).abs() <= lim).all()


@pytest.mark.parametrize("n", [65535, 66000])
def test_more_prompts_than_a_grid_has_in_y(n):
    """As many groups as sequences: the same rows attended in two calls."""
    g = torch.Generator(device=DEV).manual_seed(n)
    lens = torch.randint(1, 4, (n,), generator=g, device=DEV)
    cu = torch.cat([lens.new_zeros(1), lens.cumsum(0)]).to(torch.int32)
    T, cut = int(cu[-1]), int(cu[30000])
    qkv = torch.randn(T, 3, D, generator=g, device=DEV).bfloat16()
    q, k, v = qkv.split([1, 1, 1], 1)
    out = ops.attn_prefill_varlen(q, k, v, cu, 0.1)
    halves = [ops.attn_prefill_varlen(q[a:b], k[a:b], v[a:b], c, 0.1)
              for a, b, c in ((0, cut, cu[:30001]), (cut, T, cu[30000:] - cut))]
    assert torch.equal(out, torch.cat(halves))


def test_more_segments_than_a_grid_has_in_y():
    g = torch.Generator(device=DEV).manual_seed(3)
    n, rows, NB = 65600, 32, 8
    kc, vc = (torch.randn(NB, 1, 32, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    tables = torch.randint(0, NB, (n, 1), generator=g, device=DEV, dtype=torch.int32)
    pos = torch.zeros(n, dtype=torch.int32, device=DEV)
    q = torch.randn(n * rows, 1, D, generator=g, device=DEV).bfloat16()
    plan, short = ops.paged_prefill_plan([(0, rows)] * n, DEV)
    assert plan.groups.shape[1] == n and not short
    out = ops.attn_segments_paged(q, kc, vc, None, None, 0.1, plan, short, tables, pos)
    for lo, hi in ((0, 200), (n - 200, n)):
        part, _ = ops.paged_prefill_plan([(0, rows)] * (hi - lo), DEV)
        want = ops.attn_segments_paged(q[lo * rows:hi * rows], kc, vc, None, None, 0.1, part, [], tables[lo:hi].contiguous(),
                                       pos[lo:hi])
        assert torch.equal(out[lo * rows:hi * rows], want)


@pytest.mark.parametrize("rows", [32, 65, 300])
@pytest.mark.parametrize("at", [1, 40, 100])          # the second key beside the first, in the other half, in another tile
@pytest.mark.parametrize("group", [64, 256])
def test_segments_against_cache_keep_32_bit_probabilities(at, rows, group):
    """Two keys of nearly the same score and V of opposite sign: the result is the difference of their probabilities,
    2^-14 to 2^-8 of them, and an error of P shows in it at full size."""
    start, G, rep, BS = 128, 2, 4, 16
    L, g = start + rows, torch.Generator().manual_seed(rows + at)
    NB = (L + BS - 1) // BS
    k, v = torch.zeros(NB * BS, G, D), torch.zeros(NB * BS, G, D)
    k[..., 0] = -256.0
    k[0, :, 0], k[at, :, 0], k[at, :, 1] = 1.0, 1.0, -(2.0 ** -4)
    v[0] = torch.rand(G, D, generator=g).bfloat16().float() + 0.5
    v[0] = v[0].bfloat16().float()
    v[at] = -v[0]
    q = torch.zeros(rows, G * rep, D)
    q[..., 0] = 1.0
    q[..., 1] = torch.randint(1, 65, (rows, G * rep), generator=g) * 2.0 ** -10
    cache = [t.view(NB, BS, G, D).transpose(1, 2).contiguous().bfloat16().to(DEV) for t in (k, v)]
    bt = torch.arange(NB, dtype=torch.int32, device=DEV).view(1, NB)
    plan, short = ops.paged_prefill_plan([(start, rows)], DEV, group)
    assert plan is not None and not short
    out = ops.attn_segments_paged(q.bfloat16().to(DEV), *cache, None, None, 1.0, plan, [], bt,
                                  torch.tensor([start], dtype=torch.int32, device=DEV))
    p = torch.exp(-(q[..., 1].double() * 2.0 ** -4)).unsqueeze(-1)
    size = v[0].double().repeat_interleave(rep, 0)
    ref = (1 - p) / (1 + p) * size
    # the result's rounding to bf16, and four of 2^-24 in P and its sum
    assert ((out.double().cpu() - ref).abs() <= 2 ** -8 * ref.abs() + 4 * 2 ** -24 * size).all()


@pytest.mark.parametrize("H,G", [(4, 4), (8, 2)])
@pytest.mark.parametrize("seed", range(4))
def test_packed_tiles_in_any_order(H, G, seed):
    """Tile tables of attn_varlen_mfma that dense_tile_groups does not make: a group's waves take tiles from anywhere in
    their piece, with idle ones between them, and rows that begin between tiles."""
    g = torch.Generator().manual_seed(seed)
    pieces = [(0, 300), (300, 31), (331, 700)]
    T = 1031
    q, k, v = (torch.randn(T, n, D, generator=g).bfloat16().to(DEV) for n in (H, G, G))
    gs, gl, gq, want = [], [], [], torch.zeros(T, dtype=torch.bool)
    for row0, n in pieces:
        tiles = [t for t in torch.randperm((n + 31) // 32, generator=g).tolist() if t % 5 != seed]
        first = [t * 32 for t in tiles] + ([n - 7, 3] if n > 40 else [])
        for f in first:
            want[row0 + f:row0 + min(n, f + 32)] = True
        while first:
            slots = [-1] * 8
            for w in torch.randperm(8, generator=g).tolist()[:5]:
                if first:
                    slots[w] = first.pop()
            gs.append(row0), gl.append(n), gq.extend(slots)
    gs.append(0), gl.append(300), gq.extend([-1] * 8)               # a group without work
    t = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    out = torch.full((T, H, D), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.attn_varlen_mfma(out, q, k, v, t(gs), t(gq), t(gl), D ** -0.5)
    for row0, n in pieces:
        at = torch.arange(row0, row0 + n)[want[row0:row0 + n]]
        ref, size = causal64(q[row0:row0 + n].cpu(), k[row0:row0 + n].cpu(), v[row0:row0 + n].cpu(), D ** -0.5, 0)
        check(out[at.to(DEV)], ref[(at - row0).to(DEV)], size[(at - row0).to(DEV)])
    assert (out[~want.to(DEV)] == 7.0).all()


def test_rope_store_takes_the_head_of_longer_rows():
    """Positions and slots of a larger buffer: its first T entries, as the two kernels take them; too few are refused."""
    T, H, G = 40, 4, 2
    g = torch.Generator(device=DEV).manual_seed(1)
    rows = torch.randn(T, H + 2 * G, D, generator=g, device=DEV).bfloat16()
    pos, slots = torch.arange(T + 9, device=DEV), torch.randperm(64, generator=g, device=DEV)
    cs = torch.randn(64, D, generator=g, device=DEV)
    got = []
    for p, s in ((pos, slots), (pos[:T].clone(), slots[:T].clone())):
        q, k, v = rows.clone().split([H, G, G], 1)
        kc, vc = (torch.zeros(4, G, 16, D, device=DEV, dtype=torch.bfloat16) for _ in range(2))
        ops.rope_store(q, k, v, p, cs, kc, vc, s)
        got.append((q.clone(), k.clone(), kc, vc))
    assert all(torch.equal(a, b) for a, b in zip(*got))
    q, k, v = rows.split([H, G, G], 1)
    with pytest.raises(RuntimeError):
        ops.rope_store(q, k, v, pos[:T - 1], cs, kc, vc, slots)


@pytest.mark.parametrize("rows", [[40, 20], [150, 1, 33], [300]])
def test_step_segments_together_matches_row_by_row(rows, monkeypatch):
    """The step of test_step_segments_matches_row_by_row with its long portions on the paged prefill kernel, which the
    rule on rows and keys would not choose for a model of two kv heads."""
    from kllms_amd.models.llama import LlamaForCausalLM

    monkeypatch.setattr(ops, "PAGED_PREFILL_WORK", 0)
    plans, make = [], LlamaForCausalLM._planned

    def planned(self, ids, batch):
        batch = make(self, ids, batch)
        plans.append((batch.plans or {}).get("paged"))
        return batch

    monkeypatch.setattr(LlamaForCausalLM, "_planned", planned)
    test_step_segments_matches_row_by_row(rows)
    assert plans[-1] is not None and plans[-1][0] is not None


# group: the size that the rules choose
@pytest.mark.parametrize("rows,cached,group", [([400], 37, 256), ([150] * 3, 300, 256), ([400], 600, 64), ([129, 1, 300, 20], 1000, 64)])
def test_step_segments_of_either_group_size_match_row_by_row(rows, cached, group, monkeypatch):
    from kllms_amd.models.llama import LlamaForCausalLM

    plans, make = [], LlamaForCausalLM._planned

    def planned(self, ids, batch):
        batch = make(self, ids, batch)
        plans.append((batch.plans or {}).get("paged"))
        return batch

    monkeypatch.setattr(LlamaForCausalLM, "_planned", planned)
    test_step_segments_matches_row_by_row(rows, cached)
    assert plans[-1][0].rows == group


@pytest.mark.parametrize("T", [1, 15, 16, 17, 255, 256, 257, 4113])
@pytest.mark.parametrize("E,k,H", [(1, 1, 64), (2, 2, 64), (8, 2, 4096), (16, 3, 1088), (17, 8, 4160), (32, 8, 2048)])
def test_router_against_torch_and_the_sort(T, E, k, H):
    """Whole-number logits are exact in every order of the sums, so that choices, ties among them (the lowest expert
    first) and places are compared to the last; the weights are fp32 quotients of exponentials: a few places of 2^-24."""
    g = torch.Generator().manual_seed(T * 37 + E)
    x = (torch.rand(T, H, generator=g) < 16 / H).float() * torch.randint(-3, 4, (T, H), generator=g)
    gate = torch.randint(-1, 2, (E, H), generator=g).float()
    z = (x @ gate.t()).bfloat16().float()
    want = torch.sort(-z, dim=1, stable=True).indices[:, :k]
    p = torch.softmax(z.double(), 1).gather(1, want)
    if T > 3:
        x[3] = math.nan
    wide = torch.zeros(T, H + 8, dtype=torch.bfloat16)     # rows of a wider matrix
    wide[:, :H] = x
    topw, topi, ids, pos, offsets, cleared = ops.router_top(wide.to(DEV)[:, :H], gate.bfloat16().to(DEV), k, True)
    plain = [t for t in range(T) if t != 3 or T <= 3]
    assert torch.equal(topi.cpu()[plain].long(), want[plain])
    assert torch.allclose(topw.cpu().double()[plain], (p / p.sum(1, keepdim=True))[plain], rtol=2 ** -20, atol=0)
    if T > 3:
        assert topw[3].isnan().all() and sorted(set(topi[3].tolist())) == sorted(topi[3].tolist())
        assert 0 <= int(topi.min()) and int(topi.max()) < E
    for a, b in zip((ids, pos, offsets), ops.moe_sort(topi, E)):
        assert torch.equal(a, b)
    assert not cleared.any()


def test_router_leaves_other_calls_to_torch():
    x, gate = torch.randn(40, 128, device=DEV).bfloat16(), torch.randn(8, 128, device=DEV).bfloat16()
    assert ops.router_top(x, gate, 2, False) is not None
    assert ops.router_top(x.float(), gate.float(), 2, False) is None
    assert ops.router_top(x, gate, 9, False) is None
    assert ops.router_top(x[:, :96].contiguous(), gate[:, :96].contiguous(), 2, False) is None
    assert ops.router_top(x.t()[:40, :], gate, 2, False) is None
    assert ops.router_top(x, torch.randn(33, 128, device=DEV).bfloat16(), 2, False) is None
    assert ops.router_top(x, gate.requires_grad_(), 2, False) is None
    with torch.autocast("cuda", torch.float16):
        assert ops.router_top(x, gate.detach(), 2, False) is None


def test_mixture_layer_with_a_hooked_router():
    """The layer through the router's kernel and through the module, whose hook must run: the same up to the choices, which
    whole-number logits make the same."""
    from kllms_amd.engine.config import ModelArchConfig
    from kllms_amd.models.mixtral import MixtralMoE
    from kllms_amd.parallel.tp import ParallelContext
    cfg = ModelArchConfig(arch="mixtral", vocab_size=64, hidden_size=256, intermediate_size=128, num_layers=1, num_heads=2,
                          num_kv_heads=1, num_experts=8, num_experts_per_tok=2)
    g = torch.Generator().manual_seed(5)
    with torch.device(DEV):
        moe = MixtralMoE(cfg, ParallelContext(), torch.bfloat16)
    with torch.no_grad():
        moe.gate.weight.copy_(torch.randint(-1, 2, moe.gate.weight.shape, generator=g))
        for p in (moe.w_gate_up, moe.w_down):
            p.copy_(torch.randn(p.shape, generator=g) * 0.05)
    for T in (7, 64, 65, 300):
        x = (torch.randint(-2, 3, (T, 256), generator=g) * (torch.rand(T, 256, generator=g) < 0.05)).bfloat16().to(DEV)
        got = moe(x)
        seen = []
        h = moe.gate.register_forward_hook(lambda m, i, o: seen.append(o.shape))
        want = moe(x)
        h.remove()
        assert seen == [(T, 8)]
        # weights apart by fp32 rounding, the result rounded to bf16 once (2^-9)
        assert torch.allclose(got.float(), want.float(), rtol=2 ** -7, atol=1e-4 * float(want.float().abs().max()))


@pytest.mark.parametrize("T", [1, 2, 16, 32])
@pytest.mark.parametrize("H,I,E,k,how", [(512, 1024, 8, 2, ""), (64, 64, 4, 1, ""), (256, 192, 32, 8, ""), (512, 2624, 8, 2, ""),
                                         (128, 64, 40, 2, ""), (128, 96, 4, 2, "size"), (256, 128, 8, 2, "rows"),
                                         (256, 128, 8, 2, "transposed"), (256, 128, 8, 2, "gradient")])
def test_mixture_layer_of_few_rows(T, H, I, E, k, how):
    """As grouped products, and as batched ones where those do not take the call, against float64 on the layer's routing."""
    from kllms_amd.engine.config import ModelArchConfig
    from kllms_amd.models.mixtral import MixtralMoE
    from kllms_amd.parallel.tp import ParallelContext
    cfg = ModelArchConfig(arch="mixtral", vocab_size=64, hidden_size=H, intermediate_size=I, num_layers=1, num_heads=2,
                          num_kv_heads=1, num_experts=E, num_experts_per_tok=k)
    g = torch.Generator(device=DEV).manual_seed(T + H + I)
    with torch.device(DEV):
        moe = MixtralMoE(cfg, ParallelContext(), torch.bfloat16)
    with torch.no_grad():
        for p in moe.parameters():
            p.copy_(torch.randn(p.shape, generator=g, device=DEV) * p.shape[-1] ** -0.5)
    x = torch.randn(T, H, generator=g, device=DEV).bfloat16()
    if how == "rows":
        x = torch.cat((x, x), 1)[:, :H] if T > 1 else torch.stack((x, x), -1)[..., 0]
    elif how == "transposed":
        moe.w_down.data = moe.w_down.data.transpose(1, 2).contiguous().transpose(1, 2)
    elif how == "gradient":
        x.requires_grad_()
    assert moe._takes_grouped(x) == (how == "")
    got = moe(x)
    if how == "gradient":
        got.float().sum().backward()
        assert x.grad.isfinite().all() and x.grad.norm() > 0
        x = x.detach()
    p = torch.softmax((x.double() @ moe.gate.weight.double().t().contiguous()).bfloat16().float(), -1)
    topw, topi = torch.topk(p, k, -1)
    sure = torch.topk(p, min(k + 1, E), -1)[0]
    sure = (sure[:, k - 1] > 1.02 * sure[:, k]) if E > k else torch.ones(T, dtype=torch.bool, device=DEV)
    topw = (topw / topw.sum(-1, keepdim=True)).double()
    want = torch.zeros(T, H, dtype=torch.float64, device=DEV)
    for t in range(T):
        for w, e in zip(topw[t], topi[t].tolist()):
            gate, up = (moe.w_gate_up[e].double() @ x[t].double()).chunk(2)
            want[t] += w * (moe.w_down[e].double() @ (torch.nn.functional.silu(gate) * up))
    # gate, up, act, each expert's row and the sum are rounded to bf16 (2^-9 each); rows whose choice is not a close one
    off = (got.double() - want).norm(dim=-1) / want.norm(dim=-1)
    assert sure.float().mean() >= 0.5 or T < 8
    assert (off[sure] <= 0.015).all()

"""The sliced sampler against the same draw in float64: slice edges, short
rows, ragged vocabularies, masks, boundary bins that outgrow the LDS list."""

import numpy as np
import pytest
import torch

from kllms_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def splitmix(x):
    with np.errstate(over="ignore"):
        x = x + np.uint64(0x9E3779B97F4A7C15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return x ^ (x >> np.uint64(31))


def gumbel(seed, step, V):
    """float64 Gumbel values of one row's counter-based draw (the uniform is formed in float32, as the kernel's)."""
    with np.errstate(over="ignore"):
        base = splitmix(np.uint64(seed) * np.uint64(0x9E3779B97F4A7C15) + np.uint64(step) * np.uint64(0xBF58476D1CE4E5B9))
    h = splitmix(base ^ np.arange(V, dtype=np.uint64)) >> np.uint64(40)
    u = (h + np.uint64(1)).astype(np.float32) * np.float32(1.0 / 16777217.0)
    return -np.log(-np.log(u.astype(np.float64)))


@pytest.mark.parametrize("mode", ["plain", "greedy", "masked", "top_k", "top_p", "both", "crowded"])
@pytest.mark.parametrize("B,V", [(1, 1), (2, 5), (3, 63), (1, 2047), (1, 2048), (2, 2049), (5, 8193), (33, 32000),
                                 (250, 4099), (3, 131071)])
def test_draw_matches_float64(B, V, mode):
    g = torch.Generator().manual_seed(V * 7 + B)
    logits = torch.randn(B, V, generator=g) * (0.01 if mode == "crowded" else 3.0)
    temp = torch.zeros(B) if mode == "greedy" else torch.rand(B, generator=g) * 0.8 + 0.4
    top_p = torch.full((B,), 0.8 if mode in ("top_p", "both") else 1.0)
    top_k = torch.full((B,), 9 if mode in ("top_k", "both", "crowded") else 0, dtype=torch.int32)
    if mode == "both" and B > 1:
        top_p[0], top_k[0] = 1.0, 0          # a row without truncation among the others
    seeds = torch.randint(0, 2**40, (B,), generator=g)
    steps = torch.randint(0, 99, (B,), generator=g)
    mask = None
    x = logits.double().numpy()
    if mode == "masked":
        bits = torch.rand(B, (V + 31) // 32 * 32, generator=g) < 0.2
        bits[:, 0] = True
        w = (bits.view(B, -1, 32).long() << torch.arange(32)).sum(-1)
        mask = torch.where(w >= 2**31, w - 2**32, w).to(torch.int32)
        x = np.where(bits[:, :V].numpy(), x, -np.inf)
    dev = lambda t: t.to(DEV)  # noqa: E731
    toks, lps = ops.sample(dev(logits), dev(temp.float()), dev(top_p.float()), dev(top_k), dev(seeds), dev(steps),
                           None if mask is None else dev(mask))
    toks, lps = toks.cpu().numpy(), lps.cpu().numpy()
    for b in range(B):
        t = int(toks[b])
        assert 0 <= t < V
        m = x[b].max()
        ref = x[b, t] - m - np.log(np.exp(x[b] - m).sum())
        # fp32: the logits' own rounding (1e-6 at 16) and a tree sum of V terms
        assert abs(lps[b] - ref) < 2e-5
        if mode == "greedy":
            assert t == int(x[b].argmax())
            continue
        s = x[b] / float(np.float32(temp[b]))
        order = np.argsort(-s, kind="stable")
        p = np.exp(s[order] - s.max())
        p /= p.sum()
        before = np.cumsum(p) - p
        k = int(top_k[b]) if int(top_k[b]) > 0 else V
        # the last member is decided by fp32 mass sums and a threshold rounded to fp32 just below it: the draw may
        # count it in or out
        may, must = before < float(top_p[b]) + 1e-5, before + p < float(top_p[b]) - 1e-5
        may[k:] = must[k:] = False
        must[0] = True
        assert t in set(order[may].tolist())
        key = s + gumbel(int(seeds[b]), int(steps[b]), V)
        # two fast logarithms in fp32: 1e-7 absolute in the inner one, over a winner's 1 - u of about 1 / V
        assert key[t] >= key[order[must]].max() - max(1e-3, 4e-7 * V)


@pytest.mark.parametrize("mode", ["top_p", "top_k", "both"])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("B,V", [(3, 63), (2, 2049), (33, 4099), (2, 131071)])
def test_truncated_rows_with_minus_infinity_logits(B, V, masked, mode):
    """Rows whose logits are -inf for all but a few tokens, for a padded tail, for every token of some threads'
    strides: a thread that sees none before its first finite token adds nothing to the row's mass."""
    g = torch.Generator().manual_seed(V + B)
    logits = torch.randn(B, V, generator=g) * 2.0
    at, kind = torch.arange(V), torch.arange(B).unsqueeze(1) % 3
    logits[(kind == 0) & (torch.rand(B, V, generator=g) > max(20 / V, 0.004))] = -torch.inf
    logits[(kind == 1) & (at >= V * 2 // 3)] = -torch.inf
    logits[(kind == 2) & (at % 256 < 200)] = -torch.inf
    logits[:, V // 2] = 1.0
    mask, x = None, logits.double().numpy()
    if masked:
        bits = torch.rand(B, (V + 31) // 32, 32, generator=g) < 0.5
        bits.view(B, -1)[:, V // 2] = True
        w = (bits.long() << torch.arange(32)).sum(-1)
        mask = torch.where(w >= 2**31, w - 2**32, w).to(torch.int32).to(DEV)
        x = np.where(bits.view(B, -1)[:, :V].numpy(), x, -np.inf)
    top_p, top_k = 1.0 if mode == "top_k" else 0.5, 0 if mode == "top_p" else 7
    temp = torch.rand(B, generator=g) * 0.8 + 0.4
    seeds, steps = torch.randint(0, 2**40, (B,), generator=g), torch.randint(0, 99, (B,), generator=g)
    toks, lps = ops.sample(logits.to(DEV), temp.to(DEV), torch.full((B,), top_p, device=DEV),
                           torch.full((B,), top_k, device=DEV, dtype=torch.int32), seeds.to(DEV), steps.to(DEV), mask)
    for b, t in enumerate(toks.tolist()):
        assert np.isfinite(x[b, t])
        ref = x[b, t] - x[b].max() - np.log(np.exp(x[b] - x[b].max()).sum())
        assert abs(float(lps[b]) - ref) < 2e-5      # as above
        s = x[b] / float(temp[b])
        order = np.argsort(-s, kind="stable")
        p = np.exp(s[order] - s.max())
        p /= p.sum()
        before = np.cumsum(p) - p
        may, must = before < top_p + 1e-5, before + p < top_p - 1e-5
        if top_k:
            may[top_k:] = must[top_k:] = False
        must[0] = True
        assert t in order[may]
        key = s + gumbel(int(seeds[b]), int(steps[b]), V)
        assert key[t] >= key[order[must]].max() - max(1e-3, 4e-7 * V)


@pytest.mark.parametrize("V", [1, 70])
def test_more_rows_than_a_grid_has_in_y(V):
    g = torch.Generator(device=DEV).manual_seed(V)
    B = 65600
    logits = torch.randn(B, V, generator=g, device=DEV)
    temp = torch.rand(B, generator=g, device=DEV) + 0.3
    top_p = torch.where(torch.arange(B, device=DEV) % 2 == 0, 0.7, 1.0)
    top_k = torch.randint(0, 5, (B,), generator=g, device=DEV, dtype=torch.int32)
    seeds, steps = torch.randint(0, 2**40, (B,), generator=g, device=DEV), torch.arange(B, device=DEV)
    mask = torch.randint(-2**31, 2**31, (B, (V + 31) // 32), generator=g, device=DEV).to(torch.int32) | 1
    whole = ops.sample(logits, temp, top_p, top_k, seeds, steps, mask)
    for a, b in ((0, 300), (B - 300, B)):
        part = ops.sample(*(t[a:b] for t in (logits, temp, top_p, top_k, seeds, steps, mask)))
        assert torch.equal(whole[0][a:b], part[0]) and torch.equal(whole[1][a:b], part[1])


@pytest.mark.parametrize("V", [9000, 128256])
@pytest.mark.parametrize("temp", [0.01, 0.7])
def test_top_p_cut_does_not_move(V, temp):
    """The cut of a row with a scaled maximum in the thousands (rounded by 1e-4 there) whose outer tokens hold about
    that much, against float64; tokens and log-probabilities of the same rows at other batch sizes."""
    g = torch.Generator().manual_seed(V)
    R = 250
    s = -torch.rand(R, V, generator=g) * 4.0 - (np.log(V) + 4.5)        # outer tokens: 0.003 of the mass
    s[:, 5] = 0.0
    x = (30.0 + 0.1 * torch.rand(R, 1, generator=g) + s * temp).float()
    x64 = (x.double() - x.double().max(-1, keepdim=True).values) / float(np.float32(temp))
    order = x64.sort(-1, descending=True).values.numpy()
    share = np.exp(order).cumsum(-1) / np.exp(order).sum(-1, keepdims=True)
    top_p = np.float32(1 - 0.4 * (1 - share[:, 0]))                     # inside the outer tokens
    dev = lambda t: torch.as_tensor(t, device=DEV)  # noqa: E731
    args = [dev(x), torch.full((R,), temp, device=DEV), dev(top_p), torch.zeros(R, dtype=torch.int32, device=DEV),
            torch.randint(0, 2**40, (R,), generator=g).to(DEV), torch.zeros(R, dtype=torch.long, device=DEV)]
    dbg = torch.zeros(R, 16, device=DEV)
    toks, lps = ops.sample(*args, None, dbg)
    low = torch.where(dbg[:, 9] > 0, dbg[:, 11], dbg[:, 7]).cpu().numpy()       # the last refinement's lower edge
    for b in range(R):
        # one fp32 rounding of a mass of 1 is 6e-8, of the outer tokens' 0.003 2e-5 for each sum it went through; and of
        # x itself at 30, 2e-6 / temp in scaled logits
        kept = int((order[b] > low[b]).sum()) - 1
        want = int((share[b] < float(top_p[b])).sum())
        assert abs(kept - want) <= 0.01 * V, (b, kept, want)
    for n in (1, 7, 100):
        t, p = ops.sample(*(a[:n] for a in args))
        # the slices' sums in another order: a few fp32 roundings of each level of their tree
        assert torch.equal(t, toks[:n]) and torch.allclose(p, lps[:n], rtol=0, atol=2e-6)


@pytest.mark.parametrize("mode", ["plain", "greedy", "masked", "top_k", "top_p", "both", "crowded"])
@pytest.mark.parametrize("B,V", [(3, 64), (2, 1023), (2, 1025), (40, 4095), (3, 4096), (3, 4097)])
def test_short_rows_in_one_launch(B, V, mode):
    """Rows around the length up to which one workgroup does a whole row."""
    test_draw_matches_float64(B, V, mode)


def test_short_rows_without_an_allowed_token():
    """Nothing allowed, or nothing above -inf: token 0, as in longer rows."""
    for V in (70, 5000):
        logits = torch.randn(3, V, device=DEV)
        logits[1:] = -torch.inf
        mask = torch.full((3, (V + 31) // 32), -1, dtype=torch.int32, device=DEV)
        mask[0] = 0
        for p, k in ((1.0, 0), (0.9, 0), (1.0, 5)):
            toks, _ = ops.sample(logits, torch.ones(3, device=DEV), torch.full((3,), p, device=DEV),
                                 torch.full((3,), k, dtype=torch.int32, device=DEV), torch.arange(3, device=DEV),
                                 torch.zeros(3, dtype=torch.long, device=DEV), mask)
            assert toks.tolist() == [0, 0, 0]


@pytest.mark.parametrize("B,V", [(1, 131072), (40, 32769), (256, 131072), (257, 131072)])
@pytest.mark.parametrize("near", [40, 47, 48, 49, 300])
def test_cut_inside_and_behind_the_slices_lists(B, V, near):
    """``near`` tokens close to the max in one stretch of the row, and a flat rest 9, 16 or 30 of scaled logit below: a
    slice lists all of them, or fewer than are asked for, or the cut lies in the rest."""
    g = torch.Generator().manual_seed(near + V)
    gap = torch.tensor([9.0, 16.0, 30.0])[torch.arange(B) % 3].unsqueeze(1)
    logits = torch.rand(B, V, generator=g) - gap
    logits[:, 100:100 + near] = torch.rand(B, near, generator=g) * 2.0
    top_k = torch.full((B,), 45, dtype=torch.int32)
    top_k[1::2] = 301
    seeds, steps = torch.randint(0, 2**40, (B,), generator=g), torch.randint(0, 99, (B,), generator=g)
    one = torch.ones(B, device=DEV)
    toks, _ = ops.sample(logits.to(DEV), one, one, top_k.to(DEV), seeds.to(DEV), steps.to(DEV), None)
    for b in range(0, B, 1 if B < 100 else 41):
        x = logits[b].double().numpy()
        kept = np.argsort(-x, kind="stable")[:int(top_k[b])]
        key = x + gumbel(int(seeds[b]), int(steps[b]), V)
        t = int(toks[b])
        # ties of fp32 logits at the cut may go either way; fast logarithms are off by 4e-7 of the draw's range
        assert x[t] >= x[kept[-1]] and key[t] >= key[kept].max() - max(1e-3, 4e-7 * V)


@pytest.mark.parametrize("B,V", [(2, 50257), (3, 50257), (128, 65536), (129, 65536), (192, 65537), (193, 65537)])
def test_calls_on_either_side_of_the_lines_for_lists(B, V):
    test_cut_inside_and_behind_the_slices_lists(B, V, 49)


@pytest.mark.parametrize("B,plain", [(129, 15), (129, 16), (129, 17), (300, 37), (300, 38), (300, 300)])
def test_large_calls_with_rows_that_are_not_truncated(B, plain):
    """On either side of one row in eight, counted over more rows than a wave has lanes."""
    V = 32801
    g = torch.Generator().manual_seed(B + plain)
    logits = torch.randn(B, V, generator=g) * 2.0
    top_k = torch.full((B,), 7, dtype=torch.int32)
    top_k[torch.randperm(B, generator=g)[:plain]] = 0
    seeds, steps = torch.randint(0, 2**40, (B,), generator=g), torch.randint(0, 99, (B,), generator=g)
    one = torch.ones(B, device=DEV)
    toks, _ = ops.sample(logits.to(DEV), one, one, top_k.to(DEV), seeds.to(DEV), steps.to(DEV), None)
    for b in range(0, B, 7):
        x = logits[b].double().numpy()
        kept = np.argsort(-x, kind="stable")[:int(top_k[b]) or V]
        key = x + gumbel(int(seeds[b]), int(steps[b]), V)
        t = int(toks[b])
        assert x[t] >= x[kept[-1]] and key[t] >= key[kept].max() - max(1e-3, 4e-7 * V)      # as above


@pytest.mark.parametrize("ulps", [1, 2, 16])
def test_top_p_a_few_ulps_below_one(ulps):
    """Rows whose allowed tokens all lie in the slices' lists: whether fp32 sums of their masses reach top_p of the whole
    depends on the order of the sums, and every order has to end in a draw."""
    B, V, near = 32, 128256, 400
    top_p = float(np.float32(1.0) - np.float32(ulps * 2.0 ** -24))
    g = torch.Generator(device=DEV).manual_seed(ulps)
    for call in range(32):
        at = torch.rand(B, V, generator=g, device=DEV).topk(near, -1).indices
        x = torch.rand(B, near, generator=g, device=DEV)
        logits = torch.zeros(B, V, device=DEV).scatter_(1, at, x)
        words = torch.zeros(B, V // 32, dtype=torch.long, device=DEV)
        words.scatter_add_(1, at // 32, torch.ones_like(at) << (at % 32))
        mask = torch.where(words >= 2**31, words - 2**32, words).to(torch.int32)
        seeds = torch.randint(0, 2**40, (B,), generator=g, device=DEV)
        steps = torch.randint(0, 99, (B,), generator=g, device=DEV)
        toks, _ = ops.sample(logits, torch.ones(B, device=DEV), torch.full((B,), top_p, device=DEV),
                             torch.zeros(B, dtype=torch.int32, device=DEV), seeds, steps, mask)
        at, x, seeds, steps, toks = (t.cpu().numpy() for t in (at, x.double(), seeds, steps, toks))
        with np.errstate(over="ignore"):
            base = splitmix(seeds.astype(np.uint64) * np.uint64(0x9E3779B97F4A7C15)
                            + steps.astype(np.uint64) * np.uint64(0xBF58476D1CE4E5B9))
            h = splitmix(base[:, None] ^ at.astype(np.uint64)) >> np.uint64(40)
        u = ((h + np.uint64(1)).astype(np.float32) * np.float32(1.0 / 16777217.0)).astype(np.float64)
        key = x - np.log(-np.log(u))
        for b in range(B):
            won = np.nonzero(at[b] == toks[b])[0]
            assert won.size == 1
            # the lowest ten of 400 (a fortieth of the mass at most, the rounding of the sums is 1e-5 of it) may be out
            kept = np.argsort(-x[b])[:near - 10]
            assert key[b, won[0]] >= key[b, kept].max() - 1e-3, (call, b)


def draws(seed, step, V):
    with np.errstate(over="ignore"):
        base = splitmix(np.uint64(seed) * np.uint64(0x9E3779B97F4A7C15) + np.uint64(step) * np.uint64(0xBF58476D1CE4E5B9))
    return splitmix(base ^ np.arange(V, dtype=np.uint64)) >> np.uint64(40)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("B,V", [(1, 2049), (3, 6145), (1, 16447), (40, 50257), (200, 32801), (700, 8193)])
def test_flat_rows_draw_the_highest_hash(B, V, masked):
    """Equal logits: the draw is the hash's alone, lanes hold several near the top and ties are of equal hashes."""
    mask, ok = None, np.ones((B, V), dtype=bool)
    if masked:
        bits = torch.rand(B, (V + 31) // 32 * 32, generator=torch.Generator().manual_seed(V)) < 0.1
        bits[:, V - 1] = True
        w = (bits.view(B, -1, 32).long() << torch.arange(32)).sum(-1)
        mask = torch.where(w >= 2**31, w - 2**32, w).to(torch.int32).to(DEV)
        ok = bits[:, :V].numpy()
    one = torch.ones(B, device=DEV)
    seeds = torch.arange(B) * 7919 + V
    toks, lps = ops.sample(torch.full((B, V), 3.25, device=DEV), one, one, torch.zeros(B, dtype=torch.int32, device=DEV),
                           seeds.to(DEV), torch.full((B,), 3, device=DEV), mask)
    for b in range(B):
        h = np.where(ok[b], draws(int(seeds[b]), 3, V).astype(np.int64), -1)
        assert h[int(toks[b])] == h.max()
        assert abs(float(lps[b]) + np.log(ok[b].sum())) < 1e-5 * np.log(V) + 1e-6


@pytest.mark.parametrize("masked", [False, True])
def test_a_uniform_of_one_wins(masked):
    """One hash in 2^24 gives u = 1 in float32, an infinite key: it is drawn whatever its logit, unless masked."""
    V = 131072
    found = [(s, int(h.argmax())) for s in range(600) for h in (draws(s, 1, V),) if int(h.max()) == 0xffffff][:3]
    assert found, "600 rows of 2^17 have about 4.7"
    B = len(found)
    seeds = torch.tensor([s for s, _ in found])
    at = [t for _, t in found]
    logits = torch.randn(B, V, generator=torch.Generator().manual_seed(1))
    logits[range(B), at] = -40.0
    mask = None
    if masked:
        mask = torch.full((B, V // 32), -1, dtype=torch.int32)
        for b in range(0, B, 2):
            mask[b, at[b] // 32] ^= torch.tensor(1 << (at[b] % 32) if at[b] % 32 < 31 else -2**31, dtype=torch.int32)
        mask = mask.to(DEV)
    one = torch.ones(B, device=DEV)
    toks, _ = ops.sample(logits.to(DEV), one, one, torch.zeros(B, dtype=torch.int32, device=DEV), seeds.to(DEV),
                         one.long(), mask)
    for b in range(B):
        if masked and b % 2 == 0:
            assert int(toks[b]) != at[b]
        else:
            assert int(toks[b]) == at[b]


@pytest.mark.parametrize("near", [50, 63, 64, 65, 200])
@pytest.mark.parametrize("width", [0.0, 1e-6, 0.05])
@pytest.mark.parametrize("B,V", [(1, 131072), (3, 50257), (40, 32000), (512, 8192), (513, 8192)])
def test_cut_in_a_crowded_bin_of_the_lists(B, V, near, width):
    """The highest tokens, spread over the row's slices, within a bin of the histogram or equal: one wave orders up to 64
    of them, more are refined."""
    g = torch.Generator().manual_seed(near + V)
    logits = torch.rand(B, V, generator=g) - 12.0
    at = torch.arange(near) * (V // near) + 7
    logits[:, at] = 1.0 - width * torch.rand(B, near, generator=g)
    k = torch.tensor([45, 10, 1])[torch.arange(B) % 3].int()
    top_p = torch.tensor([1.0, 0.95])[torch.arange(B) % 2]
    seeds, steps = torch.randint(0, 2**40, (B,), generator=g), torch.randint(0, 99, (B,), generator=g)
    toks, _ = ops.sample(logits.to(DEV), torch.ones(B, device=DEV), top_p.to(DEV), k.to(DEV), seeds.to(DEV), steps.to(DEV), None)
    for b in range(0, B, 1 if B < 100 else 41):
        x = logits[b].double().numpy()
        order = np.argsort(-x, kind="stable")
        p = np.exp(x[order] - x.max())
        before = (np.cumsum(p) - p) / p.sum()
        lim = int(k[b])
        must = order[:lim][before[:lim] < float(top_p[b]) - 1e-4]
        low = x[must[-1]] - 1e-6 - (1e-4 if top_p[b] < 1 else 0.0)      # tokens that tie with the last one may be in
        t = int(toks[b])
        key = x + gumbel(int(seeds[b]), int(steps[b]), V)
        assert x[t] >= low and key[t] >= key[must].max() - max(1e-3, 4e-7 * V)


@pytest.mark.parametrize("top_k", [0, 30])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("B,V", [(2, 50257), (7, 128256), (40, 32000), (3, 3000), (600, 8192)])
def test_top_p_zero_draws_among_the_highest(B, V, masked, top_k):
    """Top-p 0 leaves what ties with the max, with the slices' lists and without: the draw is among those."""
    g = torch.Generator().manual_seed(V + B)
    logits = torch.randn(B, V, generator=g) - 6.0
    at = [7, V // 3, V // 2 + 1, V - 2]
    logits[:, at] = 2.5
    mask = torch.full((B, (V + 31) // 32), -1, dtype=torch.int32).to(DEV) if masked else None
    seeds, steps = torch.randint(0, 2**40, (B,), generator=g), torch.randint(0, 99, (B,), generator=g)
    toks, _ = ops.sample(logits.to(DEV), torch.ones(B, device=DEV), torch.zeros(B, device=DEV),
                         torch.full((B,), top_k, dtype=torch.int32, device=DEV), seeds.to(DEV), steps.to(DEV), mask)
    for b in range(0, B, 1 if B < 100 else 41):
        h = draws(int(seeds[b]), int(steps[b]), V)[at]
        assert int(toks[b]) in at and h[at.index(int(toks[b]))] == h.max()

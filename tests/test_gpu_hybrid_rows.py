"""A hybrid model's step of single decoded rows, sublayer by sublayer in native code, against the general sublayers."""

from types import SimpleNamespace

import pytest
import torch

from kllms_amd import ops
from kllms_amd.engine.config import (BlockAttnSpec, ChannelDeltaSpec, DecayLinearAttnSpec, EngineConfig, ParallelMixerSpec,
                                     RotarySpec)
from kllms_amd.engine.engine import LLMEngine
from kllms_amd.engine.kvcache import LayerState
from kllms_amd.models.mixers import ChannelDeltaMixer, ParallelMixer

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


def _logits(eng, rows, native, lens=None):
    g = torch.Generator().manual_seed(rows)
    seqs = [eng.open_sequence() for _ in range(rows)]
    lens = lens or torch.randint(1, 70, (rows,), generator=g).tolist()
    ids = [torch.randint(3, eng.arch.vocab_size, (n,), generator=g).tolist() for n in lens]
    eng.step_segments([(s, t, []) for s, t in zip(seqs, ids)])
    ok, out = ops.hybrid_rows_ok, []
    try:
        if not native:
            ops.hybrid_rows_ok = lambda *a: False
        for step in range(3):
            out.append(eng.step_segments([(s, [5 + step + i], [0]) for i, s in enumerate(seqs)]).double())
    finally:
        ops.hybrid_rows_ok = ok
        for s in seqs:
            eng.kv.free_sequence(s)
    return out


@pytest.mark.parametrize("rows", [1, 15, 17, 33, 65, 128, 129])
def test_rows_steps_against_the_general_sublayers(rows):
    eng = LLMEngine(EngineConfig(model="zutalix-1b-l6", device=DEV, seed=0, use_hip_graphs=False, max_kv_blocks=2048,
                                 max_state_slots=140, enable_prefix_caching=False, eos_token_id=-1))
    calls = []
    step = ops.hybrid_glu_rows
    try:
        ops.hybrid_glu_rows = lambda *a: calls.append(1) or step(*a)
        got = _logits(eng, rows, True)
    finally:
        ops.hybrid_glu_rows = step
    assert (len(calls) > 0) == (rows <= 128)
    # two bf16 computations of the same step, each 0.008 off 64 bits in the 2-norm, which later steps' states carry on
    for a, b in zip(got, _logits(eng, rows, False)):
        assert (a - b).norm() <= 0.025 * b.norm()


def test_rows_steps_of_ragged_contexts():
    """Contexts in several parts of the keys, rows with fewer keys than parts, and both sides of a block of the mask (1024);
    each row's logits, and what the steps write: cache, convolution and recurrent state."""
    lens = [130, 600, 1021, 1023, 1024, 1025, 1300, 1, 2047]
    runs = []
    for native in (True, False):
        eng = LLMEngine(EngineConfig(model="zutalix-1b-l6", device=DEV, seed=0, use_hip_graphs=False, max_kv_blocks=1024,
                                     max_state_slots=16, enable_prefix_caching=False, eos_token_id=-1))
        runs.append((_logits(eng, len(lens), native, lens),
                     [[t.double() for t in (st.k, st.v, st.conv, st.rec) if t is not None] for st in eng.kv.layer_caches()]))
        del eng
    # each within 0.008 of 64 bits in the 2-norm over many rows; one row of these up to twice that, both computations of it
    for a, b in zip(runs[0][0], runs[1][0]):
        assert ((a - b).norm(dim=1) <= 0.032 * b.norm(dim=1)).all()
    for got, ref in zip(runs[0][1], runs[1][1]):
        for a, b in zip(got, ref):
            a, b = a.flatten(1), b.flatten(1)
            assert ((a - b).norm(dim=1) <= 0.032 * b.norm(dim=1)).all()


def test_rows_steps_with_weights_that_lie_otherwise():
    """Transposed, or off 16 bytes: what the general sublayers' products take."""
    eng = LLMEngine(EngineConfig(model="mid-zutalix", device=DEV, seed=0, use_hip_graphs=False, max_kv_blocks=256,
                                 max_state_slots=40, enable_prefix_caching=False, eos_token_id=-1))
    ref = _logits(eng, 5, True)
    for i, layer in enumerate(eng.model.layers):
        for m in (layer.mix, layer.mlp):
            if m is not None:
                w = m.inp.weight.data
                m.inp.weight.data = (w.t().contiguous().t() if i % 2 == 0
                                     else w.new_empty(w.numel() + 1)[1:].view_as(w).copy_(w))
    for a, b in zip(_logits(eng, 5, True), ref):
        assert (a - b).norm() <= 0.025 * b.norm()      # as above


@pytest.mark.parametrize("T", [1, 64, 65, 128])
def test_gated_sublayer_against_the_general_one(T):
    """On the few-row product with the activation in it, and above 64 rows on the library's and a pass."""
    W, ff = 384, 640
    g = torch.Generator(device=DEV).manual_seed(T)
    h = torch.randn(T, W, generator=g, device=DEV).bfloat16()
    x = torch.randn(T, W, generator=g, device=DEV)
    w_in = (torch.randn(2 * ff, W, generator=g, device=DEV) * 0.1).bfloat16()
    w_down = (torch.randn(W, ff, generator=g, device=DEV) * 0.05).bfloat16()
    post, nxt = (torch.rand(W, generator=g, device=DEV) + 0.5 for _ in range(2))
    ref = x.clone()
    y = torch.nn.functional.linear(h, w_in)
    y = torch.nn.functional.linear(ops.clamped_glu(y[:, :ff], y[:, ff:], 2.0, 1.5), w_down)
    out = ops.sandwich_residual(ref, y, post, 1e-6, w_next=nxt, out_dtype=torch.bfloat16)
    got = ops.hybrid_glu_rows(x, h, w_in, w_down, post, nxt, 2.0, 1.5, 1e-6)
    # the one rounds gate, up and y to bf16 (2^-9 each), the other the activation alone; rows of a normal size
    assert (x - ref).abs().max() <= 5e-2 and (got.float() - out.float()).abs().max() <= 8e-2
    assert ((x - ref).norm(dim=1) <= 1e-2 * ref.norm(dim=1)).all()


@pytest.mark.parametrize("T", [1, 9])
@pytest.mark.parametrize("H,G,D,V,taps,ranks", [(2, 2, 64, 64, 4, (16, 8)), (4, 2, 64, 128, 4, (64, 56)), (3, 1, 40, 128, 2, (16, 72)),
                                                (4, 1, 256, 32, 3, (16, 8)), (2, 2, 256, 192, 16, (8, 32)),
                                                (8, 2, 128, 160, 5, (136, 16))])
def test_delta_sublayer_against_the_general_one(T, H, G, D, V, taps, ranks):
    """One, two and three heads to a key head, keys that fill the row groups and do not, values in one block of columns and
    more, few taps and many, ranks within and above one pass; fresh rows and carried ones, slots in any order."""
    W, eps = 256, 1e-5
    g = torch.Generator(device=DEV).manual_seed(H * D + V)
    spec = ChannelDeltaSpec(heads=H, kv_heads=G, dim=D, vdim=V, conv=taps, decay_rank=ranks[0], gate_rank=ranks[1])
    mix = ChannelDeltaMixer(spec, W, eps, torch.bfloat16).to(DEV)
    for n, p in mix.checkpoint_map("").items():
        p.data.copy_(torch.randn(p.shape, generator=g, device=DEV) * (1.0 if p.dim() == 1 else p.shape[-1] ** -0.5))
    start = torch.randint(0, 2, (T,), generator=g, device=DEV, dtype=torch.int32) * 7
    start[0] = 7
    rows = torch.arange(T + 1, device=DEV, dtype=torch.int32)
    batch = SimpleNamespace(state_slots=torch.randperm(T + 2, generator=g, device=DEV)[:T].int(), cu_seqlens=rows, seg_start=start,
                            token_seg=rows[:T].contiguous())
    states = [LayerState(rec=torch.randn(T + 2, H, D, V, generator=g, device=DEV) * 0.2,
                         conv=torch.randn(T + 2, taps - 1, mix.cp, generator=g, device=DEV).bfloat16())]
    states.append(LayerState(rec=states[0].rec.clone(), conv=states[0].conv.clone()))
    h = torch.randn(T, W, generator=g, device=DEV).bfloat16()
    x = torch.randn(T, W, generator=g, device=DEV)
    ref = x.clone()
    post, nxt = (torch.rand(W, generator=g, device=DEV) + 0.5 for _ in range(2))
    with torch.no_grad():
        out = ops.sandwich_residual(ref, mix(h, batch, states[0]), post, eps, w_next=nxt, out_dtype=torch.bfloat16)
        got = mix.rows_step(x, h, batch, states[1], post, nxt)
    # the same roundings of values summed in another order: some go the other way, 2^-8 of a term each
    for a, b in ((x, ref), (got, out), (states[1].rec, states[0].rec)):
        assert (a.double() - b.double()).norm() <= 1e-2 * b.double().norm()
    assert (states[1].conv.double() - states[0].conv.double()).abs().max() <= 2 ** -7 * states[0].conv.double().abs().max()
    assert (states[1].conv != states[0].conv).float().mean() <= 0.02


@pytest.mark.parametrize("T", [1, 9, 128])
@pytest.mark.parametrize("H,G,D,V,taps,ranks", [(4, 2, 64, 64, 4, (20, 60)), (64, 32, 32, 130, 4, (16, 16)),
                                                (8, 1, 256, 512, 4, (64, 72))])
def test_delta_sublayers_of_other_sizes_stay_native(T, H, G, D, V, taps, ranks):
    """Ranks not in eights, values not in fours, more than a workgroup keeps: the sublayer's launches one by one."""
    test_delta_sublayer_against_the_general_one(T, H, G, D, V, taps, ranks)


@pytest.mark.parametrize("name", ["a2", "g2"])
@pytest.mark.parametrize("how", ["transposed", "off 16 bytes"])
def test_delta_sublayers_with_low_rank_weights_that_lie_otherwise(name, how, monkeypatch):
    step = ChannelDeltaMixer.rows_step

    def moved(self, *a):
        w = getattr(self, name).data
        getattr(self, name).data = (w.t().contiguous().t() if how == "transposed"
                                    else w.new_empty(w.numel() + 1)[1:].view_as(w).copy_(w))
        return step(self, *a)

    monkeypatch.setattr(ChannelDeltaMixer, "rows_step", moved)
    test_delta_sublayer_against_the_general_one(9, 4, 2, 64, 64, 4, (16, 8))


@pytest.mark.parametrize("T", [1, 9])
@pytest.mark.parametrize("G,RH,RD,RV", [(2, 16, 64, 128), (4, 2, 40, 192), (4, 4, 256, 32)])
def test_parallel_sublayer_against_the_general_one(T, G, RH, RD, RV):
    """Output products of one size (one launch) and of two, keys that fill the row groups and do not, values in one block of
    columns and more; fresh rows and carried ones, slots in any order."""
    W, H, eps, BS, blocks = 256, 16, 1e-5, 16, 4
    g = torch.Generator(device=DEV).manual_seed(RH * RD + RV)
    spec = ParallelMixerSpec(left=BlockAttnSpec(heads=H, kv_heads=G, dim=128, vdim=128, scale=0.1, mask_size=32,
                                                rot=RotarySpec(dims=96)),
                             right=DecayLinearAttnSpec(heads=RH, dim=RD, vdim=RV, decay=[0.5 + 0.4 * i / RH for i in range(RH)]))
    mix = ParallelMixer(spec, W, eps, torch.bfloat16).to(DEV)
    for n, p in mix.checkpoint_map("").items():
        p.data.copy_(torch.randn(p.shape, generator=g, device=DEV) * (1.0 if p.dim() == 1 else p.shape[-1] ** -0.5))
    rows = torch.arange(T + 1, device=DEV, dtype=torch.int32)
    positions = torch.randint(0, BS * blocks, (T,), generator=g, device=DEV)
    positions[0] = BS * blocks - 1
    tables = torch.randperm(T * blocks, generator=g, device=DEV).int().view(T, blocks)
    start = torch.where(torch.randint(0, 2, (T,), generator=g, device=DEV) > 0, positions, 0).int()
    start[0] = positions[0]
    batch = SimpleNamespace(
        mode="decode", host_segs=None, plans=None, positions=positions, context_lens=(positions + 1).int(), block_tables=tables,
        slot_mapping=tables.gather(1, (positions // BS)[:, None]).squeeze(1).long() * BS + positions % BS,
        state_slots=torch.randperm(T + 2, generator=g, device=DEV)[:T].int(), cu_seqlens=rows, seg_start=start,
        token_seg=rows[:T].contiguous())
    cache = torch.randn(2, T * blocks, G, BS, 128, generator=g, device=DEV).bfloat16()
    rec = torch.randn(T + 2, RH, RD, RV, generator=g, device=DEV) * 0.2
    states = [LayerState(k=cache[0].clone(), v=cache[1].clone(), rec=rec.clone()) for _ in range(2)]
    h = torch.randn(T, W, generator=g, device=DEV).bfloat16()
    x = torch.randn(T, W, generator=g, device=DEV)
    ref = x.clone()
    post, nxt = (torch.rand(W, generator=g, device=DEV) + 0.5 for _ in range(2))
    with torch.no_grad():
        left, right = mix(h, batch, states[0])
        out = ops.sandwich_residual(ref, left, post, eps, b=right, wa=mix.left_out, wb=mix.right_out, w_next=nxt,
                                    out_dtype=torch.bfloat16)
        got = mix.rows_step(x, h, batch, states[1], post, nxt)
    # bf16 roundings at other places (q, k, v before their use, the branches' sums): 2^-9 of each, in a few steps behind another
    for a, b in ((x, ref), (got, out), (states[1].rec, states[0].rec)):
        assert (a.double() - b.double()).norm() <= 1.5e-2 * b.double().norm()
    for a, b in ((states[1].k, states[0].k), (states[1].v, states[0].v)):
        assert ((a.double() - b.double()).abs() <= 2 ** -6 * b.double().abs() + 2e-2).all()


def test_residual_of_split_sums_against_float64():
    C, W, T = ops._seq(), 384, 5
    g = torch.Generator(device=DEV).manual_seed(0)
    h = torch.randn(T, W, generator=g, device=DEV).bfloat16()
    x = torch.randn(T, W, generator=g, device=DEV)
    w_in = (torch.randn(256, W, generator=g, device=DEV) * 0.2).bfloat16()
    w_down = (torch.randn(W, 128, generator=g, device=DEV) * 0.2).bfloat16()
    post, nxt = (torch.rand(W, generator=g, device=DEV) + 0.5 for _ in range(2))
    gate, up = (h.double() @ w_in.double().t()).chunk(2, -1)
    gate, up = gate.clamp(max=2.0), up.clamp(-2.0, 2.0)
    act = (gate * torch.sigmoid(1.5 * gate) * (up + 1)).bfloat16().double()
    y = act @ w_down.double().t()
    ref = x.double() + y / torch.sqrt((y * y).mean(-1, keepdim=True) + 1e-6) * post.double()
    out = ref / torch.sqrt((ref * ref).mean(-1, keepdim=True) + 1e-6) * nxt.double()
    got = C.hybrid_glu_rows(x, h, w_in, w_down, post, nxt, 2.0, 1.5, 1e-6)
    # an activation that rounds to bf16 the other way moves a row by 2^-8 of one of its 128 terms
    assert (x.double() - ref).abs().max() <= 2e-2
    assert ((got.double() - out).abs() <= 2 ** -8 * out.abs() + 2e-2).all()


@pytest.mark.parametrize("W,ff", [(128, 1152), (256, 2304), (128, 4352), (2176, 640), (4224, 1280)])
def test_residual_of_many_split_sums_against_float64(W, ff):
    """4, 9 and 17 splits; rows of more than one vector a thread, the last one ragged."""
    C, T = ops._seq(), 5
    g = torch.Generator(device=DEV).manual_seed(ff)
    h = torch.randn(T, W, generator=g, device=DEV).bfloat16()
    x = torch.randn(T, W, generator=g, device=DEV)
    w_in = (torch.randn(2 * ff, W, generator=g, device=DEV) * W ** -0.5).bfloat16()
    w_down = (torch.randn(W, ff, generator=g, device=DEV) * ff ** -0.5).bfloat16()
    post, nxt = (torch.rand(W, generator=g, device=DEV) + 0.5 for _ in range(2))
    gate, up = (h.double() @ w_in.double().t()).chunk(2, -1)
    gate, up = gate.clamp(max=2.0), up.clamp(-2.0, 2.0)
    act = (gate * torch.sigmoid(1.5 * gate) * (up + 1)).bfloat16().double()
    y = act @ w_down.double().t()
    ref = x.double() + y / torch.sqrt((y * y).mean(-1, keepdim=True) + 1e-6) * post.double()
    out = ref / torch.sqrt((ref * ref).mean(-1, keepdim=True) + 1e-6) * nxt.double()
    got = C.hybrid_glu_rows(x, h, w_in, w_down, post, nxt, 2.0, 1.5, 1e-6)
    # as above, of more terms: 2^-8 of the few activations whose rounding falls the other way
    assert (x.double() - ref).abs().max() <= 2e-2
    assert ((got.double() - out).abs() <= 2 ** -8 * out.abs() + 2e-2).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,V", [(4, 2, 128), (3, 3, 16), (2, 1, 80)])
@pytest.mark.parametrize("lens", [[64], [16, 17, 200, 31, 1, 300, 0, 33], [300, 64]])
def test_delta_rule_by_chunks_against_float64(H, G, V, lens, dtype):
    """Segments fresh and continued, with lengths around the chunk's 16, strong and weak decays."""
    D, T, B = 64, sum(lens), len(lens)
    g = torch.Generator().manual_seed(T + V)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    q, k, v, beta = rnd(T, G, D).to(dtype), rnd(T, G, D).to(dtype), rnd(T, H, V).to(dtype), rnd(T, H).to(dtype)
    a, dt, a_log = (rnd(T, H * D) * 2).to(dtype), rnd(H * D), torch.linspace(-3, 2, H)
    state = rnd(B + 2, H, D, V)
    slots = torch.randperm(B + 2, generator=g)[:B].to(torch.int32)
    start = torch.tensor([7 * (b % 2) for b in range(B)], dtype=torch.int32)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    dev = lambda t: t.to(DEV)  # noqa: E731
    got_state = dev(state)
    assert T >= 64 * B                       # else the token-by-token form
    o = ops.gated_delta_rule(dev(q), dev(k), dev(v), dev(beta), dev(a), dev(dt), dev(a_log), got_state, dev(slots), dev(cu),
                             dev(start))
    unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    qd, kd = (unit(t.double()).repeat_interleave(H // G, 1) for t in (q, k))
    qd = qd * D ** -0.5
    decay = torch.exp(-a_log.double().exp().view(1, H, 1)
                      * torch.nn.functional.softplus(a.double() + dt.double()).view(T, H, D))
    for b in range(B):
        S = state[slots[b]].double() if start[b] else torch.zeros(H, D, V, dtype=torch.float64)
        size = max(1.0, float(S.abs().max()))
        for t in range(cu[b], cu[b + 1]):
            S = S * decay[t].unsqueeze(-1)
            u = torch.sigmoid(beta[t].double()).unsqueeze(-1) * (v[t].double() - (kd[t].unsqueeze(-2) @ S).squeeze(-2))
            S = S + kd[t].unsqueeze(-1) * u.unsqueeze(-2)
            # fp32 sums of 64 products of values of the state's size, carried on by a contraction
            assert ((qd[t].unsqueeze(-2) @ S).squeeze(-2) - o[t].double().cpu()).abs().max() <= 64 * 2 ** -23 * 8 * size
            size = max(size, float(v[t].double().abs().max()))
        assert (S - got_state[slots[b]].double().cpu()).abs().max() <= 64 * 2 ** -23 * 8 * size
    for s in set(range(B + 2)) - set(slots.tolist()):
        assert torch.equal(got_state[s].cpu(), state[s])


@pytest.mark.parametrize("name,at", [("q", 10), ("k", 0), ("k", 21), ("v", 16), ("v", 29), ("beta", 37), ("a", 32), ("a", 47)])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
def test_delta_rule_by_chunks_keeps_later_tokens_out_of_earlier_ones(name, at, value):
    """A value that is not finite reaches the tokens from its own on, as token by token, and not those before it in its
    chunk of 16; one of v stays in its column."""
    D, H, G, V, T = 64, 2, 1, 48, 80
    g = torch.Generator().manual_seed(at)
    rnd = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    x = {"q": rnd(T, G, D), "k": rnd(T, G, D), "v": rnd(T, H, V), "beta": rnd(T, H), "a": rnd(T, H * D)}
    dt, a_log, start = rnd(H * D), torch.zeros(H), rnd(1, H, D, V)

    def run(dev, dtype, op):
        i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
        state = start.to(dev, torch.float32)
        args = [x[n].to(dev, dtype) for n in ("q", "k", "v", "beta", "a")]
        o = op(*args, dt.to(dev), a_log.to(dev), state, i32(0), i32(0, T), i32(5))
        return o.double().cpu().view(T, H, V), state.double().cpu()

    clean, _ = run(DEV, torch.float32, ops.gated_delta_rule)
    x[name][at].view(-1)[1] = value
    o, state = run(DEV, torch.float32, ops.gated_delta_rule)
    assert torch.equal(o[:at], clean[:at])
    ref, ref_state = run("cpu", torch.float32, ops.gated_delta_rule)
    assert torch.equal(o.isfinite(), ref.isfinite()) and torch.equal(state.isfinite(), ref_state.isfinite())
    ok = ref.isfinite()
    assert ((o - ref)[ok].abs() <= 64 * 2 ** -23 * 8 * 8).all()      # sums of 64 products, as above; values below 8

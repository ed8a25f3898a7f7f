"""A hybrid model's step of single decoded rows, sublayer by sublayer in native code, against the general sublayers."""

import pytest
import torch

from kllms_amd import ops
from kllms_amd.engine.config import EngineConfig
from kllms_amd.engine.engine import LLMEngine

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


def _logits(eng, rows, native):
    g = torch.Generator().manual_seed(rows)
    seqs = [eng.open_sequence() for _ in range(rows)]
    lens = torch.randint(1, 70, (rows,), generator=g).tolist()
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

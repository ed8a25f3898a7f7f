"""Rules that choose between two forms of a call: which prompt portions behind a cache attend together on the matrix
cores, which steps take the few-row [gate; up] product."""

import pytest

from kllms_amd import ops


@pytest.mark.parametrize("segs,kv_heads,pays", [
    ([], 8, False),
    ([(500, 1)] * 40, 8, False),                    # decode rows
    ([(3000, 31)] * 12, 8, False),                  # short segments only
    ([(0, 32)], 8, False), ([(6000, 32)], 8, False), ([(6000, 64)], 8, False),   # too few workgroups for the keys
    ([(6000, 94)], 8, True), ([(500, 128)], 8, True), ([(2000, 64)] * 2, 8, True), ([(6000, 32)] * 4, 8, True),
    ([(6000, 128)], 4, False), ([(6000, 188)], 4, True), ([(3000, 32)], 32, True), ([(300, 64)] * 4, 1, False),
    ([(6000, 40), (10, 300)], 8, False),            # a long context with few rows beside many rows of a short one
    ([(6000, 40), (10, 300), (5000, 80)], 8, True),
    ([(1536, 150)] * 8, 8, True),
])
def test_portions(segs, kv_heads, pays):
    assert ops.paged_prefill_pays(segs, kv_heads) is pays


@pytest.mark.parametrize("segs,heads,few", [
    ([], 32, False), ([(3000, 31)] * 2, 32, False),                              # nothing on the matrix cores
    ([(447, 64)], 32, False), ([(448, 64)], 32, True), ([(5, 400)], 32, False),  # keys that are few
    ([(1536, 146)], 32, True), ([(1536, 512)] * 2, 32, True), ([(1536, 256)] * 4, 32, True), ([(1536, 300)] * 4, 32, False),
    ([(1536, 128)] * 4, 32, True), ([(1536, 65)] * 8, 32, False), ([(1536, 146)] * 8, 32, False), ([(1536, 146)] * 8, 16, True),
    ([(1536, 64)] * 12, 32, True), ([(4000, 128)] * 12, 32, True), ([(4000, 40), (10, 4000)], 32, False),
    ([(4000, 40), (3000, 1)] * 2, 32, True),                                      # decode rows beside do not count
])
def test_groups_of_portions(segs, heads, few):
    assert ops.paged_prefill_few(segs, heads) is few


def test_one_short_portion_behind_a_long_cache_goes_row_by_row(monkeypatch):
    """The model asks the rule: a step of one 32-row portion has no plan, one of eight has."""
    import torch

    from kllms_amd.models.llama import ForwardBatch, LlamaForCausalLM

    model = LlamaForCausalLM.__new__(LlamaForCausalLM)
    torch.nn.Module.__init__(model)
    model.dtype = torch.bfloat16

    class Attn:
        head_dim, num_kv_heads = 128, 8

    class Layer(torch.nn.Module):
        self_attn = Attn

    model.layers = torch.nn.ModuleList([Layer()])
    monkeypatch.setattr(ops, "_force_torch", lambda: False)
    monkeypatch.setattr(ops, "paged_prefill_plan", lambda segs, device: ("plan", []))

    class Ids:
        is_cuda, device = True, "cpu"

    def planned(segs):
        batch = ForwardBatch(mode="decode", positions=None, slot_mapping=None, kv_caches=None, host_segs=segs,
                             seg_tables=torch.zeros(len(segs), 1))
        return (LlamaForCausalLM._planned(model, Ids, batch).plans or {}).get("paged")

    assert planned([(6000, 32)]) is None
    assert planned([(1536, 150)] * 8) == ("plan", [])


@pytest.mark.parametrize("shape,most", [((1024, 512), 64), ((28672, 4096), 64), ((27648, 5120), 16), ((57344, 8192), 0)])
def test_gate_up_product(shape, most):
    import torch

    from kllms_amd.models.llama import LlamaForCausalLM

    w = torch.empty(shape, dtype=torch.bfloat16, device="meta")
    assert [LlamaForCausalLM._silu_rows(r, w) for r in (1, 16, 17, 64, 65)] == [r <= most for r in (1, 16, 17, 64, 65)]

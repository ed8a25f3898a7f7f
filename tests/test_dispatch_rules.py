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


@pytest.mark.skipif(not ops.hip_available(), reason="the extension is not built")
@pytest.mark.parametrize("rows,kv_heads,group,keys,fp8,most", [
    (1, 8, 4, 384, 0, 1), (1, 8, 4, 512, 0, 4), (1, 8, 4, 2048, 0, 16), (2, 8, 4, 8192, 0, 16), (5, 8, 4, 8192, 0, 12),
    (1, 8, 4, 32768, 0, 32), (1, 4, 4, 131072, 0, 64), (1, 1, 4, 131072, 0, 64), (1, 1, 8, 131072, 0, 128),    # few long contexts
    (20, 8, 4, 8192, 0, 3), (20, 8, 4, 1000, 0, 1), (20, 8, 4, 1000, 1, 3), (40, 8, 4, 8192, 0, 3), (128, 8, 4, 8192, 0, 1),
    (11, 8, 1, 1024, 0, 8), (21, 8, 1, 1024, 1, 3), (21, 8, 2, 1024, 1, 3), (11, 8, 2, 1024, 0, 2),     # room for contexts that share a prompt
])
def test_shares_of_a_context(rows, kv_heads, group, keys, fp8, most):
    """Few contexts fill the chip also where they are long; no more partials than fit 1024 workgroups' room."""
    splits = ops._hip_or_raise().attn_decode_splits
    assert splits(rows, kv_heads, group, keys, fp8, 0, 1) == most
    for r in (1, 3, 17, 100, 255, 1000, 70000):
        for joined in (0, 1):
            z = splits(r, kv_heads, group, 1 << 20, fp8, 0, joined)
            assert z == 1 or r * kv_heads * z <= 1024


def test_one_short_portion_behind_a_long_cache_goes_row_by_row(monkeypatch):
    """The model asks the rules: a step of one 32-row portion has no plan, one of eight has, and its groups are as large as the
    other rule says."""
    import torch

    from kllms_amd.models.llama import ForwardBatch, LlamaForCausalLM

    model = LlamaForCausalLM.__new__(LlamaForCausalLM)
    torch.nn.Module.__init__(model)
    model.dtype = torch.bfloat16

    class Attn:
        head_dim, num_heads, num_kv_heads = 128, 32, 8

    class Layer(torch.nn.Module):
        self_attn = Attn

    model.layers = torch.nn.ModuleList([Layer()])
    monkeypatch.setattr(ops, "_force_torch", lambda: False)
    monkeypatch.setattr(ops, "paged_prefill_plan", lambda segs, device, rows=256: (("plan", rows), []))

    class Ids:
        is_cuda, device = True, "cpu"

    def planned(segs):
        batch = ForwardBatch(mode="decode", positions=None, slot_mapping=None, kv_caches=None, host_segs=segs,
                             seg_tables=torch.zeros(len(segs), 1))
        return (LlamaForCausalLM._planned(model, Ids, batch).plans or {}).get("paged")

    assert planned([(6000, 32)]) is None
    assert planned([(1536, 150)] * 8) == (("plan", 256), [])
    assert planned([(1536, 150)] * 2) == (("plan", 64), [])


@pytest.mark.parametrize("shape,most", [((1024, 512), 64), ((28672, 4096), 64), ((27648, 5120), 16), ((57344, 8192), 0)])
def test_gate_up_product(shape, most):
    import torch

    from kllms_amd.models.llama import LlamaForCausalLM

    w = torch.empty(shape, dtype=torch.bfloat16, device="meta")
    assert [LlamaForCausalLM._silu_rows(r, w) for r in (1, 16, 17, 64, 65)] == [r <= most for r in (1, 16, 17, 64, 65)]


def test_models_whose_steps_find_no_weights_in_the_cache():
    """Matrices count, tables and stacks of experts do not; the model says it to the parts that ask."""
    import torch

    from kllms_amd.engine.config import ModelArchConfig
    from kllms_amd.models.llama import LlamaForCausalLM
    from kllms_amd.models.mixtral import MixtralForCausalLM

    m = torch.nn.Module()
    with torch.device("meta"):
        m.table = torch.nn.Embedding(1 << 20, 256, dtype=torch.bfloat16)
        m.experts = torch.nn.Parameter(torch.empty(64, 4096, 4096, dtype=torch.bfloat16), requires_grad=False)
        m.a = torch.nn.Linear(4096, 20480, bias=False, dtype=torch.bfloat16)
        m.b = torch.nn.Linear(4096, 20479, bias=False, dtype=torch.bfloat16)
        assert not ops.weights_once(m)              # 8 KB less than 320 MB
        m.b = torch.nn.Linear(4096, 20480, bias=False, dtype=torch.bfloat16)
        assert ops.weights_once(m)
        sizes = dict(vocab_size=32000, hidden_size=2048, intermediate_size=8192, num_heads=16, num_kv_heads=4, head_dim=128)
        assert not LlamaForCausalLM(ModelArchConfig(num_layers=1, **sizes))._once      # 249 MB with the head
        assert LlamaForCausalLM(ModelArchConfig(num_layers=2, **sizes))._once          # 370 MB
        assert not MixtralForCausalLM(ModelArchConfig(num_layers=2, num_experts=8, **sizes))._once

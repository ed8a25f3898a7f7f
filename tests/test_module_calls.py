"""Fused calls that take a module's weights pass the module by only where nothing but its forward would run."""

import pytest
import torch
import torch.nn as nn

from kllms_amd import ops
from kllms_amd.engine.config import EngineConfig
from kllms_amd.engine.engine import LLMEngine


def _engine(model):
    return LLMEngine(EngineConfig(model=model, device="cpu", seed=0, use_hip_graphs=False, max_kv_blocks=64,
                                  enable_prefix_caching=False, eos_token_id=-1))


def _step(eng, n):
    s = eng.open_sequence()
    try:
        return eng.step_segments([(s, list(range(3, 3 + n)), [n - 1])])
    finally:
        eng.kv.free_sequence(s)


class _Adapter(nn.Module):
    """A projection with something added; no weight of its own to be taken."""

    def __init__(self, inner):
        super().__init__()
        self.inner, self.calls = inner, 0
        if hasattr(inner, "split"):
            self.split = inner.split

    def forward(self, x):
        self.calls += 1
        return self.inner(x)


def _fused(*a):
    raise AssertionError("the module was passed by")


@pytest.mark.parametrize("model,owner,name,op", [("tiny-llama", "mlp", "gate_up_proj", "linear_silu"),
                                                 ("tiny-zutalix", "mlp", "inp", "linear_clamped_glu")])
def test_projections_with_hooks_or_in_place_of_the_plain_one(monkeypatch, model, owner, name, op):
    eng = _engine(model)
    owners = [getattr(layer, owner) for layer in eng.model.layers if getattr(layer, owner) is not None]
    ref = _step(eng, 7)
    monkeypatch.setattr(ops, op, _fused)
    with pytest.raises(AssertionError, match="passed by"):
        _step(eng, 7)
    seen = []
    hooks = [getattr(m, name).register_forward_hook(lambda *a: seen.append(1)) for m in owners]
    assert torch.equal(_step(eng, 7), ref) and len(seen) == len(owners)
    for h in hooks:
        h.remove()
    plain = [getattr(m, name) for m in owners]
    for m in owners:
        setattr(m, name, _Adapter(getattr(m, name)))
    assert torch.equal(_step(eng, 7), ref) and all(getattr(m, name).calls == 1 for m in owners)
    for m, p in zip(owners, plain):
        setattr(m, name, p)
        p.forward = lambda x, p=p: type(p).forward(p, x)
    assert torch.equal(_step(eng, 7), ref)


@pytest.mark.parametrize("path", ["mix", "mix.inp", "mix.left", "mix.right", "mlp", "mlp.inp"])
def test_hybrid_rows_step_leaves_modules_with_hooks_alone(monkeypatch, path):
    eng = _engine("tiny-zutalix")
    ref = _step(eng, 1)
    monkeypatch.setattr(ops, "hybrid_rows_ok", lambda *a: True)
    for op in ("hybrid_parallel_rows", "hybrid_delta_rows", "hybrid_glu_rows"):
        monkeypatch.setattr(ops, op, _fused)
    seen, taken = [], []
    for layer in eng.model.layers:
        first, _, rest = path.partition(".")
        m = getattr(layer, first)
        if m is None or (rest and not hasattr(m, rest)):
            continue
        m.rows_ok = True
        (getattr(m, rest) if rest else m).register_forward_hook(lambda *a: seen.append(1))
        taken.append(layer)
    assert torch.equal(_step(eng, 1), ref) and len(seen) == len(taken) > 0


def test_hybrid_rows_step_with_other_modules_in_the_layers(monkeypatch):
    eng = _engine("tiny-zutalix")
    ref = _step(eng, 1)
    monkeypatch.setattr(ops, "hybrid_rows_ok", lambda *a: True)
    for layer in eng.model.layers:
        if layer.mlp is not None:
            layer.mlp = _Adapter(layer.mlp)
        if layer.kind != "parallel":
            mix = layer.mix
            layer.mix = nn.Module()
            layer.mix.inner = mix
            layer.mix.forward = mix.forward
    assert torch.equal(_step(eng, 1), ref)


def test_hybrid_rows_step_that_is_not_taken(monkeypatch):
    """The native sublayers give None where the weights lie otherwise than they read them."""
    eng = _engine("tiny-zutalix")
    ref = _step(eng, 1)
    monkeypatch.setattr(ops, "hybrid_rows_ok", lambda *a: True)
    for op in ("hybrid_parallel_rows", "hybrid_delta_rows", "hybrid_glu_rows"):
        monkeypatch.setattr(ops, op, lambda *a: None)
    for layer in eng.model.layers:
        for m in (layer.mix, layer.mlp):
            if m is not None:
                m.rows_ok = True
    assert torch.equal(_step(eng, 1), ref)

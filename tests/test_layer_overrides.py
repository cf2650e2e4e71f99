"""What a subclass of a layer overrides is what `apply` runs: the one foreign call stands only for the layer's own methods."""

import pytest
import torch

from dew_amd import gpt_oss, layer_call, moe

SIZES = {moe.SparseMLP: (8, 2, 128, 128), gpt_oss.GptOssMLP: (128, 128, 8, 2)}
VARIABLES = {"params": {"gate": {"kernel": None}, "router": {"kernel": None, "bias": None},
                        "experts": {"gate_up_proj_bias": 0, "down_proj_bias": 0}},
             "quantization": {"experts": {name: {"kernel": torch.empty(8, 128, 128)}
                                          for name in ("gate_proj", "up_proj", "down_proj", "gate_up_proj")}}}


@pytest.fixture
def one_call(monkeypatch):
    monkeypatch.setattr(layer_call, "forward", lambda *args, **kwargs: "one call")


class Overridden(Exception):
    pass


def raises(*args, **kwargs):
    raise Overridden


@pytest.mark.parametrize("kind", SIZES, ids=lambda kind: kind.__name__)
def test_a_layer_and_a_subclass_that_adds_to_it_take_the_one_call(one_call, kind):
    added = type("Added", (kind,), {"describe": lambda self: "more"})
    for layer in (kind(*SIZES[kind]), added(*SIZES[kind])):
        assert layer.apply(VARIABLES, torch.zeros(4, 128)) == "one call"


@pytest.mark.parametrize("kind,name", [(moe.SparseMLP, "__call__"), (moe.SparseMLP, "gate"), (moe.SparseMLP, "experts"),
                                       (gpt_oss.GptOssMLP, "__call__"), (gpt_oss.GptOssMLP, "logits"), (gpt_oss.GptOssMLP, "experts")])
def test_an_override_is_what_runs(one_call, monkeypatch, kind, name):
    held = raises if name in ("__call__", "logits") else property(raises)
    layer = type("Changed", (kind,), {name: held})(*SIZES[kind])
    monkeypatch.setattr(moe.Router, "__call__", lambda self, *args: (torch.zeros(4, 2), torch.zeros(4, 2, dtype=torch.int32)))
    monkeypatch.setattr(gpt_oss.ops, "route", lambda *args, **kwargs: (torch.zeros(4, 2), torch.zeros(4, 2, dtype=torch.int32)))
    monkeypatch.setattr(gpt_oss.ops, "router_logits", lambda *args, **kwargs: torch.zeros(4, 8))
    with pytest.raises(Overridden):
        layer.apply(VARIABLES, torch.zeros(4, 128))


def test_a_subclass_may_replace_the_shared_expert(one_call):
    layer = type("Changed", (moe.SparseMLP,), {"shared_experts": property(raises)})(*SIZES[moe.SparseMLP], shared=128)
    assert layer._one_call is None

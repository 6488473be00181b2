"""Observers and parameters are found wherever an ordinary attribute access finds them (no GPU)."""
import types

import pytest
import torch

from llmcompressor_amd.compressors import _tensors_of
from llmcompressor_amd.modifiers.quantization.calibration import observe, update_qparams


class Forwarding(torch.nn.Module):
    """A wrapper that answers for the module it holds, as adapter and offloading wrappers do."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def __getattr__(self, name):
        try:
            return super().__getattr__(name)
        except AttributeError:
            return getattr(super().__getattr__("inner"), name)


class WithProperty(torch.nn.Linear):
    @property
    def weight_zero_point(self):
        return self.bias


class Recorder(torch.nn.Module):
    """Stands in for an observer: what it was shown, and the parameters it answers with."""

    def __init__(self):
        super().__init__()
        self.seen = []
        self.args = types.SimpleNamespace(dynamic=False)
        self.has_statistics = True

    def forward(self, value):
        self.seen.append(value)

    def qparams_into(self, *params):
        return False

    def get_qparams(self):
        return {"scale": torch.full((1,), 3.0)}


def _linear(kind):
    """A module and the Linear behind it."""
    linear = torch.nn.Linear(4, 4)
    linear.register_parameter("weight_scale", torch.nn.Parameter(torch.zeros(1), requires_grad=False))
    observer = Recorder()
    if kind == "plain attribute":
        object.__setattr__(linear, "weight_observer", observer)
    else:
        linear.weight_observer = observer
    return (Forwarding(linear) if kind == "forwarded" else linear), linear, observer


@pytest.mark.parametrize("kind", ["submodule", "plain attribute", "forwarded"])
def test_observers_are_found_as_attributes(kind):
    module, linear, observer = _linear(kind)
    observe(module, "weight")
    assert len(observer.seen) == 1 and observer.seen[0] is linear.weight
    update_qparams(module, "weight")
    assert linear.weight_scale.item() == 3.0


def test_tensors_of_a_module_are_found_as_attributes():
    linear = torch.nn.Linear(4, 4)
    linear.register_buffer("weight_g_idx", torch.arange(4))
    linear.input_scale = torch.ones(1)  # neither parameter nor buffer
    for module in (linear, Forwarding(linear)):
        assert _tensors_of(module)("bias") is linear.bias
        assert _tensors_of(module)("weight_g_idx") is linear.weight_g_idx
        assert _tensors_of(module)("input_scale") is linear.input_scale
        assert _tensors_of(module)("weight_zero_point") is None
    assert _tensors_of(torch.nn.Linear(4, 4, bias=False))("bias") is None
    own = WithProperty(4, 4)
    assert _tensors_of(own)("weight_zero_point") is own.bias

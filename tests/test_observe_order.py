"""``observe`` of many modules: each weight is seen while its module is at hand and in the order of the call, whatever shares
a launch (reference: modifiers/quantization/calibration.py observes module by module)."""
import torch

from llmcompressor_amd.modifiers.quantization.calibration import observe
from llmcompressor_amd.observers import min_max


class _Recorder(torch.nn.Module):
    """An observer that keeps what it is shown."""

    def __init__(self):
        super().__init__()
        self.seen = []

    def forward(self, value):
        self.seen.append(value.detach().clone())


def _modules(n):
    out = []
    for i in range(n):
        m = torch.nn.Linear(64, 16, bias=False)
        torch.nn.init.constant_(m.weight, float(i + 1))
        m.weight_observer = _Recorder()
        out.append(m)
    return out


def test_modules_of_an_iterator_are_observed_one_at_a_time():
    """As a loop sees them that brings a module's weight in and takes it away again."""
    mods = _modules(3)

    def one_at_a_time():
        for m in mods:
            yield m
            m.weight.data.zero_()

    observe(one_at_a_time(), "weight")
    assert [int(m.weight_observer.seen[0][0, 0]) for m in mods] == [1, 2, 3]
    for m, v in zip(mods, (4.0, 5.0, 6.0)):
        m.weight.data.fill_(v)
    observe(mods, "weight")
    observe({m: None for m in mods}.keys(), "weight")
    assert [[int(s[0, 0]) for s in m.weight_observer.seen] for m in mods] == [[1, 4, 4], [2, 5, 5], [3, 6, 6]]


def test_an_observer_of_two_modules_sees_the_first_one_first(monkeypatch):
    """A weight's observer keeps the first value that it is shown; what could share a launch but finds no partner keeps its place."""
    monkeypatch.setattr(min_max, "_group_of", lambda observer, value: 64)
    first, second = _modules(2)
    second.weight_observer = first.weight_observer
    observe([first, second], "weight")
    assert [int(s[0, 0]) for s in first.weight_observer.seen] == [1, 2]

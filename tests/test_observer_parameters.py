"""Which parameters an observer writes in place, and which it leaves to the general path (no GPU: the operators are
replaced by recorders and the tensors only say which device they are on)."""
import types

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from llmcompressor_amd.observers import Observer, base
from llmcompressor_amd.quantization import preset_name_to_scheme


def _on(device, *shape, dtype=torch.bfloat16):
    with FakeTensorMode():
        return torch.empty(shape, dtype=dtype, device=device)


@pytest.mark.parametrize("preset,where", [("W8A16", {"scale": "cuda:1"}), ("W8A16", {"scale": "cpu"}), ("W8A16", {}),
                                          ("NVFP4A16", {"global_scale": "cuda:1"}), ("NVFP4A16", {"scale": "cuda:1"}),
                                          ("NVFP4A16", {"global_scale": "cpu"}), ("NVFP4A16", {})])
def test_parameters_of_another_device_are_left_to_the_general_path(monkeypatch, preset, where):
    """Statistics on one GPU and parameters on another: the general path copies, the in-place one steps back with
    nothing done."""
    calls = []
    monkeypatch.setattr(base, "llmc", types.SimpleNamespace(
        global_scale_into_=lambda *a: calls.append("global_scale"), qparams_into_=lambda *a: calls.append("qparams")))
    args = preset_name_to_scheme(preset, ["Linear"]).weights
    observer = Observer.load_from_registry("memoryless_minmax", base_name="weight", args=args)
    grouped = preset == "NVFP4A16"
    stats = (4, 2) if grouped else (4, 1)
    observer.update_statistics(_on("cuda:0", *stats), _on("cuda:0", *stats))
    scale = _on(where.get("scale", "cuda:0"), *stats, dtype=torch.float32 if grouped else torch.bfloat16)
    global_scale = _on(where.get("global_scale", "cuda:0"), 1, dtype=torch.float32) if grouped else None
    done = observer.qparams_into(scale, None, global_scale)
    assert done is (not where)
    assert calls == ([] if where else ["global_scale", "qparams"] if grouped else ["qparams"])
    assert observer.has_statistics is bool(where)


def test_statistics_that_a_subclass_registers_are_written_where_it_keeps_them():
    class Buffered(Observer):
        def __init__(self, **kw):
            super().__init__(**kw)
            self.register_buffer("min_vals", torch.zeros(2))
            self.register_buffer("max_vals", torch.zeros(2))

    args = preset_name_to_scheme("W8A16", ["Linear"]).weights
    observer = Buffered(base_name="weight", args=args)
    observer.update_statistics(torch.tensor([-1.0, -2.0]), torch.tensor([3.0, 4.0]))
    assert observer.state_dict()["min_vals"].tolist() == [-1.0, -2.0]
    assert observer.state_dict()["max_vals"].tolist() == [3.0, 4.0]
    observer.delete_statistics()
    assert not observer.has_statistics

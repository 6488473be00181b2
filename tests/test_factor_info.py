"""What callers do with a factorisation's ``info``: a failed pivot falls back to rounding with a warning
(gptq_quantize.py:157-164), a wait of the chain that gave up (negative) raises and changes nothing."""
import logging
from types import SimpleNamespace

import pytest
import torch

from llmcompressor_amd.modifiers.gptq import GPTQModifier
from llmcompressor_amd.modifiers.gptq import gptq_quantize
from llmcompressor_amd.modifiers.pruning.sparsegpt import sgpt_sparsify
from llmcompressor_amd.quantization import QuantizationArgs


def _native(info):
    """The operators that follow each other in a call, their results made up."""
    return SimpleNamespace(
        gptq_prepare_hinv_=lambda H, *a: (torch.zeros(H.shape[0], dtype=torch.uint8), torch.tensor([info], dtype=torch.int32)),
        gptq_quantize=lambda W, *a, **kw: (torch.zeros_like(W), torch.zeros(1)),
        sparsegpt_sparsify=lambda W, *a: (torch.zeros_like(W), torch.zeros(1)))


def _single(monkeypatch, info):
    monkeypatch.setattr(gptq_quantize, "llmc", _native(info))
    observer = SimpleNamespace(get_qparams=lambda: dict(scale=torch.ones(8, 1), zero_point=torch.zeros(8, 1, dtype=torch.int8),
                                                        global_scale=None))
    args = QuantizationArgs(num_bits=4, strategy="channel")
    return gptq_quantize.quantize_weight_tensors(torch.ones(8, 64), observer, args, torch.eye(64))[1]["weight"]


def _sets(monkeypatch, info):
    modules = [torch.nn.Linear(64, 8, bias=False) for _ in range(3)]
    before = [m.weight.detach().clone() for m in modules]
    infos = [0, info, 0]
    results = [(torch.zeros(()), {"weight": torch.zeros(8, 64)}, torch.tensor(i, dtype=torch.int32)) for i in infos]
    try:
        GPTQModifier(targets="Linear", scheme="W4A16")._finish_sets([(modules[:2], ["a", "b"], results[:2]),
                                                                   (modules[2:], ["c"], results[2:])])
    except RuntimeError:
        assert all(torch.equal(m.weight, w) for m, w in zip(modules, before))
        raise
    return torch.cat([m.weight.data for m in modules])


def _sparse(monkeypatch, info):
    monkeypatch.setattr(sgpt_sparsify, "llmc", _native(info))
    module = torch.nn.Linear(64, 8, bias=False)
    return sgpt_sparsify.sparsify_weight(module, {module: torch.eye(64)}, 0.5, 0, 0, 128, 0.01, False)[1]


@pytest.mark.parametrize("call", [_single, _sets, _sparse])
@pytest.mark.parametrize("info", [-1, 0, 5])
def test_info(monkeypatch, caplog, call, info):
    with caplog.at_level(logging.WARNING):
        if info < 0:
            with pytest.raises(RuntimeError, match="gave up waiting"):
                call(monkeypatch, info)
        else:
            assert not call(monkeypatch, info).any()
    assert ("Failed to invert hessian" in caplog.text) == (info > 0)

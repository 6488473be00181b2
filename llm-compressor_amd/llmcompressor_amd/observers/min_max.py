"""Min-max observers (reference: observers/min_max.py:10-74)."""
import torch
from torch.nn.modules import module as nn_module

from .. import _lib
from ..quantization import QuantizationStrategy
from ..torch_ops import llmc
from .base import Observer
from .helpers import lerp

__all__ = ["MemorylessMinMaxObserver", "StaticMinMaxObserver", "MinMaxObserver", "observe_weights_together"]


@Observer.register("memoryless_minmax")
class MemorylessMinMaxObserver(Observer):
    """min/max of the observed value."""


# what a call goes through before the statistics are kept, as a caller may have set it on one observer
_REPLACED = {"forward", "compute_min_max", "_min_max_kernel"}
_DTYPE_CODES = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}


def _group_of(observer, value):
    """Columns that share a scale, where calling ``observer`` on the weight ``value`` would do nothing but replace its
    statistics by the min-max of such groups (no hooks, no step replaced, no fused partner, nothing observed before); else 0."""
    if (type(observer) is not MemorylessMinMaxObserver or not observer.is_weight_obs or observer._forward_hooks
            or observer._forward_pre_hooks or nn_module._global_forward_hooks or nn_module._global_forward_pre_hooks
            or not _REPLACED.isdisjoint(observer.__dict__) or observer.has_statistics or observer._buffers or observer._parameters
            or observer.fusion_handler.is_fused):
        return 0
    if not (type(value) in (torch.Tensor, torch.nn.Parameter) and value.is_cuda and value.ndim == 2 and value.numel()
            and value.is_contiguous() and value.data_ptr() % 16 == 0 and value.dtype in _DTYPE_CODES):
        return 0
    args = observer.args
    if args.strategy == QuantizationStrategy.CHANNEL:
        return value.shape[1]
    if args.strategy in (QuantizationStrategy.GROUP, QuantizationStrategy.TENSOR_GROUP):
        return args.group_size if value.shape[1] % args.group_size == 0 else 0
    return 0


def observe_weights_together(observed):
    """``observer(value)`` for the pairs that can share a launch: weights of one shape and dtype in groups of one size (an MoE
    layer's experts, q / k / v, gate / up), whose statistics become slices of one tensor.  Returns the others, in their order."""
    sets, seen, done = {}, set(), set()
    for at, (observer, value) in enumerate(observed):
        group = 0 if observer in seen else _group_of(observer, value)
        seen.add(observer)
        # (slices of whole 16-byte vectors, int8 zero points' too: every kernel finds them as aligned as a tensor of their own)
        if group and value.shape[0] * (value.shape[1] // group) % 16 == 0:
            sets.setdefault((value.shape, value.dtype, value.device, group), []).append(at)
    for (shape, dtype, _, group), members in sets.items():
        if len(members) < 2 or not _lib.lib().llmc_minmax_groups_many_fits(_DTYPE_CODES[dtype], *shape, group):
            continue
        mins, maxs = llmc.minmax_observe_many([observed[at][1].detach() for at in members], group)
        for at, mn, mx in zip(members, mins.unbind(0), maxs.unbind(0)):
            observed[at][0].update_statistics(mn, mx)
        done.update(members)
    return [pair for at, pair in enumerate(observed) if at not in done]


@Observer.register("static_minmax")
class StaticMinMaxObserver(MemorylessMinMaxObserver):
    """min/max over everything observed so far."""

    def update_statistics(self, min_vals, max_vals):
        if hasattr(self, "min_vals"):
            min_vals = torch.min(min_vals, self.min_vals)
            max_vals = torch.max(max_vals, self.max_vals)
        self.min_vals, self.max_vals = min_vals, max_vals


@Observer.register("minmax")
class MinMaxObserver(Observer):
    """exponential moving average of min/max."""

    def __init__(self, *args, **kwargs):
        super().__init__(*args, **kwargs)
        self.avg_constant = self.args.observer_kwargs.get("averaging_constant", 0.01)

    def update_statistics(self, min_vals, max_vals):
        if hasattr(self, "min_vals") and self.avg_constant != 1.0:
            min_vals = lerp(self.min_vals, min_vals, self.avg_constant)
            max_vals = lerp(self.max_vals, max_vals, self.avg_constant)
        self.min_vals, self.max_vals = min_vals, max_vals

"""``torch.ops.llmc.*``: the C ABI of ``libllmc_amd.so`` registered with the torch dispatcher.

Every op is a thin shim: the registered implementation extracts ``data_ptr``, sizes, strides and the current HIP
stream from its tensor arguments and calls one plain ``extern "C"`` function of the library.  The ops of the short
calls (observers, scales, quantise / pack, one Hessian batch) are implemented natively in ``csrc/torch_bind.cpp``,
whose host time per call is a third of the interpreter's; the others are the functions of ``ops.py``.
The ops are registered for the CUDA (= HIP on ROCm) dispatch key only.  There is no CPU implementation on
purpose: a call with host tensors fails in the dispatcher ("could not run 'llmc::...' with arguments from the
'CPU' backend") instead of silently computing somewhere else.

Seams of the reference that the ops stand behind (src/llmcompressor/...):
``hessian_accum_`` -> accumulate_hessian (modifiers/gptq/gptq_quantize.py:28-64);
``gptq_prepare_hinv_`` / ``gptq_quantize`` -> quantize_weight (:144-164 / :167-250);
``minmax_observe*`` -> _get_min_max (observers/min_max.py:70-74); ``mse_observe*`` -> _grid_search_mse
(observers/mse_quant.py:19-141); ``qparams`` / ``global_scale`` -> Observer.get_qparams / get_global_scale
(observers/base.py:78-123); ``quant_pack`` -> fake_quantize / quantize / the compressors' pack step;
``fp8_dynamic_per_token`` -> forward_quantize with strategy "token" (modifiers/quantization/calibration.py:178-183).
"""
from __future__ import annotations

import os
from typing import List

import torch

from . import _lib
from . import ops as _impl

NAMESPACE = "llmc"

_defs = torch.library.Library(NAMESPACE, "DEF")
_cuda = torch.library.Library(NAMESPACE, "IMPL", "CUDA")

OP_NAMES: List[str] = []


def _register(schema: str, fn=None) -> None:
    """Define an op; without ``fn`` its implementation is in the native library."""
    name = schema.split("(", 1)[0]
    _defs.define(schema)
    if fn is None and not os.path.exists(_lib.BIND_PATH):
        fn = _lib.missing_native
    if fn is not None:
        _cuda.impl(name, fn)
    OP_NAMES.append(name)


# ---- GPTQ Hessian --------------------------------------------------------------------------------------------

def _hessian_accum_segments_(H, Xs, alpha=2.0, assume_symmetric=True):
    _impl.hessian_accumulate_segments_(H, list(Xs), alpha=alpha, assume_symmetric=assume_symmetric)


def _hessian_accum_grouped_(Hs, Xs, alpha=2.0, assume_symmetric=True):
    _impl.hessian_accumulate_grouped_(list(Hs), list(Xs), alpha=alpha, assume_symmetric=assume_symmetric)


_register("hessian_accum_(Tensor(a!) H, Tensor X, float alpha=2.0, bool assume_symmetric=True, "
          "bool use_workspace=True) -> ()")
_register("hessian_accum_counted_(Tensor(a!) H, Tensor X, Tensor(b!) count, float samples, float alpha=2.0, "
          "bool assume_symmetric=True, bool use_workspace=True) -> ()")
_register("hessian_accum_segments_(Tensor(a!) H, Tensor[] Xs, float alpha=2.0, bool assume_symmetric=True) -> ()",
          _hessian_accum_segments_)
_register("hessian_accum_grouped_(Tensor(a!)[] Hs, Tensor[] Xs, float alpha=2.0, bool assume_symmetric=True) -> ()",
          _hessian_accum_grouped_)


# ---- damped Cholesky chain and the column loop ------------------------------------------------------------------

def _gptq_prepare_hinv_(H, perm=None, divisor=1.0, percdamp=0.01, form=0):
    _, dead, info = _impl.gptq_hinv_(H, perm, divisor=divisor, percdamp=percdamp, form=form)
    return dead, info


def _gptq_prepare_hinv_grouped(Hs, perms=None, divisors=None, percdamp=0.01, form=0, n_inverse=0):
    return _impl.gptq_hinv_grouped(list(Hs), perms, None if divisors is None else list(divisors), percdamp, form=form,
                                   n_inverse=n_inverse)


def _gptq_quantize(W, Hinv, scale, zero_point, fmt, num_bits, row_div, scale_row_stride, g_idx=None, perm=None,
                   dead=None, global_scale=None, blocksize=128, form=0):
    return _impl.gptq_quantize(W, Hinv, scale, zero_point, fmt, num_bits, row_div, scale_row_stride, g_idx=g_idx,
                               perm=perm, dead=dead, global_scale=global_scale, blocksize=blocksize, form=form)


def _gptq_quantize_grouped(Ws, Hinv, scales, zero_points, fmt, num_bits, row_div, scale_row_stride, g_idxs=None,
                           perms=None, dead=None, global_scales=None, blocksize=128, form=0):
    outs, loss = _impl.gptq_quantize_grouped(
        list(Ws), Hinv, list(scales), None if zero_points is None else list(zero_points), fmt, num_bits, row_div,
        scale_row_stride, g_idxs=None if g_idxs is None else list(g_idxs), perms=perms, dead=dead,
        global_scales=None if global_scales is None else list(global_scales), blocksize=blocksize, form=form)
    return outs, loss


def _sparsegpt_sparsify(W, Hinv, sparsity, prune_n=0, prune_m=0, dead=None, blocksize=128,
                        preserve_sparsity_mask=False, form=0):
    return _impl.sparsegpt_sparsify(W, Hinv, sparsity, prune_n=prune_n, prune_m=prune_m, dead=dead,
                                    blocksize=blocksize, preserve_sparsity_mask=preserve_sparsity_mask, form=form)


_register("gptq_prepare_hinv_(Tensor(a!) H, Tensor? perm=None, float divisor=1.0, float percdamp=0.01, int form=0) "
          "-> (Tensor dead, Tensor info)", _gptq_prepare_hinv_)
_register("gptq_prepare_hinv_grouped(Tensor[] Hs, Tensor? perms=None, float[]? divisors=None, float percdamp=0.01, "
          "int form=0, int n_inverse=0) "
          "-> (Tensor U, Tensor dead, Tensor info)", _gptq_prepare_hinv_grouped)
_register("gptq_quantize(Tensor W, Tensor Hinv, Tensor scale, Tensor? zero_point, int fmt, int num_bits, int row_div, "
          "int scale_row_stride, Tensor? g_idx=None, Tensor? perm=None, Tensor? dead=None, Tensor? global_scale=None, "
          "int blocksize=128, int form=0) -> (Tensor weight, Tensor loss)", _gptq_quantize)
_register("gptq_quantize_grouped(Tensor[] Ws, Tensor Hinv, Tensor[] scales, Tensor[]? zero_points, int fmt, "
          "int num_bits, int row_div, int scale_row_stride, Tensor[]? g_idxs=None, Tensor? perms=None, "
          "Tensor? dead=None, Tensor[]? global_scales=None, int blocksize=128, int form=0) "
          "-> (Tensor[] weights, Tensor loss)",
          _gptq_quantize_grouped)
_register("sparsegpt_sparsify(Tensor W, Tensor Hinv, float sparsity, int prune_n=0, int prune_m=0, Tensor? dead=None, "
          "int blocksize=128, bool preserve_sparsity_mask=False, int form=0) -> (Tensor weight, Tensor loss)",
          _sparsegpt_sparsify)


# ---- observers ---------------------------------------------------------------------------------------------------

def _sumsq_accum_(total, x):
    _impl.sumsq_accumulate_(total, x)


def _sumsq_accum_noalloc_(total, x):
    _impl.sumsq_accumulate_noalloc_(total, x)


def _imatrix_observe(W, group, fmt, num_bits, symmetric, scale_mode=0, importance=None, maxshrink=0.95, patience=5,
                     grid=20.0, norm=3.0, expand=1.0):
    return _impl.imatrix_observe_groups(W, group, fmt, num_bits, symmetric, scale_mode, importance=importance,
                                        maxshrink=maxshrink, patience=patience, grid=grid, norm=norm, expand=expand)


def _imatrix_observe_blocks(W, block_h, block_w, fmt, num_bits, symmetric, scale_mode=0, maxshrink=0.95, patience=5,
                            grid=20.0, norm=3.0, expand=1.0):
    return _impl.imatrix_observe_blocks(W, block_h, block_w, fmt, num_bits, symmetric, scale_mode,
                                        maxshrink=maxshrink, patience=patience, grid=grid, norm=norm, expand=expand)


def _imatrix_observe_strided(x, n0, n1, group, stride0, stride1, fmt, num_bits, symmetric, scale_mode=0,
                             maxshrink=0.95, patience=5, grid=20.0, norm=3.0, expand=1.0):
    return _impl.imatrix_observe_strided(x, n0, n1, group, stride0, stride1, fmt, num_bits, symmetric, scale_mode,
                                         maxshrink=maxshrink, patience=patience, grid=grid, norm=norm, expand=expand)


_SEARCH = ("int fmt, int num_bits, bool symmetric, int scale_mode=0, float maxshrink=0.20, int patience=5, "
           "float grid=100.0, float norm=2.4, float expand=1.0) -> (Tensor min, Tensor max)")
_ISEARCH = ("float maxshrink=0.95, int patience=5, float grid=20.0, float norm=3.0, float expand=1.0) "
            "-> (Tensor min, Tensor max)")
_register("minmax_observe(Tensor W, int group, Tensor? workspace=None) -> (Tensor min, Tensor max)")
_register("minmax_observe_many(Tensor[] Ws, int group) -> (Tensor min, Tensor max)")
_register("minmax_observe_blocks(Tensor W, int block_h, int block_w) -> (Tensor min, Tensor max)")
_register("minmax_observe_strided(Tensor x, int n0, int n1, int group, int stride0, int stride1) "
          "-> (Tensor min, Tensor max)")
_register("mse_observe(Tensor W, int group, " + _SEARCH)
_register("mse_observe_blocks(Tensor W, int block_h, int block_w, " + _SEARCH)
_register("mse_observe_strided(Tensor x, int n0, int n1, int group, int stride0, int stride1, " + _SEARCH)
_register("sumsq_accum_(Tensor(a!) total, Tensor x) -> ()", _sumsq_accum_)
_register("sumsq_accum_noalloc_(Tensor(a!) total, Tensor x) -> ()", _sumsq_accum_noalloc_)
_register("imatrix_observe(Tensor W, int group, int fmt, int num_bits, bool symmetric, int scale_mode=0, "
          "Tensor? importance=None, " + _ISEARCH, _imatrix_observe)
_register("imatrix_observe_blocks(Tensor W, int block_h, int block_w, int fmt, int num_bits, bool symmetric, "
          "int scale_mode=0, " + _ISEARCH, _imatrix_observe_blocks)
_register("imatrix_observe_strided(Tensor x, int n0, int n1, int group, int stride0, int stride1, int fmt, "
          "int num_bits, bool symmetric, int scale_mode=0, " + _ISEARCH, _imatrix_observe_strided)


# ---- qparams, quantise, pack ---------------------------------------------------------------------------------------

_register("global_scale(Tensor[] mins, Tensor[] maxs) -> Tensor")
_register("global_scale_into_(Tensor[] mins, Tensor[] maxs, Tensor(a!) out) -> ()")
_register("qparams(Tensor min_vals, Tensor max_vals, int fmt, int num_bits, bool symmetric, int scale_mode=0, "
          "Tensor? global_scale=None, bool want_codes=False) -> (Tensor scale, Tensor zero_point, Tensor? scale_code)")
_register("qparams_into_(Tensor min_vals, Tensor max_vals, Tensor(a!) scale, Tensor(b!)? zero_point, int fmt, "
          "int num_bits, bool symmetric, int scale_mode=0, Tensor? global_scale=None) -> ()")
_QUANT = ("Tensor x, Tensor scale, Tensor? zero_point, int fmt, int num_bits, int row_div, int scale_row_stride, "
          "int col_div, int out_mode=0, Tensor? g_idx=None, Tensor? global_scale=None")
_register("quant_pack(" + _QUANT + ", ScalarType? out_dtype=None) -> Tensor")
_register("quant_pack_shaped(" + _QUANT + ") -> (Tensor out, Tensor shape)")
_register("fp8_dynamic_per_token(Tensor X, int fmt=1, int num_bits=8, int out_mode=0) -> (Tensor out, Tensor scale)")
_register("dynamic_token_quantize(Tensor x, int fmt, int num_bits) -> Tensor")
_register("dynamic_group_quantize(Tensor x, int group, int fmt, int num_bits, int scale_mode=0, "
          "Tensor? global_scale=None) -> Tensor")

if os.path.exists(_lib.BIND_PATH):
    torch.ops.load_library(_lib.BIND_PATH)


class _Ops:
    """The ops by name, each as its one overload: a packet looks its overload up at every call."""

    def __init__(self):
        packets = getattr(torch.ops, NAMESPACE)
        for name in OP_NAMES:
            setattr(self, name, getattr(packets, name).default)


llmc = _Ops()

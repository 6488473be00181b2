"""The native operators' argument checks, without a GPU.  The dispatcher picks the GPU implementation when any one
argument is on the GPU; here it is called directly, with fake tensors that say they are on one, so that an argument
that slips through a check fails on the missing device and never on a host pointer inside a kernel."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from llmcompressor_amd.torch_ops import llmc

CUDA_KEY = torch._C.DispatchKeySet(torch._C.DispatchKey.CUDA)
BIG = 1 << 40


def _host(*shape, dtype=torch.bfloat16):
    return torch.zeros(shape, dtype=dtype)


def _fake(device, *shape, dtype=torch.bfloat16):
    with FakeTensorMode():
        return torch.empty(shape, dtype=dtype, device=device)


def _call(name, *args):
    return getattr(llmc, name).redispatch(CUDA_KEY, *args)


def _spec():
    """Operator -> the (shape, dtype) of its tensors in order of the schema, and the call."""
    bf, f32, i8, i32 = torch.bfloat16, torch.float32, torch.int8, torch.int32
    W, S, ST = ((4, 32), bf), ((4, 1), bf), ((4, 2), bf)
    one = ((1,), f32)
    return {
        "hessian_accum_": ([((32, 32), f32), W], lambda H, x: (H, x)),
        "hessian_accum_counted_": ([((32, 32), f32), W, ((), f32)], lambda H, x, n: (H, x, n, 1.0)),
        "minmax_observe": ([W], lambda w: (w, 16)),
        "minmax_observe_blocks": ([W], lambda w: (w, 2, 16)),
        "minmax_observe_strided": ([W], lambda w: (w, 4, 1, 32, 32, 32)),
        "mse_observe": ([W], lambda w: (w, 16, 0, 4, True)),
        "mse_observe_blocks": ([W], lambda w: (w, 2, 16, 0, 4, True)),
        "mse_observe_strided": ([W], lambda w: (w, 4, 1, 32, 32, 32, 0, 4, True)),
        "global_scale": ([ST, ST, ST, ST], lambda a, b, c, d: ([a, b], [c, d])),
        "global_scale_into_": ([ST, ST, ST, ST, one], lambda a, b, c, d, o: ([a, b], [c, d], o)),
        "qparams": ([ST, ST, one], lambda a, b, g: (a, b, 2, 4, True, 1, g)),
        "qparams_into_": ([ST, ST, ((4, 2), f32), ((4, 2), i8), one],
                          lambda a, b, s, z, g: (a, b, s, z, 2, 4, True, 1, g)),
        "quant_pack": ([W, S, ((4, 1), i8), ((32,), i32), one],
                       lambda x, s, z, gi, g: (x, s, z, 0, 4, 1, 1, BIG, 0, gi, g)),
        "quant_pack_shaped": ([W, S, ((4, 1), i8), ((32,), i32), one],
                              lambda x, s, z, gi, g: (x, s, z, 0, 4, 1, 1, BIG, 2, gi, g)),
        "fp8_dynamic_per_token": ([W], lambda x: (x,)),
        "dynamic_token_quantize": ([W], lambda x: (x, 1, 8)),
        "dynamic_group_quantize": ([W, one], lambda x, g: (x, 16, 2, 4, 1, g)),
    }


@pytest.mark.parametrize("name,position", [(n, i) for n, (ts, _) in _spec().items() for i in range(len(ts))])
def test_a_host_tensor_in_any_place_is_refused(name, position):
    tensors, build = _spec()[name]
    args = [_host(*s, dtype=d) if i == position else _fake("cuda:0", *s, dtype=d) for i, (s, d) in enumerate(tensors)]
    with pytest.raises(RuntimeError, match="device tensors only; got a cpu tensor"):
        _call(name, *build(*args))


@pytest.mark.parametrize("name,position", [(n, i) for n, (ts, _) in _spec().items() for i in range(1, len(ts))])
def test_a_tensor_of_another_gpu_in_any_place_is_refused(name, position):
    tensors, build = _spec()[name]
    args = [_fake("cuda:1" if i == position else "cuda:0", *s, dtype=d) for i, (s, d) in enumerate(tensors)]
    with pytest.raises(RuntimeError, match="expected every tensor on cuda:"):
        _call(name, *build(*args))


def _stats(*sizes, dtype=torch.float32):
    return [_fake("cuda:0", n, dtype=dtype) for n in sizes]


@pytest.mark.parametrize("mins,maxs", [((4,), ()), ((4, 4), (4,)), ((4,), (4, 4)), ((), ())])
def test_global_scale_refuses_lists_that_do_not_pair_up(mins, maxs):
    out = _fake("cuda:0", 1, dtype=torch.float32)
    with pytest.raises(ValueError, match="one array of maxima per array of minima"):
        _call("global_scale_into_", _stats(*mins), _stats(*maxs), out)
    with pytest.raises(ValueError, match="one array of maxima per array of minima"):
        _call("global_scale", _stats(*mins), _stats(*maxs))


@pytest.mark.parametrize("mn,mx", [((8, torch.float32), (4, torch.float32)), ((4, torch.float32), (4, torch.bfloat16))])
def test_minima_and_maxima_of_another_size_or_dtype_are_refused(mn, mx):
    a, b = (_fake("cuda:0", n, dtype=d) for n, d in (mn, mx))
    for call in (lambda: _call("global_scale", [b, a], [b, b]), lambda: _call("qparams", a, b, 0, 4, True),
                 lambda: _call("qparams_into_", a, b, a, None, 0, 4, True)):
        with pytest.raises(ValueError, match="must agree in size and dtype"):
            call()


@pytest.mark.parametrize("shape", [(0,), (3, 0), (0, 0), ()])
def test_a_value_without_columns_is_refused(shape):
    x = _fake("cuda:0", *shape)
    for call in (lambda: _call("dynamic_token_quantize", x, 1, 8), lambda: _call("dynamic_group_quantize", x, 16, 1, 8)):
        with pytest.raises(ValueError, match="a value with columns"):
            call()


@pytest.mark.parametrize("maxshrink,grid", [(float("nan"), 100.0), (0.2, float("inf")), (1e300, 1e300)])
def test_a_search_range_that_is_not_finite_is_refused(maxshrink, grid):
    w = _fake("cuda:0", 4, 32)
    with pytest.raises(ValueError, match="not finite"):
        _call("mse_observe", w, 16, 0, 4, True, 0, maxshrink, 5, grid)


def _gptq_args(host):
    f32, bf = torch.float32, torch.bfloat16
    made = {"weight": ((4, 32), bf), "U": ((32, 32), f32), "scale": ((4, 1), bf), "zero_point": ((4, 1), torch.int8),
            "g_idx": ((32,), torch.int32), "perm": ((32,), torch.int32), "dead": ((32,), torch.uint8), "global_scale": ((1,), f32)}
    return {k: _host(*s, dtype=d) if k == host else _fake("cuda:0", *s, dtype=d) for k, (s, d) in made.items()}


@pytest.mark.parametrize("host", list(_gptq_args("")))
def test_the_column_loop_refuses_a_host_tensor_in_any_place(host):
    from llmcompressor_amd import ops

    a = _gptq_args(host)
    with pytest.raises(RuntimeError, match="device tensors only; got a cpu tensor"):
        ops.gptq_quantize(a["weight"], a["U"], a["scale"], a["zero_point"], 0, 4, 1, 1, g_idx=a["g_idx"], perm=a["perm"],
                          dead=a["dead"], global_scale=a["global_scale"])
    with pytest.raises(RuntimeError, match="device tensors only; got a cpu tensor"):
        ops.gptq_quantize_grouped([a["weight"]], a["U"][None], [a["scale"]], [a["zero_point"]], 0, 4, 1, 1,
                                  g_idxs=[a["g_idx"]], perms=a["perm"][None], dead=a["dead"][None],
                                  global_scales=[a["global_scale"]])

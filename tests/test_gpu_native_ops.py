"""GPU: the one-pass and whole-matrix kernels at the sizes where their indexing can go wrong -- one column chunk, rows
that are no multiple of 16 columns, the boundaries between the row kernels, ragged blocks, tails of a workgroup --
against the oracle, or against the separate kernels (themselves tested against it) that they stand in for."""
import pytest
import torch

from oracle import qformat as F

pytestmark = pytest.mark.gpu

BIG = 1 << 40


def _llmc():
    from llmcompressor_amd.torch_ops import llmc

    return llmc


def _values(rows, cols, dtype=torch.bfloat16, seed=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, cols, generator=g) * torch.logspace(-2, 1, cols)
    x[rows // 2] = 0.0
    return x.to(dtype)


@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 24), (257, 40), (5, 16), (700, 264), (64, 4104), (2, 13320)])
@pytest.mark.parametrize("scheme", ["int8", "int4", "fp8"])
def test_rows_of_eight_column_chunks(rows, cols, scheme):
    """Per-channel codes, packed words and fake-quantised values where K is a multiple of 8, and of 16 or not."""
    from llmcompressor_amd import ops

    args = F.QArgs(num_bits=8 if scheme != "int4" else 4, type="float" if scheme == "fp8" else "int", strategy="channel")
    x = _values(rows, cols)
    scale, zp = F.calculate_qparams(x.amin(1, keepdim=True), x.amax(1, keepdim=True), args)
    fmt = ops.FMT_FP8 if scheme == "fp8" else ops.FMT_INT
    for mode, want in ((ops.OUT_FAKEQUANT, F.fake_quantize(x, scale, zp, args)),
                       (ops.OUT_CODES, F.quantize(x, scale, zp, args, dtype=torch.float8_e4m3fn if scheme == "fp8" else torch.int8))):
        got = _llmc().quant_pack(x.cuda(), scale.cuda(), None, fmt, args.num_bits, 1, 1, BIG, mode).cpu()
        assert torch.equal(got.view(torch.uint8), want.to(got.dtype).view(torch.uint8))
    if scheme != "fp8":
        from oracle import pack as P

        got, shape = _llmc().quant_pack_shaped(x.cuda(), scale.cuda(), None, fmt, args.num_bits, 1, 1, BIG, ops.OUT_PACKED)
        assert shape.tolist() == [rows, cols]
        assert torch.equal(got.cpu(), P.pack_to_int32(F.quantize(x, scale, zp, args, dtype=torch.int8), args.num_bits))


@pytest.mark.parametrize("rows,cols,group", [(1, 16, 16), (3, 64, 32), (9, 128, 128), (130, 1024, 1024), (33, 3168, 32),
                                             (7, 2432, 128), (1, 14336, 128)])
@pytest.mark.parametrize("kind", ["fp8", "int8", "mxfp4", "nvfp4"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_dynamic_groups_in_one_pass_equal_the_three_kernels(rows, cols, group, kind, dtype):
    from llmcompressor_amd import ops

    llmc = _llmc()
    fmt, bits, mode = {"fp8": (ops.FMT_FP8, 8, ops.SCALE_PLAIN), "int8": (ops.FMT_INT, 8, ops.SCALE_PLAIN),
                       "mxfp4": (ops.FMT_FP4, 4, ops.SCALE_MXFP4), "nvfp4": (ops.FMT_FP4, 4, ops.SCALE_NVFP4)}[kind]
    x = _values(rows, cols, dtype).cuda()
    gs = torch.tensor([37.0], device="cuda") if kind == "nvfp4" else None
    if kind == "mxfp4" and dtype is torch.float16:
        with pytest.raises(ValueError):
            llmc.dynamic_group_quantize(x, group, fmt, bits, mode, gs)
        return
    mn, mx = llmc.minmax_observe(x, group)
    scale, _, codes = llmc.qparams(mn, mx, fmt, bits, True, mode, gs, kind == "mxfp4")
    want = llmc.quant_pack(x, codes if kind == "mxfp4" else scale, None, fmt, bits, 1, cols // group, group,
                           ops.OUT_FAKEQUANT, None, gs)
    got = llmc.dynamic_group_quantize(x.view(1, rows, cols), group, fmt, bits, mode, gs)
    assert got.shape == (1, rows, cols) and torch.equal(got[0], want)


@pytest.mark.parametrize("rows,cols", [(1, 8), (1, 4096), (3, 8192), (2, 8200), (1030, 1032), (5, 16384), (2, 16392),
                                       (1, 65536), (4, 100)])
@pytest.mark.parametrize("kind", ["float", "int"])
def test_dynamic_tokens_at_the_row_kernels_boundaries(rows, cols, kind):
    x = _values(rows, cols)
    args = F.QArgs(num_bits=8, type=kind, strategy="token", dynamic=True)
    want, _ = F.forward_quantize_dynamic(x.unsqueeze(0), args)
    got = _llmc().dynamic_token_quantize(x.cuda(), 1 if kind == "float" else 0, 8)
    assert torch.equal(got.cpu(), want[0])


@pytest.mark.parametrize("rows,cols,bh,bw", [(1, 8, 128, 128), (128, 128, 128, 128), (130, 264, 128, 128), (5, 20, 2, 3),
                                             (300, 1000, 64, 24)])
def test_block_min_max_on_ragged_edges(rows, cols, bh, bw):
    x = _values(rows, cols).abs() + 1  # the zero padding of an edge block is its minimum
    mn, mx = _llmc().minmax_observe_blocks(x.cuda(), bh, bw)
    p = torch.nn.functional.pad(x, (0, -cols % bw, 0, -rows % bh))
    p = p.view(p.shape[0] // bh, bh, p.shape[1] // bw, bw)
    assert torch.equal(mn.cpu(), p.amin((1, 3))) and torch.equal(mx.cpu(), p.amax((1, 3)))


@pytest.mark.parametrize("sizes", [(1,), (7,), (131072,), (131080,), (300001, 5), (5, 300001), (5, 9, 200000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_global_scale_over_arrays_of_any_size(sizes, dtype):
    g = torch.Generator().manual_seed(len(sizes))
    stats = []
    for i, n in enumerate(sizes):
        mn, mx = -torch.rand(n, generator=g), torch.rand(n, generator=g)
        (mn if i % 2 else mx)[n - 1] = (-40.0 if i % 2 else 40.0) - i  # the largest magnitude is the last value
        stats.append((mn.to(dtype), mx.to(dtype)))
    got = _llmc().global_scale([m.cuda() for m, _ in stats], [m.cuda() for _, m in stats])
    top = max(max(-mn.min().item(), mx.max().item()) for mn, mx in stats)
    want = (torch.tensor([top], dtype=dtype).reciprocal() * 2688.0).float()
    assert torch.equal(got.cpu(), want)


@pytest.mark.parametrize("scheme", ["W4A16", "W4A16_ASYM", "W8A8", "FP8_BLOCK", "NVFP4A16", "MXFP4A16"])
def test_parameters_written_in_place_equal_the_observers_own_answer(scheme):
    from llmcompressor_amd.modifiers.quantization.calibration import initialize_observer, observe, update_qparams
    from llmcompressor_amd.quantization import initialize_module_for_quantization, preset_name_to_scheme

    module = torch.nn.Linear(512, 96, bias=False, dtype=torch.bfloat16, device="cuda")
    initialize_module_for_quantization(module, preset_name_to_scheme(scheme, ["Linear"]))
    initialize_observer(module, "weight")
    observe(module, "weight")
    want = module.weight_observer.get_qparams()
    observe(module, "weight")
    update_qparams(module, "weight")
    assert not module.weight_observer.has_statistics
    for name in ("scale", "zero_point", "global_scale"):
        if want[name] is not None:
            got = getattr(module, f"weight_{name}").data
            assert torch.equal(got.float(), want[name].float()), name


@pytest.mark.parametrize("rows,cols", [(3, 24), (2, 257), (5, 511), (3, 513), (2, 1025), (1030, 600), (2, 6145), (1, 16384),
                                       (2, 16392)])
@pytest.mark.parametrize("scheme", ["int8", "int4_asym", "fp8"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_mse_search_over_long_groups(rows, cols, scheme, dtype):
    """One group per row, held in registers up to 16384 values: every boundary of the values per thread."""
    from llmcompressor_amd import ops
    from oracle import observers as O

    args = {"int8": F.QArgs(num_bits=8, strategy="channel"), "fp8": F.QArgs(num_bits=8, type="float", strategy="channel"),
            "int4_asym": F.QArgs(num_bits=4, strategy="channel", symmetric=False)}[scheme]
    g = torch.Generator().manual_seed(cols)
    w = (torch.randn(rows, cols, generator=g) * 0.02).to(dtype)
    mn, mx = _llmc().mse_observe(w.cuda(), cols, ops.FMT_FP8 if scheme == "fp8" else ops.FMT_INT, args.num_bits, args.symmetric)
    emn, emx = O.grid_search_mse(O.flatten_for_calibration(w, "weight", args), args)
    same = ((mn.cpu().reshape(-1) == emn.reshape(-1)) & (mx.cpu().reshape(-1) == emx.reshape(-1))).float().mean().item()
    # the sums of long groups run in another order than torch's, and rounded errors of neighbouring candidates tie
    assert same >= 0.99, same


@pytest.mark.parametrize("rows,cols,bh,bw", [(1, 8, 128, 128), (130, 136, 128, 128), (7, 20, 3, 5), (64, 48, 16, 24)])
def test_mse_search_over_blocks_equals_its_rows_form(rows, cols, bh, bw):
    """A block is searched like one row that holds its elements (zeros past the edges)."""
    from llmcompressor_amd import ops

    llmc = _llmc()
    x = _values(rows, cols)
    mn, mx = llmc.mse_observe_blocks(x.cuda(), bh, bw, ops.FMT_FP8, 8, True)
    p = torch.nn.functional.pad(x, (0, -cols % bw, 0, -rows % bh))
    p = p.view(p.shape[0] // bh, bh, p.shape[1] // bw, bw).transpose(1, 2).reshape(-1, bh * bw).contiguous()
    emn, emx = llmc.mse_observe(p.cuda(), bh * bw, ops.FMT_FP8, 8, True)
    if bh * bw % 8 == 0 and (bh * bw // 8) & (bh * bw // 8 - 1) == 0 and bh * bw <= 512:
        return  # such groups take the other kernel, whose sums run in another order
    assert torch.equal(mn.reshape(-1), emn.reshape(-1)) and torch.equal(mx.reshape(-1), emx.reshape(-1))


def test_dynamic_groups_of_one_very_wide_row():
    """2^28 columns in one row are 2^24 runs of 16: far below the 2^32 that the kernel numbers."""
    from llmcompressor_amd import ops

    llmc = _llmc()
    x = torch.randn(1, 1 << 28, device="cuda", dtype=torch.bfloat16)
    got = llmc.dynamic_group_quantize(x, 32, ops.FMT_FP8, 8)
    want = llmc.dynamic_group_quantize(x.view(1 << 14, -1), 32, ops.FMT_FP8, 8)
    assert torch.equal(got.view_as(want), want)


# 64 MiB is where the last rows come first: just below, just above with 0 to 7 blocks left over, a row of eight-column lanes
@pytest.mark.parametrize("rows,cols", [(8192, 4096), (8193, 4096), (8200, 4112), (9001, 4112), (8448, 4096), (16385, 2056)])
def test_large_inputs_from_the_end(rows, cols):
    """Every row of an input that is walked from its end has the values that it has in an input walked in order."""
    from llmcompressor_amd import ops

    llmc = _llmc()
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, cols, device="cuda", dtype=torch.bfloat16, generator=g)
    scale = torch.rand(rows, 1, device="cuda", generator=g).bfloat16() + 0.25
    parts = [slice(i, i + 4000) for i in range(0, rows, 4000)]
    for mode in (ops.OUT_FAKEQUANT, ops.OUT_CODES, ops.OUT_PACKED):
        quantised = [llmc.quant_pack(x[p], scale[p], None, ops.FMT_INT, 4, 1, 1, cols, mode, None, None) for p in [slice(None)] + parts]
        assert torch.equal(quantised[0], torch.cat(quantised[1:]))
    if cols % 16 == 0:
        dynamic = [llmc.dynamic_group_quantize(x[p], 16, ops.FMT_FP8, 8) for p in [slice(None)] + parts]
        assert torch.equal(dynamic[0], torch.cat(dynamic[1:]))


@pytest.mark.parametrize("form", ["lanes", "rows", "blocks"])
@pytest.mark.parametrize("symmetric", [True, False])
def test_mse_search_over_f16_rounds_the_shrunk_range_twice(form, symmetric):
    """The range times the shrink factor is an fp32 value before it is an f16 one.  Every f16 magnitude between 8 and 16
    where rounding the exact product to f16 at once gives another value, with one other value in its group (a sum of two
    does not depend on its order): 28 of the 4000 symmetric searches end elsewhere when rounded once."""
    from oracle import observers as O

    args = F.QArgs(num_bits=4, strategy="group", group_size=8, symmetric=symmetric)
    a = (torch.arange(1024) * 2.0 ** -7 + 8).half()
    factors = torch.tensor([1.0 - i / 100.0 for i in range(20)]).float()
    twice = (a.float()[:, None] * factors).half()
    step = torch.where(a[:, None].double() * factors.double() < 8, 2.0 ** -8, 2.0 ** -7)
    once = torch.round(a[:, None].double() * factors.double() / step) * step
    a = a[(twice.double() != once).any(1)]
    w = torch.zeros(4000, 8, dtype=torch.float16)
    w[:, 3] = -a[torch.arange(4000) % len(a)]
    w[:, 6] = ((torch.rand(4000, generator=torch.Generator().manual_seed(0)) * 2 - 1) * w[:, 3].float()).half()
    want = O.grid_search_mse(O.flatten_for_calibration(w, "weight", args), args)
    if form == "rows":  # two bytes off a 16-byte boundary
        x = torch.cat([w.view(-1)[:1], w.view(-1)]).cuda()[1:].view(4000, 8)
    else:
        x = w.cuda()
    got = (_llmc().mse_observe_blocks(x, 1, 8, 0, 4, symmetric) if form == "blocks"
           else _llmc().mse_observe(x, 8, 0, 4, symmetric))
    for g, e in zip(got, want):
        assert torch.equal(g.cpu().reshape(-1), e.reshape(-1)), (g.cpu().reshape(-1) != e.reshape(-1)).sum()

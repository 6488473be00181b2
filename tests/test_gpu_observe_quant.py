"""GPU parity (bit-exact): min-max observers, qparams, fake-quant and packed storage vs the CPU oracle."""
import pytest
import torch

from oracle import observers as O
from oracle import pack as P
from oracle import qformat as F

pytestmark = pytest.mark.gpu

E4M3 = torch.float8_e4m3fn


def _w(R, K, dtype=torch.bfloat16, seed=0, std=0.02):
    g = torch.Generator().manual_seed(seed)
    w = torch.randn(R, K, generator=g) * std
    w[0, 0] = 0.0
    if R > 1:
        w[1, :] = 0.0  # an all-zero row: zero scale -> epsilon substitution
    return w.to(dtype)


def _bits(t):
    if t.dtype == torch.float32:
        return t.view(torch.int32)
    if t.dtype in (torch.bfloat16, torch.float16):
        return t.view(torch.int16)
    return t


def _same(a, b):
    """bit-exact up to the sign of zero"""
    a, b = a.cpu(), b.cpu()
    assert a.shape == b.shape and a.dtype == b.dtype, (a.shape, b.shape, a.dtype, b.dtype)
    return torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("R,K,g", [(64, 512, 16), (64, 512, 32), (64, 512, 128), (64, 512, 512), (8, 56, 7),
                                   (3, 8200, 8200), (1, 64 * 512, 64 * 512), (5, 24, 3), (16, 4096, 4096)])
def test_minmax_groups(dtype, R, K, g):
    from llmcompressor_amd import ops

    w = _w(R, K, dtype, seed=R + K + g)
    mn, mx = ops.minmax_groups(w.cuda(), g)
    flat = w.unflatten(-1, (-1, g)).unsqueeze(0)
    emn, emx = O.get_min_max(flat)
    assert _same(mn, emn) and _same(mx, emx)


def test_minmax_tensor_large_and_blocks_and_strided():
    from llmcompressor_amd import ops

    w = _w(1024, 4096, seed=3)
    mn, mx = ops.minmax_groups(w.cuda().view(1, -1), w.numel())
    assert mn.item() == w.min().item() and mx.item() == w.max().item()
    for (R, K, bh, bw) in [(10, 8, 3, 3), (10, 8, 5, 4), (256, 512, 128, 128), (4, 6, 2, 3)]:
        w = _w(R, K, seed=R)
        args = F.QArgs(strategy="block", block_structure=[bh, bw])
        emn, emx = O.get_min_max(O.flatten_for_calibration(w, "weight", args))
        mn, mx = ops.minmax_blocks(w.cuda(), bh, bw)
        assert _same(mn, emn) and _same(mx, emx)
    x = _w(6 * 10, 64, seed=9, std=1.0).reshape(6, 10, 64)
    args = F.QArgs(strategy="group", group_size=16)
    emn, emx = O.get_min_max(O.flatten_for_calibration(x, "input", args))
    mn, mx = ops.minmax_strided(x.cuda(), 60, 4, 16, 64, 16)
    assert _same(mn, emn) and _same(mx, emx)


SCHEMES = {
    "int4_sym_g128": dict(num_bits=4, strategy="group", group_size=128),
    "int4_asym_g32": dict(num_bits=4, strategy="group", group_size=32, symmetric=False),
    "int8_sym_channel": dict(num_bits=8, strategy="channel"),
    "int8_asym_tensor": dict(num_bits=8, strategy="tensor", symmetric=False),
    "fp8_channel": dict(num_bits=8, type="float", strategy="channel"),
    "nvfp4": dict(num_bits=4, type="float", strategy="tensor_group", group_size=16, scale_dtype=E4M3),
    "mxfp4": dict(num_bits=4, type="float", strategy="group", group_size=32, scale_dtype=torch.uint8),
    "int4_block": dict(num_bits=4, strategy="block", block_structure=[128, 128]),
    "int3_g64": dict(num_bits=3, strategy="group", group_size=64),
}


def _fmt(args):
    from llmcompressor_amd import ops

    if args.type == "int":
        return ops.FMT_INT, args.num_bits
    return (ops.FMT_FP8, 8) if args.num_bits == 8 else (ops.FMT_FP4, 4)


def _gpu_pipeline(w, args, dtype):
    """observe -> qparams -> fake-quant / codes / packed, all through the C ABI."""
    from llmcompressor_amd import ops

    wg = w.cuda()
    R, K = w.shape
    s = args.strategy
    if s == "tensor":
        mn, mx = ops.minmax_groups(wg.view(1, -1), R * K)
        mn, mx = mn.view(1), mx.view(1)
        idx = (1 << 40, 0, 1 << 40)
    elif s == "channel":
        mn, mx = ops.minmax_groups(wg, K)
        idx = (1, 1, 1 << 40)
    elif s in ("group", "tensor_group"):
        mn, mx = ops.minmax_groups(wg, args.group_size)
        idx = (1, K // args.group_size, args.group_size)
    else:
        bh, bw = args.block_structure
        mn, mx = ops.minmax_blocks(wg, bh, bw)
        idx = (bh, (K + bw - 1) // bw, bw)
    fmt, bits = _fmt(args)
    mode = ops.SCALE_MXFP4 if args.is_mx else (ops.SCALE_NVFP4 if s == "tensor_group" and args.scale_dtype else ops.SCALE_PLAIN)
    gs = ops.global_scale_from_stats([(mn, mx)]) if s == "tensor_group" else None
    scale, zp, codes = ops.calculate_qparams(mn, mx, fmt, bits, args.symmetric, mode, gs, want_codes=mode != ops.SCALE_PLAIN)
    zpa = None if args.symmetric else zp
    fq = ops.quantize(wg, scale, zpa, fmt, bits, *idx, out_mode=ops.OUT_FAKEQUANT, global_scale=gs)
    cd = ops.quantize(wg, scale, zpa, fmt, bits, *idx, out_mode=ops.OUT_CODES, global_scale=gs)
    pk = ops.quantize(wg, scale, zpa, fmt, bits, *idx, out_mode=ops.OUT_PACKED, global_scale=gs)
    return dict(min=mn, max=mx, scale=scale, zp=zp, scale_codes=codes, gs=gs, fq=fq, codes=cd, packed=pk)


@pytest.mark.parametrize("name", list(SCHEMES))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rtn_pipeline_bit_exact(name, dtype):
    args = F.QArgs(**SCHEMES[name])
    if args.is_mx and dtype != torch.bfloat16:
        # the exponent rule reads the bf16 bit pattern of the group maximum: other dtypes are refused, not guessed
        from llmcompressor_amd.quantization import QuantizationArgs
        from llmcompressor_amd.quantization.lifecycle import calculate_qparams

        stats = torch.ones(4, 2, dtype=dtype, device="cuda")
        qa = QuantizationArgs(num_bits=4, type="float", strategy="group", group_size=32, scale_dtype="uint8")
        with pytest.raises(TypeError, match="bfloat16 statistics"):
            calculate_qparams(-stats, stats, qa)
        return
    w = _w(256, 512, dtype, seed=len(name), std=0.05)
    w[7, 100] = 3.0  # outlier
    got = _gpu_pipeline(w, args, dtype)

    obs = O.Observer("memoryless_minmax", "weight", args)
    obs(w)
    assert _same(got["min"], obs.min_vals) and _same(got["max"], obs.max_vals)
    qp = obs.get_qparams()
    scale, zp, gs = qp["scale"], qp["zero_point"], qp["global_scale"]
    assert _same(got["scale"], scale), name
    if not args.symmetric:
        assert _same(got["zp"], zp.to(torch.int8))
    if gs is not None:
        assert _same(got["gs"], gs)
    exp_fq = F.fake_quantize(w, scale, zp, args, global_scale=gs)
    assert _same(got["fq"], exp_fq.to(dtype)), name

    if args.type == "int":
        codes = F.quantize(w, scale, zp, args, dtype=torch.int8)
        assert _same(got["codes"], codes)
        assert _same(got["packed"], P.pack_to_int32(codes, args.num_bits))
        assert torch.equal(P.unpack_from_int32(got["packed"].cpu(), args.num_bits, w.shape), codes)
    elif args.num_bits == 8:
        q8 = F.quantize(w, scale, zp, args, dtype=E4M3)
        assert torch.equal(got["codes"].cpu().view(torch.uint8), q8.view(torch.uint8))
        assert torch.equal(got["packed"].cpu().view(torch.uint8), q8.view(torch.uint8))
    else:
        q4 = F.quantize(w, scale, zp, args, global_scale=gs)
        exp_pk = P.pack_fp4_to_uint8(q4)
        assert _same(got["packed"], exp_pk), name
        if args.is_mx:
            exp_codes = (torch.log2(scale.float()) + 127).to(torch.uint8)
        else:
            exp_codes = scale.to(E4M3).view(torch.uint8)
        assert _same(got["scale_codes"], exp_codes)


def test_quantize_with_g_idx_and_fp32_input():
    """GPTQ-style call: fp32 weights, bf16 scales, column -> group map through g_idx."""
    from llmcompressor_amd import ops

    torch.manual_seed(0)
    R, K, g = 32, 256, 64
    w = _w(R, K, torch.bfloat16, seed=11, std=0.05)
    args = F.QArgs(num_bits=4, strategy="group", group_size=g)
    obs = O.Observer("memoryless_minmax", "weight", args)
    obs(w)
    qp = obs.get_qparams()
    perm = torch.randperm(K)
    g_idx = (torch.arange(K, dtype=torch.int32) // g)[perm]
    wp = w[:, perm].float().contiguous()
    got = ops.quantize(wp.cuda(), qp["scale"].cuda(), None, ops.FMT_INT, 4, 1, K // g, 1, g_idx=g_idx.cuda(),
                       out_dtype=torch.bfloat16)
    chan = args.copy(strategy="channel")
    exp = torch.stack([F.fake_quantize(wp[:, j], qp["scale"][:, g_idx[j]], qp["zero_point"][:, g_idx[j]], chan)
                       for j in range(K)], dim=1)
    assert exp.dtype == torch.bfloat16
    assert _same(got, exp)


@pytest.mark.parametrize("case", ["int4_bf16scale", "int8_asym_bf16scale", "fp8_f32scale", "fp4_bf16scale", "fp4_gscale"])
def test_quantize_every_bf16_value_and_extreme_scales(case):
    """Every finite-or-infinite bf16 bit pattern as a dividend, against per-row scales from 2^-100 to 2^100:
    the shared-divisor division of the row kernel must give the bytes the plain division gives
    (quotients that overflow, underflow, hit ties or vanish included).  NaN inputs are left out:
    the reference's integer cast of NaN is not defined."""
    from llmcompressor_amd import ops

    bits = torch.arange(65536, dtype=torch.int32)
    exp_field = (bits >> 7) & 0xFF
    keep = ~((exp_field == 0xFF) & ((bits & 0x7F) != 0))
    vals = bits[keep].to(torch.int16).view(torch.bfloat16)  # 65282 values
    K = 256
    vals = vals[: (vals.numel() // K) * K]
    g = torch.Generator().manual_seed(3)
    vals = vals[torch.randperm(vals.numel(), generator=g)]
    w = vals.view(-1, K).repeat(4, 1).contiguous()  # every value meets several scales
    R = w.shape[0]
    exps = torch.tensor([-100.0, -70.0, -61.0, -59.0, -40.0, -20.0, -9.0, -5.5, -1.0, 0.0, 0.3, 3.0, 11.0, 40.0, 59.0, 61.0, 100.0])
    sc = torch.exp2(exps[torch.arange(R) % exps.numel()]) * (1.0 + torch.rand(R, generator=g))
    kw = dict(global_scale=None)
    zp = None
    if case == "int4_bf16scale":
        args, fmt, nb, scale = F.QArgs(num_bits=4, strategy="channel"), ops.FMT_INT, 4, sc.bfloat16()
    elif case == "int8_asym_bf16scale":
        args, fmt, nb, scale = F.QArgs(num_bits=8, strategy="channel", symmetric=False), ops.FMT_INT, 8, sc.bfloat16()
        zp = torch.randint(-128, 128, (R, 1), generator=g).to(torch.int8)
    elif case == "fp8_f32scale":
        args, fmt, nb, scale = F.QArgs(num_bits=8, type="float", strategy="channel"), ops.FMT_FP8, 8, sc.float()
    elif case == "fp4_bf16scale":
        args, fmt, nb, scale = F.QArgs(num_bits=4, type="float", strategy="channel"), ops.FMT_FP4, 4, sc.bfloat16()
    else:
        args, fmt, nb = F.QArgs(num_bits=4, type="float", strategy="channel"), ops.FMT_FP4, 4
        scale = sc.clamp(min=2.0**-9, max=448.0).to(E4M3).float()  # an e4m3 scale is never stored as zero
        kw = dict(global_scale=torch.tensor([37.25]))
    scale = scale.view(R, 1)
    ozp = zp.to(scale.dtype) if zp is not None else torch.zeros_like(scale)
    exp_fq = F.fake_quantize(w, scale, ozp, args, **kw)
    gkw = {k: (v.cuda() if v is not None else None) for k, v in kw.items()}
    gzp = zp.cuda() if zp is not None else None
    fq = ops.quantize(w.cuda(), scale.cuda(), gzp, fmt, nb, 1, 1, 1 << 40, out_mode=ops.OUT_FAKEQUANT, **gkw)
    fin = torch.isfinite(exp_fq.float())
    assert torch.equal(torch.isfinite(fq.float().cpu()), fin)
    assert torch.equal(_bits(fq.cpu())[fin], _bits(exp_fq.to(torch.bfloat16))[fin]), case
    pk = ops.quantize(w.cuda(), scale.cuda(), gzp, fmt, nb, 1, 1, 1 << 40, out_mode=ops.OUT_PACKED, **gkw)
    if fmt == ops.FMT_INT:
        codes = F.quantize(w, scale, ozp, args, dtype=torch.int8)
        assert _same(pk, P.pack_to_int32(codes, nb)), case
    elif fmt == ops.FMT_FP8:
        q8 = F.quantize(w, scale, ozp, args, dtype=E4M3)
        assert torch.equal(pk.cpu().view(torch.uint8), q8.view(torch.uint8))
    else:
        q4 = F.quantize(w, scale, ozp, args, **kw)
        assert _same(pk, P.pack_fp4_to_uint8(q4)), case


@pytest.mark.parametrize("N,K", [(64, 4096), (7, 100), (3, 12288), (5, 512), (9, 8192), (6, 1000)])
def test_dynamic_per_token_fp8(N, K):
    from llmcompressor_amd import ops

    torch.manual_seed(N)
    x = torch.randn(N, K)
    mask = torch.rand(N, K) < 0.02
    x[mask] = torch.distributions.StudentT(3.0).sample((int(mask.sum()),))
    x[0] = 0
    x = x.bfloat16()
    args = F.QArgs(num_bits=8, type="float", strategy="token", dynamic=True)
    exp_fq, exp_scale = F.forward_quantize_dynamic(x.unsqueeze(0), args)
    fq, scale = ops.dynamic_per_token_quantize(x.cuda())
    assert _same(scale, exp_scale[0])
    assert _same(fq, exp_fq[0])
    codes, _ = ops.dynamic_per_token_quantize(x.cuda(), out_mode=ops.OUT_CODES)
    exp_codes = F.quantize(x.unsqueeze(0), exp_scale, None, args, dtype=E4M3)[0]
    assert torch.equal(codes.cpu().view(torch.uint8), exp_codes.view(torch.uint8))


def test_full_size_properties():
    """Config-2/3 shapes: properties that do not need the (slow) oracle at full size."""
    from llmcompressor_amd import ops

    torch.manual_seed(0)
    w = (torch.randn(14336, 4096, device="cuda") * 0.02).bfloat16()
    # idempotence: fake-quantising a fake-quantised weight with the same qparams is a fixed point
    mn, mx = ops.minmax_groups(w, 128)
    scale, _, _ = ops.calculate_qparams(mn, mx, ops.FMT_INT, 4, True)
    fq = ops.quantize(w, scale, None, ops.FMT_INT, 4, 1, 4096 // 128, 128)
    fq2 = ops.quantize(fq, scale, None, ops.FMT_INT, 4, 1, 4096 // 128, 128)
    assert torch.equal(fq, fq2)
    # pack -> unpack -> dequantise reproduces the fake-quantised weight
    pk = ops.quantize(w, scale, None, ops.FMT_INT, 4, 1, 4096 // 128, 128, out_mode=ops.OUT_PACKED)
    shifts = torch.arange(8, device="cuda", dtype=torch.int32) * 4
    codes = (((pk.unsqueeze(-1) >> shifts) & 15) - 8).reshape(14336, 4096)
    deq = (codes.to(torch.bfloat16).unflatten(-1, (-1, 128)) * scale.unsqueeze(-1)).flatten(-2)
    assert torch.equal(deq, fq)
    # min/max against torch on the same device
    assert torch.equal(mn, w.unflatten(-1, (-1, 128)).amin(-1)) and torch.equal(mx, w.unflatten(-1, (-1, 128)).amax(-1))
    # fp8 per-channel: codes decode to the fake-quantised weight
    mn, mx = ops.minmax_groups(w, 4096)
    s8, _, _ = ops.calculate_qparams(mn, mx, ops.FMT_FP8, 8, True)
    fq8 = ops.quantize(w, s8, None, ops.FMT_FP8, 8, 1, 1, 1 << 40)
    c8 = ops.quantize(w, s8, None, ops.FMT_FP8, 8, 1, 1, 1 << 40, out_mode=ops.OUT_PACKED)
    assert torch.equal((c8.to(torch.bfloat16) * s8), fq8)


def test_full_size_microscale_and_mse_properties():
    """Config-3 shapes (14336 x 4096): NVFP4 / MXFP4 packed bytes decode to the fake-quantised weight;
    the MSE observer's ranges lie inside the min-max ranges and do not quantise worse than min-max."""
    from llmcompressor_amd import ops

    torch.manual_seed(1)
    R, K = 14336, 4096
    w = (torch.randn(R, K, device="cuda") * 0.02).bfloat16()
    e2m1 = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], device="cuda")
    grid = torch.cat([e2m1, -e2m1])

    def decode(pk):
        lo, hi = (pk & 0xF).long(), (pk >> 4).long()
        return torch.stack([grid[lo], grid[hi]], dim=-1).reshape(R, K)

    # NVFP4: group 16, e4m3 scales times a global scale
    mn, mx = ops.minmax_groups(w, 16)
    gs = ops.global_scale_from_stats([(mn, mx)])
    s4, _, codes = ops.calculate_qparams(mn, mx, ops.FMT_FP4, 4, True, ops.SCALE_NVFP4, gs, want_codes=True)
    assert torch.equal(codes.view(torch.float8_e4m3fn).float(), s4.float())  # stored scales are e4m3 values
    fq = ops.quantize(w, s4, None, ops.FMT_FP4, 4, 1, K // 16, 16, global_scale=gs)
    pk = ops.quantize(w, s4, None, ops.FMT_FP4, 4, 1, K // 16, 16, out_mode=ops.OUT_PACKED, global_scale=gs)
    eff = (s4.float() / gs).repeat_interleave(16, dim=1)
    assert torch.equal((decode(pk) * eff).to(torch.bfloat16), fq)
    fq2 = ops.quantize(fq, s4, None, ops.FMT_FP4, 4, 1, K // 16, 16, global_scale=gs)
    assert torch.equal(fq2, fq)  # idempotent
    # MXFP4: group 32, power-of-two scales
    mn, mx = ops.minmax_groups(w, 32)
    sm, _, e8 = ops.calculate_qparams(mn, mx, ops.FMT_FP4, 4, True, ops.SCALE_MXFP4, want_codes=True)
    assert torch.equal(torch.exp2(e8.float() - 127).to(torch.bfloat16), sm)
    fqm = ops.quantize(w, sm, None, ops.FMT_FP4, 4, 1, K // 32, 32)
    pkm = ops.quantize(w, sm, None, ops.FMT_FP4, 4, 1, K // 32, 32, out_mode=ops.OUT_PACKED)
    assert torch.equal((decode(pkm) * sm.float().repeat_interleave(32, dim=1)).to(torch.bfloat16), fqm)
    # MSE observer (default grid) vs min-max, int4 group 128
    mn, mx = ops.minmax_groups(w, 128)
    mmn, mmx = ops.mse_observe_groups(w, 128, ops.FMT_INT, 4, True, ops.SCALE_PLAIN)
    assert bool((mmn >= mn).all()) and bool((mmx <= mx).all())

    def qerr(a, b):
        s, _, _ = ops.calculate_qparams(a, b, ops.FMT_INT, 4, True)
        f = ops.quantize(w, s, None, ops.FMT_INT, 4, 1, K // 128, 128)
        return (f.float() - w.float()).abs().pow(2.4).sum().item()

    assert qerr(mmn, mmx) <= 1.0001 * qerr(mn, mx)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_global_scale_matches_oracle_for_many_absmax_values(dtype):
    """The NVFP4 global scale for 600 absmax values per statistics dtype, bit for bit against the oracle
    (reciprocal rounded to the dtype, then the product rounded again)."""
    from llmcompressor_amd import ops

    torch.manual_seed(4)
    vals = torch.cat([torch.rand(300) * 60 + 0.01, torch.rand(200) * 2.0 ** -6, torch.tensor([40.0, 23.0, 11.0]),
                      torch.rand(97) * 3000]).to(dtype)
    bad = []
    for v in vals:
        t = v.reshape(1)
        want = F.generate_gparam(-t, t).item()
        got = ops.global_scale_from_stats([(-t.cuda(), t.cuda())]).item()
        if got != want:
            bad.append((v.item(), got, want))
    assert not bad, bad[:5]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_global_scale_in_two_steps_equals_the_one_call(dtype):
    """llmc_absmax_accumulate over every array and llmc_generate_gparam, for callers of the C ABI that keep the cell."""
    from llmcompressor_amd import _lib, ops

    torch.manual_seed(5)
    arrays = [torch.randn(n, device="cuda").to(dtype) for n in (1, 2055, 70000)]
    stats = [(-t.abs(), t.abs() * 0.5) for t in arrays]
    lib, st = _lib.lib(), torch.cuda.current_stream().cuda_stream
    cell, out = torch.zeros(1, device="cuda"), torch.empty(1, device="cuda")
    for mn, mx in stats:
        assert lib.llmc_absmax_accumulate(mn.data_ptr(), mx.data_ptr(), mn.numel(), ops._DT[dtype], cell.data_ptr(), st) == 0
    assert lib.llmc_generate_gparam(cell.data_ptr(), ops._DT[dtype], out.data_ptr(), st) == 0
    assert torch.equal(out, ops.global_scale_from_stats(stats))

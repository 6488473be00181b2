"""GPU: llmc_sgemm, the fp32 product of the lazy trailing updates (W[:, i2:] -= Err1 @ Hinv[i1:i2, i2:],
gptq_quantize.py:245, and the products inside the Cholesky chain), through the C ABI against an fp64 product.

Tolerance: relative Frobenius error <= 2e-6 (fp32 accumulation over up to 2048 terms), and the split product on
the 16-bit matrix cores must be at least as accurate as 1.5 x the fp32 matrix instruction's error on the same
operands -- the property that lets it stand in for fp32 inside the Cholesky chain."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(M, N, Kc, trans_b, flags, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    # rows of very different magnitude, as the panels of a Cholesky factor have
    A = torch.randn(M, Kc, device="cuda", generator=g) * torch.exp(2 * torch.randn(M, 1, device="cuda", generator=g))
    Bp = torch.randn(Kc, N, device="cuda", generator=g)
    if flags & 2:
        A = torch.tril(A)
    if flags & 4:
        Bp = torch.tril(Bp)
    B = Bp.t().contiguous() if trans_b else Bp.contiguous()
    C0 = torch.randn(M, N, device="cuda", generator=g)
    return A, B, Bp, C0


@pytest.mark.parametrize("M,N,Kc,trans_b,flags,alpha,beta", [
    (256, 512, 128, True, 0, -1.0, 1.0),      # 128-wide tiles, split
    (256, 512, 128, False, 0, -1.0, 1.0),
    (2048, 4096, 512, False, 0, -1.0, 1.0),   # 256-wide tiles, split: the rank-512 update of the column loop
    (4096, 4096, 256, True, 1, -1.0, 1.0),    # trailing update of the factorisation (lower triangle only)
    (1024, 2048, 2048, False, 4, 1.0, 0.0),   # inverse, first product (B lower triangular)
    (1024, 2048, 1024, False, 2, -1.0, 0.0),  # inverse, second product (A lower triangular)
    (200, 328, 72, True, 0, 0.5, 2.0),        # ragged: fp32 matrix instruction
    (64, 64, 64, False, 0, 1.0, 0.0),         # too small to split
])
def test_sgemm_matches_fp64(M, N, Kc, trans_b, flags, alpha, beta):
    from llmcompressor_amd import ops

    A, B, Bp, C0 = _operands(M, N, Kc, trans_b, flags, seed=M + N + Kc + flags)
    ref = alpha * (A.double() @ Bp.double()) + beta * C0.double()
    errs = {}
    for name, extra in (("auto", 0), ("fp32", ops.SGEMM_FP32_MFMA)):
        C = C0.clone()
        ops.sgemm_(C, A, B, alpha, beta, trans_b, flags | extra)
        if flags & ops.SGEMM_C_LOWER:
            low = torch.tril(torch.ones(M, N, dtype=torch.bool, device="cuda"))
            assert torch.equal(C[~low], C0[~low])  # nothing above the diagonal is written
            errs[name] = ((C.double() - ref)[low].norm() / ref[low].norm()).item()
        else:
            errs[name] = ((C.double() - ref).norm() / ref.norm()).item()
    print(f"rel err auto {errs['auto']:.2e} fp32 {errs['fp32']:.2e}")
    assert errs["auto"] <= 2e-6 and errs["fp32"] <= 2e-6
    assert errs["auto"] <= 1.5 * errs["fp32"] + 1e-8


@pytest.mark.parametrize("M,N,Kc", [(64, 64, 512), (192, 64, 544), (256, 256, 1024), (128, 1024, 512), (4160, 512, 512)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_sgemm_below_sixteen_large_tiles_is_closer_than_the_fp32_instruction(M, N, Kc, trans_b):
    """These products round their whole sum once per 16 k where the fp32 instruction rounds it 16 times: a quarter of
    its error if every rounding is to nearest, half of it if the matrix instruction's own rounding truncates."""
    from llmcompressor_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M + N + Kc)
    A, Bp = torch.randn(M, Kc, device="cuda", generator=g), torch.randn(Kc, N, device="cuda", generator=g)
    B = Bp.t().contiguous() if trans_b else Bp
    ref = A.double() @ Bp.double()
    errs = []
    for flags in (0, ops.SGEMM_FP32_MFMA):
        C = ops.sgemm_(torch.empty(M, N, device="cuda"), A, B, trans_b=trans_b, flags=flags)
        errs.append((C.double() - ref).norm().item())
    assert errs[0] <= 0.5 * errs[1], (errs[0] / errs[1])


def test_sgemm_rejects_bad_arguments():
    from llmcompressor_amd import _lib

    lib = _lib.lib()
    a = torch.zeros(8, 8, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    assert lib.llmc_sgemm(0, 8, a.data_ptr(), 8, a.data_ptr(), 8, 8, 8, 8, 1.0, 0.0, 0, 0, st) == -1
    assert lib.llmc_sgemm(a.data_ptr(), 8, a.data_ptr(), 8, a.data_ptr(), 4, 8, 8, 8, 1.0, 0.0, 0, 0, st) == -5
    assert lib.llmc_sgemm(a.data_ptr(), 8, a.data_ptr(), 8, a.data_ptr(), 8, 8, 8, 8, 1.0, 0.0, 0, 64, st) == -13


@pytest.mark.parametrize("M,N,Kc,trans_b,flags,alpha,beta", [
    (64, 64, 256, False, 0, 1.0, 0.0),      # one tile of the fp32 instruction
    (64, 192, 288, True, 0, -1.0, 1.0),
    (192, 320, 352, False, 0, -1.0, 1.0),
    (448, 448, 256, True, 1, -1.0, 1.0),    # lower triangle only, diagonal tiles
    (320, 256, 256, False, 4, 1.0, 0.0),
    (256, 320, 256, False, 2, -1.0, 0.0),
    (64, 64, 512, False, 0, 1.0, 0.0),      # split: one tile, as few k-steps as it takes with two sums
    (64, 192, 544, True, 0, -1.0, 1.0),     # a contraction that is no multiple of the four steps in flight
    (192, 320, 608, False, 0, -1.0, 1.0),
    (448, 448, 512, True, 1, -1.0, 1.0),    # lower triangle only, diagonal tiles
    (320, 512, 512, False, 4, 1.0, 0.0),    # contractions from 512 down to 64: two steps
    (512, 320, 512, False, 2, -1.0, 0.0),
    (640, 640, 256, True, 1, -1.0, 1.0),    # from sixteen 128-wide tiles on: one sum
])
def test_sgemm_small_tiles(M, N, Kc, trans_b, flags, alpha, beta):
    """Products of a few 64 x 64 tiles: within the fp32 matrix instruction's error, nothing outside C written."""
    from llmcompressor_amd import ops

    A, B, Bp, C0 = _operands(M, N, Kc, trans_b, flags, seed=M + N + Kc + flags)
    ref = alpha * (A.double() @ Bp.double()) + beta * C0.double()
    bound = A.double().abs() @ Bp.double().abs() + C0.double().abs()
    wide = torch.full((M + 2, N + 8), 7.0, device="cuda")
    C = wide[1:M + 1, 4:N + 4]
    C.copy_(C0)
    ops.sgemm_(C, A, B, alpha=alpha, beta=beta, trans_b=trans_b, flags=flags)
    err = ((C.double() - ref).abs() / bound)
    if flags & 1:
        assert torch.equal(torch.triu(C, 1), torch.triu(C0, 1))
        err = torch.tril(err)
    assert err.max().item() < 8 * 2 ** -24, err.max().item() * 2 ** 24
    C.fill_(7.0)
    assert bool((wide == 7.0).all())

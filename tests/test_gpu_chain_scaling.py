"""GPU: the Cholesky chain works on D H D, D a diagonal of powers of two, and from 3072 columns on takes its updates as
two-term f16 products, whose operands that scaling keeps in range (gptq_quantize.py:144-164 is the chain's definition)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _hessian(K, T, seed, spread=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(T, K, device="cuda", generator=g)
    x *= torch.logspace(-spread, spread, K, device="cuda")[torch.randperm(K, device="cuda", generator=g)]
    H = (x.T @ x) / T
    return (H + H.T) / 2


def _chain(H, form=0, percdamp=0.01):
    from llmcompressor_amd import ops

    U, _, info = ops.gptq_hinv_(H.clone(), None, percdamp=percdamp, form=form)
    return U, int(info.item())


# trailing matrices of one tile and less, of odd numbers of 64-wide tiles, of whole 128-wide ones, with regions cut short by the
# width.  Two-term products from 3072 on: 3136 and 4160 on 64-wide tiles only, the others on 128-wide ones
# too; 512-wide panels from 8320 on, whose second regions take a product of their own, the last one of 128 columns there
@pytest.mark.parametrize("K", [320, 384, 576, 832, 1280, 2304, 3072, 3136, 4160, 8320, 11008])
def test_factor_against_64_bits(K):
    H = _hessian(K, 2 * K, seed=K)
    form = 1 if K >= 8320 else 0  # there the factor itself outside the 512-wide diagonal blocks: no long inverse
    U, info = _chain(H, form)
    assert info == 0
    Hd = H.double().cpu()
    Hd += 0.01 * Hd.diagonal().mean() * torch.eye(K, dtype=torch.float64)
    ref = torch.linalg.cholesky(Hd.flip(0, 1)).flip(0, 1)
    ends = list(range(K, 0, -512)) if form == 1 else [K]
    for end in ends:  # the inverse: of the whole factor, or of its diagonal blocks
        block = slice(max(0, end - 512) if form == 1 else 0, end)
        eye = torch.eye(block.stop - block.start, dtype=torch.float64)
        ref[block, block] = torch.linalg.solve_triangular(ref[block, block].clone(), eye, upper=True)
    ref = ref.cuda()
    # a triangular factor in fp32: columns off by sqrt(K) 2^-24 times a condition number of some tens at these matrices
    err = (U.double() - ref).norm(dim=0) / ref.norm(dim=0)
    assert err.max().item() < K ** 0.5 * 2 ** -24 * 30, err.max().item()


def _common_directions(K):
    """Channels that all read the same 64 directions, most of the quiet ones' energy: the first updates of the factorisation
    take nearly all of the matrix away, and the rounding of their sums is what is left."""
    g = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn(2 * K, K, device="cuda", generator=g)
    x *= torch.logspace(-1, 1, K, device="cuda")[torch.randperm(K, device="cuda", generator=g)]
    x += torch.randn(2 * K, 64, device="cuda", generator=g) @ (torch.randn(64, K, device="cuda", generator=g) * 0.3)
    x = x[:, x.square().sum(0).argsort(descending=True)].contiguous()
    H = torch.zeros(K, K, dtype=torch.float64, device="cuda")
    for part in x.split(2048):
        H += part.double().T @ part.double()
    return (H / (2 * K)).float()


# Bounds: what three-term products give in the same panels of 256 columns (512 from 8192 on).  Measured 6.2e-6, 7.2e-6 and
# 1.47e-5; 8.3e-6, 9.9e-6 and 1.95e-5 with panels twice as wide, whose sums are rounded twice as often.
@pytest.mark.parametrize("K,bound", [(3072, 7.28e-6), (4096, 8.47e-6), (8192, 1.62e-5)])
def test_sums_of_an_update_are_short(K, bound):
    H = _common_directions(K)
    V, info = _chain(H, form=1)
    assert info == 0
    Hd = H.double().cpu()
    Hd += 0.01 * Hd.diagonal().mean() * torch.eye(K, dtype=torch.float64)
    want = torch.linalg.cholesky(Hd.flip(0, 1)).flip(0, 1).cuda()
    block = torch.arange(K, device="cuda").flip(0) // 512  # inside these blocks V holds the inverse
    far = block[:, None] != block[None, :]
    err = ((V.double() - want)[far].norm() / want[far].norm()).item()
    assert err < bound, err


@pytest.mark.parametrize("K,form", [(320, 0), (1000, 0), (1152, 1), (2304, 0), (3072, 0), (3136, 0), (4224, 1)])
@pytest.mark.parametrize("shift", [-60, 24])
def test_powers_of_two_pass_through(K, form, shift):
    """Without damping, scaling row and column c of H by 2^e[c] scales column c of the inverse factor by 2^-e[c] and row c
    of the factor itself by 2^e[c], and changes no other bit."""
    H = _hessian(K, 2 * K, seed=K + 1)
    g = torch.Generator().manual_seed(K)
    e = torch.randint(-8, 9, (K,), generator=g).cuda() + shift // 2
    d = torch.exp2(e.double()).float()
    U, info = _chain(H, form, percdamp=0.0)
    Us, infos = _chain(H * d[:, None] * d[None, :], form, percdamp=0.0)
    assert info == infos == 0
    want = U / d[None, :]
    if form == 1:
        block = torch.arange(K, device="cuda").flip(0) // 512
        want = torch.where(block[:, None] == block[None, :], want, U * d[:, None])
    assert torch.equal(Us, want)


# (row, column): eliminated from the last column on, so the pivot of the lower index fails.  The last ones go through all of
# the chain's products, as infinities in the two-term ones (1e18 against diagonal entries near 1), before their pivot comes
@pytest.mark.parametrize("K,at", [(320, (5, 40)), (1280, (5, 40)), (3072, (5, 40)), (3072, (5, 3000)), (3136, (1500, 3100)),
                                  (4224, (64, 4200))])
@pytest.mark.parametrize("big", [1e4, 1e18])
def test_indefinite_matrix_is_found_at_its_pivot(K, at, big):
    """An off-diagonal entry far above what a positive matrix allows leaves the range of the products, in the row whose
    pivot fails for it; nothing before that pivot may notice."""
    H = _hessian(K, 2 * K, seed=K + 2, spread=0.3)
    H[at[0], at[1]] = H[at[1], at[0]] = big
    U, info = _chain(H)
    assert info == at[0] + 1
    assert torch.equal(U, torch.eye(K, device="cuda"))


def test_forms_of_the_factor():
    from llmcompressor_amd import ops

    assert ops.gptq_quantize_form(1536, 128) == ops.gptq_quantize_form(4096, 128) == ops.FACTOR_GROUPS
    assert ops.gptq_quantize_form(1408, 128) == ops.gptq_quantize_form(1600, 128) == ops.FACTOR_INVERSE
    assert ops.gptq_quantize_form(4096, 64) == ops.FACTOR_INVERSE


# A weight of many rows on few columns takes longer with the factor in groups (14336 x 2048 1.79 ms, 1.66 with the inverse).
# In a lock-step set every member has the factor that it would be given alone: the same bits.  q and k are fed one input.
@torch.no_grad()
@pytest.mark.parametrize("K", [1536, 1664])
def test_tall_weights_keep_the_inverse_factor(K):
    from llmcompressor_amd import ops
    from llmcompressor_amd.modifiers.gptq.gptq_quantize import quantize_weight, quantize_weight_group
    from llmcompressor_amd.modifiers.quantization.calibration import observe

    assert ops.gptq_quantize_form(K, 128, K) == ops.FACTOR_GROUPS
    assert ops.gptq_quantize_form(K, 128, K + 1) == ops.gptq_quantize_form(3968, 128, 1 << 17) == ops.FACTOR_INVERSE
    assert ops.gptq_quantize_form(4096, 128, 1 << 17) == ops.FACTOR_GROUPS
    few, tall = _linears(K, 192, 3)[0], _linears(K, K + 8, 2)[0]
    mods = [few[0], tall[0], few[1], tall[1], few[2]]
    Hs = [_hessian(K, 2 * K, seed) for seed in range(3)]
    Hs = [Hs[0], Hs[1], Hs[0], Hs[1], Hs[2]]
    calls, raw, raw_s = [], ops.gptq_hinv_grouped, ops.gptq_hinv_
    ops.gptq_hinv_grouped = lambda h, *a, **kw: (calls.append((len(h), kw["form"], kw["n_inverse"])), raw(h, *a, **kw))[1]
    ops.gptq_hinv_ = lambda h, *a, **kw: (calls.append(kw["form"]), raw_s(h, *a, **kw))[1]
    try:
        observe(mods, "weight")
        got = quantize_weight_group(mods, Hs, [2.0] * 5)
        observe(mods, "weight")
        alone = [quantize_weight(m, m.quantization_scheme.weights, H.clone(), hessian_divisor=2.0) for m, H in zip(mods, Hs)]
    finally:
        ops.gptq_hinv_grouped, ops.gptq_hinv_ = raw, raw_s
    assert calls[0] == (3, ops.FACTOR_GROUPS, 1)
    assert calls[1:] == [ops.FACTOR_GROUPS, ops.FACTOR_INVERSE] * 2 + [ops.FACTOR_GROUPS]
    for (loss, q, info), (want_loss, want) in zip(got, alone):
        assert int(info) == 0 and abs(loss.item() - want_loss) <= 1e-6 * want_loss
        assert q.keys() == want.keys() and all(torch.equal(q[k], want[k]) for k in want)


# rows of one 64-wide tile and of several, with padding; widths with a short first group and with a last piece shorter than
# the others
@pytest.mark.parametrize("R,K", [(64, 1536), (100, 1664), (129, 2432), (700, 3584)])
@pytest.mark.parametrize("spread", [0.5, 2.0])
def test_column_loop_on_two_term_products(R, K, spread):
    """The loop whose far updates are two-term products (FACTOR_GROUPS) against the one with three-term products and the
    inverse factor: as many of the weights as an fp64 run of either would give.  Channel scales over four decades, weights
    whose rows differ by as much, and activations whose Hessian is far from 1."""
    from llmcompressor_amd import ops

    H = _hessian(K, 3 * K, seed=R + K, spread=spread) * 2.0 ** 30
    g = torch.Generator(device="cuda").manual_seed(R)
    w = torch.randn(R, K, device="cuda", generator=g) * torch.logspace(-3, 1, R, device="cuda")[:, None]
    scale = (w.abs().amax(1, keepdim=True) / 7.5).expand(R, K // 128).contiguous().bfloat16()
    w = w.bfloat16()
    g_idx = torch.arange(K, dtype=torch.int32, device="cuda") // 128
    out = []
    for form in (ops.FACTOR_INVERSE, ops.FACTOR_GROUPS):
        U, info = _chain(H, form)
        assert info == 0
        q, _ = ops.gptq_quantize(w, U, scale, None, ops.FMT_INT, 4, 1, K // 128, g_idx=g_idx, form=form)
        out.append(q)
    agree = (out[0] == out[1]).float().mean().item()
    assert agree >= 0.998, agree  # each within 99.9 % of the exact loop's
    errs = [((w - q).float() @ H / H.diagonal().mean() * (w - q).float()).sum(1) for q in out]
    assert torch.allclose(errs[0], errs[1], rtol=0.02)


def _exact_loop(W, H, scale, percdamp):
    """int4 codes of 128-column groups by the column loop in 64 bits, from the 64-bit factor of H."""
    K = H.shape[0]
    Hd = H.double().cpu() + percdamp * H.diagonal().double().mean().cpu() * torch.eye(K, dtype=torch.float64)
    V = torch.linalg.cholesky(Hd.flip(0, 1)).flip(0, 1)
    U = torch.linalg.solve_triangular(V, torch.eye(K, dtype=torch.float64), upper=True).cuda()
    W, codes = W.double().clone(), torch.empty(W.shape, device=W.device)
    for j in range(K):
        s = scale[:, j // 128].double()
        codes[:, j] = torch.round(W[:, j] / s).clamp(-8, 7)
        W[:, j + 1:] -= ((W[:, j] - codes[:, j] * s) / U[j, j])[:, None] * U[j, j + 1:]
    return codes


def _two_sets(K, T, seed, other):
    """Activations of which the channels `other` never fire together with the rest."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(T, K, device="cuda", generator=g)
    x *= torch.logspace(-0.5, 0.5, K, device="cuda")[torch.randperm(K, device="cuda", generator=g)]
    x[:T // 4, ~other] = 0
    x[T // 4:, other] = 0
    return x


def _loop_agreement(x, percdamp, form, seed):
    """Share of the int4 codes of a column loop on x^T x that are those of 64 bits."""
    from llmcompressor_amd import ops

    K, R = x.shape[1], 256
    H = (x.double().T @ x.double()).float()
    H = (H + H.T) / 2
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randn(R, K, device="cuda", generator=g) * 0.02
    scale = w.view(R, K // 128, 128).abs().amax(-1) / 7.5
    U, info = _chain(H, form, percdamp)
    assert info == 0
    q, _ = ops.gptq_quantize(w, U, scale, None, ops.FMT_INT, 4, 1, K // 128, form=form,
                             g_idx=torch.arange(K, dtype=torch.int32, device="cuda") // 128)
    codes = torch.round(q / scale.repeat_interleave(128, 1))
    return (codes == _exact_loop(w, H, scale, percdamp)).float().mean().item()


@pytest.mark.parametrize("channels", [1, 8])
@pytest.mark.parametrize("exponent", [0, -15, -20, -40])
def test_rows_of_the_factor_without_later_columns(channels, exponent):
    """Channels of the first group that fire only by themselves: their rows of the factor are zero beyond the diagonal
    block, and what the loop keeps of their weights must not push the other columns out of the products' range, however
    small the Hessian is."""
    from llmcompressor_amd import ops

    K = 1536
    other = torch.zeros(K, dtype=torch.bool, device="cuda")
    other[torch.arange(channels, device="cuda") * 37] = True
    x = _two_sets(K, 3 * K, 5 + channels, other) * 2.0 ** exponent
    assert _loop_agreement(x, 0.01, ops.FACTOR_GROUPS, seed=2) >= 0.999


@pytest.mark.parametrize("percdamp", [0.01, 1e-6])
@pytest.mark.parametrize("louder", [4, 8, 14])
def test_loud_channels_that_fire_apart(louder, percdamp):
    """Half of the channels 2^louder times as loud as the others, which never fire together with them: the row scales follow
    the loud ones, and the sums of the others, which they add nothing to, keep their codes.  (An element 2^-14 below a row's
    largest loses bits below 2^-38 of that, and the damping keeps what a column is divided by above percdamp^(1/2) of the
    loudest channels' norm: 2^-38 K^(1/2) / percdamp^(1/2) of a quantisation step at most.)"""
    from llmcompressor_amd import ops

    K = 1536
    other = torch.rand(K, generator=torch.Generator().manual_seed(louder)).cuda() < 0.5
    x = _two_sets(K, 3 * K, louder, other)
    x[:, other] *= 2.0 ** louder
    groups, inverse = (_loop_agreement(x, percdamp, form, seed=3) for form in (ops.FACTOR_GROUPS, ops.FACTOR_INVERSE))
    assert groups >= 0.999 and groups >= inverse - 0.0005, (groups, inverse)


@pytest.mark.parametrize("K", [1, 3, 64, 65, 1023, 1025, 16384])
def test_diagonal_order_at_the_edges_of_its_workgroups(K):
    from llmcompressor_amd import ops

    g = torch.Generator(device="cuda").manual_seed(K)
    Hs = [torch.randint(-3, 4, (K, K), device="cuda", generator=g).float() for _ in range(3)]  # many equal entries
    Hs[1].fill_(float("-inf"))
    got = ops.diag_argsort_desc(Hs)
    for row, H in zip(got, Hs):
        assert torch.equal(row, torch.argsort(H.diagonal(), descending=True, stable=True))


# either side of 72000 entries, from where on they are sorted and not counted; more problems than one launch takes
@pytest.mark.parametrize("n,K", [(71, 1000), (72, 1000), (70, 1024), (71, 1024), (128, 2048), (256, 513), (300, 100), (600, 352)])
def test_diagonal_order_of_many_problems(n, K):
    from llmcompressor_amd import ops

    g = torch.Generator(device="cuda").manual_seed(n)
    diagonals = torch.randint(-50, 51, (n, K), device="cuda", generator=g).float()
    space = torch.zeros(n, K, K, device="cuda")
    space.diagonal(dim1=1, dim2=2).copy_(diagonals)
    got = ops.diag_argsort_desc(list(space))
    assert torch.equal(got, torch.argsort(diagonals, dim=1, descending=True, stable=True))


def _linears(K, rows, count, seed=0):
    """(modules, their Hessians): W4A16 in groups of 128 columns, static activation order."""
    from llmcompressor_amd.modifiers.quantization.calibration import initialize_observer
    from llmcompressor_amd.quantization import initialize_module_for_quantization, preset_name_to_scheme

    g = torch.Generator(device="cuda").manual_seed(seed)
    mods = []
    for i in range(count):
        m = torch.nn.Linear(K, rows, bias=False, dtype=torch.bfloat16, device="cuda")
        m.weight.data = (torch.randn(rows, K, device="cuda", generator=g) * 0.02).bfloat16()
        initialize_module_for_quantization(m, preset_name_to_scheme("W4A16", ["Linear"]))
        initialize_observer(m, "weight")
        mods.append(m)
    return mods, [_hessian(K, 2 * K, seed + 10 + i) for i in range(count)]


@torch.no_grad()
@pytest.mark.parametrize("K", [1024, 1536])
def test_weight_group_finished_in_another_block_size(K):
    """The halves of ``quantize_weight_group`` take block sizes of their own: the block size only regroups fp32 sums, whatever
    form of the factor the first half has asked for (below 8192 columns, where that depends on it)."""
    from llmcompressor_amd.modifiers.gptq.gptq_quantize import (begin_weight_group, finish_weight_group,
                                                                quantize_weight_group)
    from llmcompressor_amd.modifiers.quantization.calibration import observe

    mods, Hs = _linears(K, 256, 3)
    divisors = [1.0] * len(mods)
    observe(mods, "weight")
    want = quantize_weight_group(mods, Hs, divisors)
    for first, second in ((128, 64), (64, 128)):
        observe(mods, "weight")
        got = finish_weight_group(begin_weight_group(mods, Hs, divisors, blocksize=first), second)
        agree = torch.stack([(a[1]["weight"] == b[1]["weight"]).float().mean() for a, b in zip(got, want)])
        assert agree.min().item() >= 0.999, (first, second, agree)


@torch.no_grad()
@pytest.mark.parametrize("K,rows", [(1536, 200), (1024, 256)])
def test_loops_of_a_group_in_runs_give_the_same_bits(K, rows):
    from llmcompressor_amd import ops
    from llmcompressor_amd.modifiers.gptq.gptq_quantize import quantize_weight_group
    from llmcompressor_amd.modifiers.quantization.calibration import observe

    mods, Hs = _linears(K, rows, 5)
    bytes_of = lambda n: ops.gptq_quantize_grouped_workspace_bytes(n, rows, K, ops.gptq_quantize_form(K, 128, rows))  # noqa: E731
    factors = 5 * 4 * K * K
    sizes, results, raw, raw_s = [], [], ops.gptq_quantize_grouped, ops.gptq_quantize
    ops.gptq_quantize_grouped = lambda w, *a, **kw: (sizes.append(len(w)), raw(w, *a, **kw))[1]
    ops.gptq_quantize = lambda w, *a, **kw: (sizes.append(1), raw_s(w, *a, **kw))[1]
    try:
        for room in (5, 2, 0):
            observe(mods, "weight")
            results.append(quantize_weight_group(mods, Hs, [1.0] * 5, max_bytes=factors + room * bytes_of(1)))
    finally:
        ops.gptq_quantize_grouped, ops.gptq_quantize = raw, raw_s
    assert sizes == [5] + [1, 2, 2] + [1] * 5
    for got in results[1:]:
        for a, b in zip(got, results[0]):
            assert torch.equal(a[0], b[0]) and all(torch.equal(a[1][k], b[1][k]) for k in b[1])

"""GPU: the quantiser's group kernel takes in what a group owes to earlier columns by itself and leaves D = W - Q behind
(csrc/gptq_group.h), here against the loop on the inverse factor (gptq_quantize.py:180-260 is the loop's definition)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# 16 and 32 rows to a workgroup (up to 4096 rows, and more), the last one partly filled; zero points, which share the LDS
# with P; a short first group; one piece of P, several and (few rows, wide) as many as there can be; one problem and several
@pytest.mark.parametrize("R,K,sym,n", [(1, 1024, True, 1), (17, 1152, False, 1), (40, 9216, True, 1), (4097, 1536, False, 1),
                                       (4120, 1664, True, 1), (300, 2048, False, 3), (1500, 1536, False, 3)])
def test_groups_against_the_inverse_factor(R, K, sym, n):
    from llmcompressor_amd import ops

    whole = -(-R // 32) * 32  # the last workgroup filled up with other rows; R and this have the same padding and pieces
    g = torch.Generator(device="cuda").manual_seed(R + K)
    Hs, ws, scales, zps = [], [], [], []
    for _ in range(n):
        x = torch.randn(3 * K, K, device="cuda", generator=g) * torch.logspace(-0.5, 0.5, K, device="cuda").flip(0)
        Hs.append((x.T @ x) / (3 * K))
        w = (torch.randn(whole, K, device="cuda", generator=g) * 0.02).bfloat16()
        blocks = w.float().view(whole, K // 128, 128)
        if sym:
            scales.append((blocks.abs().amax(-1) / 7.5).bfloat16())
            zps.append(None)
        else:
            low, high = blocks.amin(-1), blocks.amax(-1)
            scales.append(((high - low) / 15).bfloat16())
            zps.append((-8 - low / scales[-1].float()).round().clamp(-8, 7).to(torch.int8))
        ws.append(w)
    gi = torch.arange(K, dtype=torch.int32, device="cuda") // 128

    def quantize(form, first, last):
        """The column loop on rows [first, last) of every weight -> codes' values, losses."""
        w, s, z = ([None if t is None else t[first:last].contiguous() for t in ts] for ts in (ws, scales, zps))
        if n == 1:
            q, loss = ops.gptq_quantize(w[0], U[0], s[0], z[0], ops.FMT_INT, 4, 1, K // 128, g_idx=gi, dead=dead[0], form=form)
            return [q], loss
        return ops.gptq_quantize_grouped(w, U, s, None if sym else z, ops.FMT_INT, 4, 1, K // 128, g_idxs=[gi] * n, dead=dead,
                                         form=form)

    U, dead, info = ops.gptq_hinv_grouped(Hs, None, [1.0] * n, form=ops.FACTOR_INVERSE)
    assert not info.any()
    # a row's loss is a sum of squared rounding errors, uniform ones, over the squared diagonal of U
    weight = U.diagonal(dim1=1, dim2=2).double().pow(-2)
    a, la = quantize(ops.FACTOR_INVERSE, 0, R)
    U, dead, info = ops.gptq_hinv_grouped(Hs, None, [1.0] * n, form=ops.FACTOR_GROUPS)
    assert not info.any()
    b, lb = quantize(ops.FACTOR_GROUPS, 0, R)
    assert torch.allclose(la, lb, rtol=2e-3)
    # each form's codes are those of a 64-bit loop up to a share of 0.1 %, which is less than one row here: a row that
    # meets a rounding boundary differs in about a third of what follows
    for x, y in zip(a, b):
        differ = x != y
        assert differ.float().mean().item() <= 2e-3 or differ.any(1).sum().item() <= 1
    # and every row's error is that of a row quantised well, also where the codes took another path: a mean of squares of uniform
    # errors varies by sqrt(4 / 5 / (their effective number)), the difference of two by sqrt(2) that; 6 times it
    for x, y, w, H, v in zip(a, b, ws, Hs, weight):
        ex, ey = (((w[:R].double() - q.double()) @ H.double() * (w[:R].double() - q.double())).sum(1) for q in (x, y))
        spread = (1.6 * v.square().sum().item()) ** 0.5 / v.sum().item()
        assert ((ey / ex - 1).abs().max().item()) <= 6 * spread
    # a row does not depend on its neighbours: the same bits as in a workgroup without empty rows, and its share of the loss
    full, lfull = quantize(ops.FACTOR_GROUPS, 0, whole)
    for x, y in zip(b, full):
        assert torch.equal(x, y[:R])
    if whole > R:
        _, rest = quantize(ops.FACTOR_GROUPS, R, whole)
        assert (((lfull - lb - rest) / lfull).abs() * whole).max().item() <= 0.5

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

    g = torch.Generator(device="cuda").manual_seed(R + K)
    Hs, ws, scales, zps = [], [], [], []
    for _ in range(n):
        x = torch.randn(3 * K, K, device="cuda", generator=g) * torch.logspace(-0.5, 0.5, K, device="cuda").flip(0)
        Hs.append((x.T @ x) / (3 * K))
        w = (torch.randn(R, K, device="cuda", generator=g) * 0.02).bfloat16()
        blocks = w.float().view(R, K // 128, 128)
        if sym:
            scales.append((blocks.abs().amax(-1) / 7.5).bfloat16())
            zps.append(None)
        else:
            low, high = blocks.amin(-1), blocks.amax(-1)
            scales.append(((high - low) / 15).bfloat16())
            zps.append((-8 - low / scales[-1].float()).round().clamp(-8, 7).to(torch.int8))
        ws.append(w)
    gi = torch.arange(K, dtype=torch.int32, device="cuda") // 128
    out = {}
    for form in (ops.FACTOR_INVERSE, ops.FACTOR_GROUPS):
        U, dead, info = ops.gptq_hinv_grouped(Hs, None, [1.0] * n, form=form)
        assert not info.any()
        if n == 1:
            q, loss = ops.gptq_quantize(ws[0], U[0], scales[0], zps[0], ops.FMT_INT, 4, 1, K // 128, g_idx=gi, dead=dead[0],
                                        form=form)
            out[form] = [q], loss
        else:
            out[form] = ops.gptq_quantize_grouped(ws, U, scales, None if sym else zps, ops.FMT_INT, 4, 1, K // 128,
                                                  g_idxs=[gi] * n, dead=dead, form=form)
    (a, la), (b, lb) = out.values()
    assert torch.allclose(la, lb, rtol=2e-3)
    # each form's codes are those of a 64-bit loop up to a share of 0.1 %, which is less than one row here: a row that
    # meets a rounding boundary differs in about a third of what follows
    for x, y in zip(a, b):
        differ = x != y
        assert differ.float().mean().item() <= 2e-3 or differ.any(1).sum().item() <= 1

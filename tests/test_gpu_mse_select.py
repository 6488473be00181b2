"""The MSE search's last kernel: a thread picks the ranges of one group or of four, from one word of improvements per group (up to
64 steps) or four; against the eager search of the oracle (mse_quant.py:19-141)."""
import pytest
import torch

from oracle import observers as O
from oracle import qformat as F

pytestmark = pytest.mark.gpu


# one group, a thread's worth of a workgroup and one more, a whole workgroup and one more; 20 steps, 64, 65 and 80 (the
# search's words), a patience that ends it early, at the last step of a word and never
@pytest.mark.parametrize("groups", [1, 255, 257, 1024, 1025])
@pytest.mark.parametrize("kw", [{}, dict(maxshrink=0.64, patience=62), dict(maxshrink=0.65, patience=63),
                                dict(maxshrink=0.8, patience=7), dict(maxshrink=0.8, patience=1000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_ranges_are_the_oracles(groups, kw, dtype):
    from llmcompressor_amd import ops

    gen = torch.Generator().manual_seed(groups)
    w = (torch.randn(groups, 16, generator=gen) * 0.02).to(dtype)
    w[0] = 0.0  # improves once and never again
    args = F.QArgs(num_bits=4, strategy="group", group_size=16)
    want = O.grid_search_mse(O.flatten_for_calibration(w, "weight", args), args, **kw)
    got = ops.mse_observe_groups(w.cuda(), 16, ops.FMT_INT, 4, True, ops.SCALE_PLAIN, **kw)
    for g, e in zip(got, want):
        assert torch.equal(g.cpu().reshape(e.shape), e)


# a thread takes four groups from 2^19 of them on: the same groups 512 times over have the same ranges, whatever they are cut into
@pytest.mark.parametrize("groups,times", [(1025, 512), (1023, 513), (4096, 129)])
@pytest.mark.parametrize("kw", [{}, dict(maxshrink=0.64, patience=62), dict(maxshrink=0.8, patience=7),
                                dict(maxshrink=0.8, patience=1000)])
def test_many_groups_are_few_groups_repeated(groups, times, kw):
    from llmcompressor_amd import ops

    gen = torch.Generator().manual_seed(groups)
    w = (torch.randn(groups, 16, generator=gen) * 0.02).bfloat16().cuda()
    few = ops.mse_observe_groups(w, 16, ops.FMT_INT, 4, True, ops.SCALE_PLAIN, **kw)
    many = ops.mse_observe_groups(w.repeat(times, 1), 16, ops.FMT_INT, 4, True, ops.SCALE_PLAIN, **kw)
    for f, m in zip(few, many):
        assert torch.equal(m.reshape(times, -1), f.reshape(1, -1).expand(times, -1))

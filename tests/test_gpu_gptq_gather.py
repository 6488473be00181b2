"""The gather of permuted columns in front of the column loop, several rows at a time: the results are those of weights that
were gathered before the call, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(R, K, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    W = torch.randn(R, K, device="cuda", generator=g).to(dtype)
    U = torch.triu(torch.randn(K, K, device="cuda", generator=g) * (0.3 / K ** 0.5), 1) + torch.eye(K, device="cuda")
    scale = torch.full((R, 1), 0.25, device="cuda", dtype=dtype)
    perm = torch.randperm(K, device="cuda", generator=g).to(torch.int32)
    dead = (torch.rand(K, device="cuda", generator=g) < 0.1).to(torch.uint8)
    return W, U, scale, perm, dead


# rows that fill no set of four or two; columns that are no multiple of four; a thread's worth, and where the threads, the rows
# at a time (8192) and the form (16384) change; weights at an odd element and with an odd stride
@pytest.mark.parametrize("R,K,dtype,at", [
    (1, 8, torch.bfloat16, 0), (3, 132, torch.bfloat16, 0), (5, 130, torch.bfloat16, 0), (6, 2048, torch.float16, 0),
    (7, 2052, torch.bfloat16, 0), (4, 4100, torch.bfloat16, 0), (5, 8192, torch.bfloat16, 0), (3, 8196, torch.float16, 0),
    (6, 256, torch.bfloat16, 1), (6, 256, torch.bfloat16, 2), (6, 256, torch.float32, 0), (9, 1024, torch.bfloat16, 0)])
def test_gathered_in_the_call_is_gathered_before_it(R, K, dtype, at):
    from llmcompressor_amd import ops

    W, U, scale, perm, dead = _case(R, K, dtype, R * K)
    wide = torch.empty(R, K + 2 * at, device="cuda", dtype=dtype)
    view = wide[:, at : at + K]
    view.copy_(W)
    for d in (None, dead):
        kw = dict(dead=d, form=0)
        q, loss = ops.gptq_quantize(view if at else W, U, scale, None, ops.FMT_INT, 4, 1, 1, perm=perm, **kw)
        want, wloss = ops.gptq_quantize(W[:, perm.long()].contiguous(), U, scale, None, ops.FMT_INT, 4, 1, 1, **kw)
        assert torch.equal(q[:, perm.long()], want) and torch.equal(loss, wloss)


@pytest.mark.parametrize("R,K", [(6, 512), (5, 514), (3, 8448)])
def test_of_several_problems(R, K):
    from llmcompressor_amd import ops

    cases = [_case(R, K, torch.bfloat16, 10 * R + b) for b in range(3)]
    Ws, Us, scales, perms, deads = zip(*cases)
    U, perm, dead = torch.stack(Us), torch.stack(perms), torch.stack(deads)
    q, loss = ops.gptq_quantize_grouped(list(Ws), U, list(scales), None, ops.FMT_INT, 4, 1, 1, perms=perm, dead=dead, form=0)
    for b in range(3):
        want, wloss = ops.gptq_quantize(Ws[b][:, perms[b].long()].contiguous(), Us[b], scales[b], None, ops.FMT_INT, 4, 1, 1,
                                        dead=deads[b], form=0)
        assert torch.equal(q[b][:, perms[b].long()], want), b
        torch.testing.assert_close(loss[b : b + 1], wloss, rtol=1e-6, atol=0)  # (its rows may be added in another order)

"""GPU: a region of the Cholesky chain is one launch whose workgroups hand blocks to each other (csrc/chol_region.h); the
chain's definition is gptq_quantize.py:144-164."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _hessian(K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(2 * K, K, device="cuda", generator=g) * torch.logspace(-1, 1, K, device="cuda")
    return (x.T @ x) / (2 * K)


def _factor(H, percdamp=0.01):
    Hd = H.double().cpu()
    Hd += percdamp * Hd.diagonal().mean() * torch.eye(len(Hd), dtype=torch.float64)
    R = torch.linalg.cholesky(Hd.flip(0, 1)).flip(0, 1)
    return torch.linalg.solve_triangular(R, torch.eye(len(Hd), dtype=torch.float64), upper=True).cuda()


# one to four blocks in the last region, with none, one and several sets of rows below the first one, padded widths among them
@pytest.mark.parametrize("K", [1, 63, 64, 100, 128, 192, 256, 257, 320, 400, 512, 704, 1088])
def test_regions_against_64_bits(K):
    from llmcompressor_amd import ops

    H = _hessian(K, K)
    U, _, info = ops.gptq_hinv_(H.clone())
    assert int(info) == 0
    want = _factor(H)
    # columns off by sqrt(K) 2^-24 times a condition number of some tens, as for every width of the chain
    err = (U.double() - want).norm(dim=0) / want.norm(dim=0)
    assert err.max().item() < max(K, 64) ** 0.5 * 2 ** -24 * 30, err.max().item()


# more tasks than the chip holds at a time: 300 x (3 + 6) and 700 x 1, two workgroups to a CU
@pytest.mark.parametrize("K,n", [(448, 300), (128, 700), (1024, 65)])
def test_more_tasks_than_the_chip_holds(K, n):
    from llmcompressor_amd import ops

    Hs = [_hessian(K, b) for b in range(5)]
    U, _, info = ops.gptq_hinv_grouped([Hs[b % 5] for b in range(n)])
    assert not info.any()
    single = [ops.gptq_hinv_(H.clone())[0] for H in Hs]
    for b in range(n):
        assert torch.equal(U[b], single[b % 5]), b


def test_chains_beside_each_other_and_beside_other_work():
    """Four streams' chains at once, while products fill the chip: every wait ends and the bits are those of a call alone."""
    from llmcompressor_amd import ops

    sizes = [2048, 1536, 1024, 2304]
    Hs = [_hessian(K, K) for K in sizes]
    want = [ops.gptq_hinv_(H.clone())[0] for H in Hs]
    busy = torch.randn(8192, 8192, device="cuda", dtype=torch.bfloat16)
    streams = [torch.cuda.Stream() for _ in range(5)]
    torch.cuda.synchronize()
    got = [[] for _ in sizes]
    for _ in range(4):
        with torch.cuda.stream(streams[4]):
            torch.mm(busy, busy)
        for i, H in enumerate(Hs):
            with torch.cuda.stream(streams[i]):
                got[i].append(ops.gptq_hinv_(H.clone()))
    torch.cuda.synchronize()
    for i in range(len(sizes)):
        for U, _, info in got[i]:
            assert int(info) == 0 and torch.equal(U, want[i]), sizes[i]


def test_replayed_from_a_graph():
    from llmcompressor_amd import ops

    K = 768
    H, other = _hessian(K, 1), _hessian(K, 2)
    static = H.clone()
    ops.gptq_hinv_(static.clone())  # the workspace exists
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        U = static.clone()
        _, _, info = ops.gptq_hinv_(U)
    for src in (H, other, H, other):
        static.copy_(src)
        graph.replay()
        torch.cuda.synchronize()
        want = ops.gptq_hinv_(src.clone())[0]
        torch.cuda.synchronize()
        assert int(info) == 0 and torch.equal(U, want)


# one region, whose row blocks wait; one with rows below it; regions after the one that gives up
@pytest.mark.parametrize("K", [320, 256, 1088])
def test_waits_that_give_up_end_the_call(K):
    """With no time to wait every task leaves, the result is the identity and info -1; the next call is as ever."""
    from llmcompressor_amd import ops

    H = _hessian(K, K)
    want = ops.gptq_hinv_(H.clone())[0]
    U, _, info = ops.gptq_hinv_(H.clone(), wait_us=0)
    assert int(info) == -1 and torch.equal(U, torch.eye(K, device="cuda"))
    with pytest.raises(RuntimeError, match="gave up waiting"):
        ops.factorisation_failed(int(info))
    again, _, info = ops.gptq_hinv_(H.clone())
    assert int(info) == 0 and torch.equal(again, want)

"""The tile kernel for linear layers of some hundred rows (csrc/kernels/tile_linear.hip) against an fp64 product of the same bf16
operands, and the rule that sends a call to it.

Bound of every output: it is rounded to bf16 once, 2^-8 of itself, and the fp32 sum of its K products errs by about sqrt(K) 2^-24 of the
norms of its two rows; four times that.
"""
import pytest
import torch

from symmetry_amd import ops
from symmetry_amd.models.transformer import Workspace


def within(out, x, w):
    y = x.double() @ w.double().t()
    sums = 4 * x.shape[1] ** 0.5 * 2.0 ** -24 * x.double().norm(dim=1)[:, None] * w.double().norm(dim=1)[None]
    return bool(((out.double() - y).abs() <= 2.0 ** -8 * y.abs() + sums).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 63, 64, 65, 128, 129, 257, 700])
@pytest.mark.parametrize("N,K", [(4, 512), (130, 576), (1024, 1088), (1000, 3072)])
def test_tile_linear(gpu, M, N, K):
    """Tiles at their ends; outputs that fill no tile; as many stages as the ring has and more; one slice of K, several, a last one that
    is shorter; column ranges of wider matrices, 16-byte stores and single ones."""
    print("tile_linear", M, N, K, flush=True)
    g = torch.Generator(device=gpu).manual_seed(N + K + M)
    slab, counters = ops.mid_workspace(Workspace(), torch.device(gpu))
    x = torch.randn(M, K + 24, device=gpu, generator=g).bfloat16()[:, 8:8 + K]
    w = (torch.randn(N, K, device=gpu, generator=g) * K ** -0.5).bfloat16()
    H, tried = ops._hyb(), 0
    for rows in (64, 128):
        tiles = -(-M // rows) * -(-N // 128)
        for splits in (1, 2, 3, 4):
            for more in (8, 9):
                room = torch.full((M + 1, N + more), 7.0, device=gpu, dtype=torch.bfloat16)
                out = room[:M, :N]
                if not H.tile_linear(x, w, out, rows, splits, slab, counters):
                    per = (K // 64 + splits - 1) // splits
                    assert tiles * splits > 256 or K // 64 - (splits - 1) * per < (6 if rows == 64 else 5)
                    assert bool((room == 7).all())
                    continue
                tried += 1
                assert within(out, x, w), (rows, splits, more)
                assert bool((room[:, N:] == 7).all()) and bool((room[M] == 7).all())
    assert tried >= 4 and not bool(counters.any())


@pytest.mark.gpu
def test_a_model_gets_it(gpu):
    """ops.linear sends rows past the medium range to it with and without a workspace, in the order of its rule, and leaves to the
    library what it does not take; slices of K replay in a graph, with eager calls of other sizes in between."""
    g = torch.Generator(device=gpu).manual_seed(1)
    ws = Workspace()
    x = torch.randn(600, 8192, device=gpu, generator=g).bfloat16()
    w = (torch.randn(2048, 8192, device=gpu, generator=g) * 0.01).bfloat16()
    out, other = torch.empty(600, 2048, device=gpu, dtype=torch.bfloat16), torch.empty(300, 1024, device=gpu, dtype=torch.bfloat16)
    assert not ops.tile_linear(x, w, out) and ops.tile_linear(x, w, out, ws)
    w2 = w[:1024, :2048].contiguous()
    assert not ops.tile_linear(x[:300, :2048], w2, other) and ops.tile_linear(x[:300, :2048], w2, other, ws)
    assert ops.tile_linear(x[:, :2048], w[:, :2048].contiguous(), out)
    assert not ops.tile_linear(x[:256, :2048], w2, other[:256]) and not ops.tile_linear(x[:300, 1:2049], w2, other)
    assert not ops.tile_linear(x[:300, :2048].float(), w2.float(), other.float())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.linear(x, w, out, ws)
    for _ in range(3):
        x.normal_(generator=g)
        graph.replay()
        got = out.clone()
        ops.linear(x[:300, :2048], w2, other, ws)
        assert within(got, x, w) and within(other, x[:300, :2048], w2)


def test_the_rule():
    """The lines' two sides; what is taken is one round of tiles, with stages enough for the ring in every slice."""
    plan = ops.tile_plan
    assert plan(256, 2048, 2048, True) is None and plan(257, 2048, 2048, False) is None and plan(257, 2048, 2048, True) == (64, 2)
    assert plan(512, 2048, 2048, False) is None and plan(512, 2048, 2048, True) == plan(513, 2048, 2048, False) == (64, 1)
    assert plan(1024, 2048, 2048, False) == (64, 1) and plan(1025, 2048, 2048, False) == plan(2048, 2048, 2048, True) == (128, 1)
    assert plan(2049, 2048, 2048, True) is None and plan(900, 2048, 2560, True) is None and plan(600, 16, 2048, True) is None
    assert plan(512, 2048, 4096, True) == (64, 2) and plan(512, 2048, 4096, False) is None and plan(513, 2048, 4096, True) is None
    assert plan(600, 2048, 8192, True) == (128, 2) and plan(600, 2048, 8192, False) is None
    assert plan(300, 2048, 8192, True) == (128, 4) and plan(1100, 2048, 8192, True) is None
    for M in range(257, 2100, 61):
        for N in (512, 1000, 2048, 3072, 6144, 17440):
            for K in (1024, 1536, 2048, 2560, 3072, 4096, 5120, 6144, 8192, 14336):
                for split in (False, True):
                    form = plan(M, N, K, split)
                    if form is not None:
                        rows, S = form
                        per = -(-(K // 64) // S)
                        assert -(-M // rows) * -(-N // 128) * S <= 256 and K // 64 - (S - 1) * per >= (6 if rows == 64 else 5)
                        assert split or S == 1

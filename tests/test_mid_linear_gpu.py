"""The medium-row linear kernel (csrc/kernels/mid_linear.hip) against an fp64 product of the same bf16 operands, and the rule
that sends a call to it.

Bounds: fp32 accumulation of K terms errs by at most about sqrt(K) 2^-24 of the terms' norm, far below the rounding of a bf16
result, 2^-8 of itself: 2^-7 of the largest.  Of a gated pair gate, up and product are rounded, 2^-8 each; the gate's error
reaches silu(y) times 1 + y (1 - sigmoid(y)), at most 1.28 for y > 0: 3.28 x 2^-8, under 2^-6 of the largest result.
"""
import pytest
import torch

from symmetry_amd import ops
from symmetry_amd.models.transformer import Workspace

ROWS = [17, 32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 256]


@pytest.mark.gpu
@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("N,K", [(4, 64), (60, 128), (64, 192), (260, 576), (1000, 1024), (2048, 2048), (5000, 512), (16300, 320)])
def test_mid_linear(gpu, M, N, K):
    """Tiles of rows at their ends; outputs that fill no workgroup; one slice of K, several, a last one that is shorter; fewer chunks
    than the ring has slots and more; column ranges of wider matrices."""
    g = torch.Generator(device=gpu).manual_seed(N + K + M)
    ws = Workspace()
    x = torch.randn(M, K + 24, device=gpu, generator=g).bfloat16()[:, 8:8 + K]
    w = (torch.randn(2 * N, K, device=gpu, generator=g) * K ** -0.5).bfloat16()
    y, u = x.double() @ w[:N].double().t(), x.double() @ w[N:].double().t()
    room = torch.full((M + 1, N + 8), 7.0, device=gpu, dtype=torch.bfloat16)
    out = room[:M, :N]
    for _ in range(2):                                     # (the counters are left at zero)
        assert ops.mid_linear(x, w[:N], out, ws)
        assert float((out.double() - y).abs().max()) <= 2 ** -7 * float(y.abs().max())
        out.fill_(3.0)
        assert ops.mid_linear(x, w, out, ws, glu=True)
        p = y * torch.sigmoid(y) * u
        assert float((out.double() - p).abs().max()) <= 2 ** -6 * max(float(p.abs().max()), 1.0)
    assert bool((room[:, N:] == 7).all()) and bool((room[M] == 7).all())
    assert not bool(ops.mid_workspace(ws, x.device)[1].any())


@pytest.mark.gpu
def test_a_graph_replays(gpu):
    """Slices of K in a captured graph, eager calls of other shapes between its replays: counters and parts are everyone's."""
    g = torch.Generator(device=gpu).manual_seed(1)
    ws = Workspace()
    x = torch.randn(40, 8192, device=gpu, generator=g).bfloat16()
    w = (torch.randn(2048, 8192, device=gpu, generator=g) * 0.01).bfloat16()
    out, other = torch.empty(40, 2048, device=gpu, dtype=torch.bfloat16), torch.empty(20, 2048, device=gpu, dtype=torch.bfloat16)
    assert ops.mid_rows(x, w, out, ws)
    ops.linear(x, w, out, ws)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.linear(x, w, out, ws)
    for i in range(3):
        x.normal_(generator=g)
        graph.replay()
        got = out.clone()
        ops.linear(x[:20], w, other, ws)
        y = x.double() @ w.double().t()
        assert float((got.double() - y).abs().max()) <= 2 ** -7 * float(y.abs().max())
        assert float((other.double() - y[:20]).abs().max()) <= 2 ** -7 * float(y.abs().max())


@pytest.mark.gpu
def test_what_stays_with_the_library(gpu):
    """Strides, types, sizes and alignments that the kernel does not take give the library's product, with a workspace as without."""
    g = torch.Generator(device=gpu).manual_seed(3)
    ws = Workspace()

    def rnd(*shape):
        return torch.randn(*shape, device=gpu, generator=g).bfloat16()

    flat = rnd(2100 * 2100)
    forms = [(rnd(2048, 20).t(), rnd(2048, 2048)), (rnd(20, 2048), rnd(2048, 2048).t()), (rnd(20, 4096)[:, ::2], rnd(2048, 2048)),
             (rnd(20, 2052)[:, :2048], rnd(2048, 2048)), (flat[1:1 + 20 * 2048].view(20, 2048), rnd(2048, 2048)),
             (rnd(20, 2048), flat[1:1 + 2048 * 2048].view(2048, 2048)), (rnd(20, 2080), rnd(2048, 2080)), (rnd(20, 2048), rnd(2050, 2048)),
             (rnd(1, 2048).expand(20, 2048), rnd(2048, 2048)), (rnd(257, 2048), rnd(2048, 2048)), (rnd(20, 1024), rnd(2048, 1024))]
    for x, w in forms:
        out = torch.empty(x.shape[0], w.shape[0], device=gpu, dtype=torch.bfloat16)
        assert not ops.mid_rows(x, w, out, ws)
        y = x.double() @ w.double().t()
        ops.linear(x, w, out, ws)
        assert float((out.double() - y).abs().max()) <= 2 ** -7 * float(y.abs().max())
    x, w = rnd(20, 2048), rnd(2048, 2048)
    out = torch.empty(20, 2048, device=gpu, dtype=torch.bfloat16)
    assert ops.mid_rows(x, w, out, ws) and not ops.mid_rows(x, w, out, None)
    wide = torch.empty(17, 20500, device=gpu, dtype=torch.bfloat16)      # (more columns than one wave of workgroups has)
    assert not ops.mid_linear(rnd(17, 2048), rnd(20500, 2048), wide, ws)
    w.requires_grad_(True)
    assert not ops.mid_rows(x, w, out, ws)


def test_on_the_cpu_everything_is_the_librarys():
    x, w = torch.randn(20, 2048).bfloat16(), torch.randn(2048, 2048).bfloat16()
    out = torch.empty(20, 2048, dtype=torch.bfloat16)
    ws = Workspace()
    assert not ops.mid_rows(x, w, out, ws) and not ops.linear_glu(x, w, out[:, :1024].contiguous(), ws)
    assert torch.equal(ops.linear(x, w, out, ws), torch.matmul(x, w.t())) and not ws.buffers

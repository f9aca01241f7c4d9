"""The few-row linear kernel (csrc/kernels/row_linear.hip) against an fp64 product of the same bf16 operands, and the rule
that sends a call to it.

Bounds: fp32 accumulation of K terms errs by at most about sqrt(K) 2^-24 of the terms' norm, far below the rounding of a
bf16 result, 2^-8 of itself.  A squared ReLU on the way in rounds every term by 2^-8 more: together 2^-7.  Of a gated pair
gate, up and product are rounded, 2^-8 each; the gate's error reaches silu(y) times 1 + y (1 - sigmoid(y)), at most 1.28 for
y > 0 (for y < 0 the value is below 0.28 of the pair's scale): 3.28 x 2^-8, under 2^-6.  All relative to the largest
result.
"""
import pytest
import torch

from symmetry_amd import ops

# (outputs, K): one and several 8- and 16-row tiles with remainders, one chunk, an odd and an even number of chunks, four waves
SHAPES = [(4, 8), (1000, 16), (20, 200), (2052, 256), (2048, 2048), (68, 512), (3068, 8192), (3084, 1024), (4100, 1280),
          (5000, 14336), (24580, 2048), (24588, 1536)]


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", SHAPES)
@pytest.mark.parametrize("M", [1, 3, 16])
def test_row_linear(gpu, M, N, K):
    g = torch.Generator(device=gpu).manual_seed(N + K + M)
    wide = torch.randn(M, K + 24, device=gpu, generator=g).bfloat16()
    x = wide[:, 8:8 + K]                                   # a column range of a wider matrix
    w = (torch.randn(2 * N, K, device=gpu, generator=g) * K ** -0.5).bfloat16()
    y = x.double() @ w[:N].double().t()
    for dtype in (torch.bfloat16, torch.float32):
        room = torch.full((M, N + 8), 7.0, device=gpu, dtype=dtype)
        out = room[:, :N]
        assert ops.few_rows(x, w[:N], out)
        (ops.linear if dtype == torch.bfloat16 else ops.linear_f32)(x, w[:N], out)
        assert float((out.double() - y).abs().max()) <= (2 ** -7 if dtype == torch.bfloat16 else 2 ** -14) * float(y.abs().max())
        assert bool((room[:, N:] == 7).all())
    out = torch.empty(M, N, device=gpu, dtype=torch.bfloat16)
    r = torch.relu(x.double()) ** 2 @ w[:N].double().t()
    ops.row_linear(x, w[:N], out, relu2=True)
    assert float((out.double() - r).abs().max()) <= 2 ** -7 * float(r.abs().max())
    u = x.double() @ w[N:].double().t()
    ops.row_linear(x, w, out, glu=True)
    p = y * torch.sigmoid(y) * u
    assert float((out.double() - p).abs().max()) <= 2 ** -6 * max(float(p.abs().max()), 1.0)


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(20, 1536), (4100, 1536), (4100, 2048), (12308, 2048), (4104, 3072), (4108, 4096), (20, 4096),
                                 (40972, 2048), (6144, 4096)])
@pytest.mark.parametrize("M", [1, 8, 9, 16])
def test_row_linear_tiles_in_turn(gpu, M, N, K):
    """Workgroups that walk several tiles: every width they take, one tile, a second one of some, an odd number, a cut last one;
    gated pairs of one tile; and up to 8 rows against up to 16 of the forms without a walk."""
    test_row_linear(gpu, M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(12, 512), (2044, 768), (2048, 1024), (60, 1280), (28, 1536), (36, 1792), (2048, 2816), (20, 8192), (36, 3072),
                                 (2052, 512), (4096, 768), (4092, 1280), (4100, 1024), (8192, 512), (8188, 2816), (8196, 768), (12292, 512),
                                 (17444, 1280), (24572, 512), (2052, 8192), (40964, 768), (50304, 768), (49148, 768), (73732, 512),
                                 (4100, 8448), (8196, 8448)])
@pytest.mark.parametrize("M", [1, 8, 9, 16])
def test_row_linear_waves_and_tiles(gpu, M, N, K):
    """Every number of waves, 8-row tiles up to 2048 outputs, then one, two and three 16-row tiles a workgroup, at the lines between
    them with cut last tiles, one block of K a wave, an odd and an even number of them; one, two and three tiles past 40960 outputs."""
    test_row_linear(gpu, M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(32768, 2048), (8192, 2048), (12292, 1024), (6148, 4096), (20484, 2560), (3000, 8192), (64, 4096), (2048, 14336)])
@pytest.mark.parametrize("M", [1, 8, 16])
def test_row_linear_fp32_sums(gpu, M, N, K):
    """fp32 results are sums of parts.  An fp32 rounding errs by 0.4 x 2^-24 of the value (uniform in an ulp, values spread over a
    binade) and the value of a chain of n grows as sqrt(j / n): 0.4 x 2^-24 sqrt(n / 2) of its end.  A matrix instruction
    rounds once for each 8 products: 16 times in a block of 128 (outputs up to 2048: 32 in one of 256), then once a block.  A fifth
    for what this model leaves out."""
    g = torch.Generator(device=gpu).manual_seed(N + K + M)
    x, out = torch.randn(M, K, device=gpu, generator=g).bfloat16(), torch.empty(M, N, device=gpu)
    w = (torch.randn(N, K, device=gpu, generator=g) * K ** -0.5).bfloat16()
    assert ops.few_rows(x, w, out)
    ops.linear_f32(x, w, out)
    want, block = x.double() @ w.double().t(), 256 if N <= 2048 else 128
    assert float((out.double() - want).norm() / want.norm()) <= 1.2 * 0.4 * 2 ** -24 * (block / 16 + K / block / 2) ** 0.5


@pytest.mark.gpu
def test_linear_accepts_every_form(gpu):
    """Strides, types, sizes and alignments that the kernel does not take stay with the library and give the same product."""
    g = torch.Generator(device=gpu).manual_seed(3)

    def rnd(*shape):
        return torch.randn(*shape, device=gpu, generator=g).bfloat16()

    flat = rnd(40 * 300)
    forms = [
        (rnd(256, 8).t(), rnd(64, 256), None), (rnd(8, 256), rnd(256, 64).t(), None), (rnd(8, 512)[:, ::2], rnd(64, 256), None),
        (rnd(8, 260)[:, :256], rnd(64, 256), None), (flat[1:1 + 8 * 256].view(8, 256), rnd(64, 256), None),
        (rnd(8, 256), flat[1:1 + 40 * 256].view(40, 256), None), (rnd(8, 300), rnd(64, 300), None), (rnd(8, 256), rnd(63, 256), None),
        (rnd(1, 256).expand(8, 256), rnd(64, 256), None), (rnd(17, 256), rnd(64, 256), None), (rnd(0, 256), rnd(64, 256), None),
        (rnd(8, 256), rnd(64, 256), torch.empty(64, 8, device=gpu, dtype=torch.bfloat16).t()),
    ]
    for x, w, out in forms:
        if out is None:
            out = torch.empty(x.shape[0], w.shape[0], device=gpu, dtype=torch.bfloat16)
        assert not ops.few_rows(x, w, out)
        y = x.double() @ w.double().t()
        ops.linear(x, w, out)
        if y.numel():
            assert float((out.double() - y).abs().max()) <= 2 ** -7 * float(y.abs().max())
    x, w = rnd(8, 256), rnd(64, 256)
    assert torch.equal(ops.linear(x, w), torch.matmul(x, w.t()))                 # no out: the library allocates it
    w.requires_grad_(True)
    assert not ops.few_rows(x, w, torch.empty(8, 64, device=gpu, dtype=torch.bfloat16))
    ops.linear(x, w).float().sum().backward()
    assert w.grad is not None


def test_linear_of_traced_tensors():
    """A tracer's fake GPU tensors have no memory: they take the library's product (nothing is launched here)."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode():
        x, w = torch.empty(8, 256, device="cuda", dtype=torch.bfloat16), torch.empty(64, 256, device="cuda", dtype=torch.bfloat16)
        out, wide = torch.empty(8, 64, device="cuda", dtype=torch.bfloat16), torch.empty(8, 64, device="cuda")
        assert not ops.few_rows(x, w, out)
        assert ops.linear(x, w, out=out) is out
        assert ops.linear_f32(x, w, out=wide) is wide


def test_linear_while_compiling(monkeypatch):
    monkeypatch.setattr(ops, "_gpu", lambda t: True)
    x, w, out = torch.zeros(8, 256).bfloat16(), torch.zeros(64, 256).bfloat16(), torch.empty(8, 64).bfloat16()
    assert ops.few_rows(x, w, out)
    monkeypatch.setattr(torch.compiler, "is_compiling", lambda: True)
    assert not ops.few_rows(x, w, out)


@pytest.mark.parametrize("strict", [False, True])
@pytest.mark.parametrize("workspace", [False, True])
def test_linear_exports_any_number_of_rows(workspace, strict):
    """One graph for row counts on both sides of the kernels' limits (16 and 256): no size is compared while tracing."""
    from symmetry_amd.models.transformer import Workspace

    ws = Workspace() if workspace else None
    w = torch.randn(64, 256).bfloat16()

    class Layer(torch.nn.Module):
        def forward(self, x, w, out):
            return ops.linear(x, w, out, ws)

    def args(rows):
        return torch.randn(rows, 256).bfloat16(), w, torch.empty(rows, 64).bfloat16()

    rows = torch.export.Dim("rows", min=2, max=1000)
    layer = torch.export.export(Layer(), args(40), dynamic_shapes=({0: rows}, None, {0: rows}), strict=strict).module()
    for n in (2, 12, 300):
        x, _, out = args(n)
        assert torch.equal(layer(x, w, out), x @ w.t())


def test_linear_is_compiled_and_traced_once_for_all_rows():
    from torch.fx.experimental.proxy_tensor import make_fx

    from symmetry_amd.models.transformer import Workspace

    ws, w, graphs = Workspace(), torch.randn(64, 256).bfloat16(), []

    def layer(x, out):
        return ops.linear(x, w, out, ws), ops.linear_glu(x, w, out[:, :32], ws)

    def keep(graph, example):
        graphs.append(graph)
        return graph.forward

    compiled = torch.compile(layer, dynamic=True, backend=keep)
    for n in (40, 12, 300):
        compiled(torch.randn(n, 256).bfloat16(), torch.empty(n, 64).bfloat16())
    assert len(graphs) == 1
    traced = make_fx(layer, tracing_mode="symbolic", _allow_non_fake_inputs=True)(torch.randn(40, 256).bfloat16(),
                                                                                  torch.empty(40, 64).bfloat16())
    assert not [g for g in traced.shape_env.guards if "<" in str(g.expr) or ">" in str(g.expr)]      # (sizes that have to be equal aside)


def test_linear_of_dual_tensors(monkeypatch):
    """A product into ``out`` has no forward derivative: refused by the library, not computed without it."""
    monkeypatch.setattr(ops, "_gpu", lambda t: True)
    x, w, out = torch.zeros(8, 256).bfloat16(), torch.zeros(64, 256).bfloat16(), torch.empty(8, 64).bfloat16()
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        with pytest.raises(RuntimeError, match="forward AD"):
            ops.linear(dual, w, out=out)


def test_row_linear_reference_cpu():
    x, w = torch.randn(3, 32).bfloat16(), torch.randn(16, 32).bfloat16()
    out = torch.empty(3, 8, dtype=torch.bfloat16)
    assert not ops.few_rows(x, w, out)                                            # CPU tensors: the plain product
    ops.row_linear(x, w, out, glu=True)
    y = (x.float() @ w.float().t()).bfloat16().float()
    assert torch.equal(out, (y[:, :8] * torch.sigmoid(y[:, :8]) * y[:, 8:]).bfloat16())
    ops.row_linear(x, w[:8], out, relu2=True)
    assert torch.equal(out, ((torch.relu(x.float()) ** 2).bfloat16().float() @ w[:8].float().t()).bfloat16())


@pytest.mark.gpu
@pytest.mark.parametrize("M", [17, 32, 33, 500])
@pytest.mark.parametrize("N,K", [(4, 128), (16, 896), (12, 1152), (8, 1920), (16, 2048)])
def test_few_outputs_of_many_rows(gpu, M, N, K):
    """ops.linear_f32 of up to 16 outputs: blocks of K that fill no turn of the waves, one and more; column ranges of wider matrices.
    fp32 sums of K products against 64 bits, at most four times sqrt(K) 2^-24 of the vectors' norms."""
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    x = torch.randn(M, K + 24, device=gpu, generator=g).bfloat16()[:, 8:8 + K]
    w = (torch.randn(N, K, device=gpu, generator=g) * K ** -0.5).bfloat16()
    room = torch.full((M + 1, N + 8), 7.0, device=gpu)
    out = room[:M, :N]
    assert ops.narrow_f32(x, w, out) and not ops.narrow_f32(x[:16], w, out[:16]) and not ops.narrow_f32(x[:, 1:], w[:, 1:], out)
    ops.linear_f32(x, w, out)
    want = x.double() @ w.double().t()
    bound = 4 * K ** 0.5 * 2.0 ** -24 * float(x.double().norm(dim=1).max() * w.double().norm(dim=1).max())
    assert float((out.double() - want).abs().max()) <= bound
    assert bool((room[:, N:] == 7).all()) and bool((room[M] == 7).all())

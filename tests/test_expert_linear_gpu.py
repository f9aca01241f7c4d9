"""Gated and fp32-output expert products (``ops.expert_linear``): every form at the edges of its tiles."""
import pytest
import torch

from symmetry_amd import ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def segments(E: int, R: int) -> torch.Tensor:
    """Uneven segments: an empty one, a single row, the rest at random cuts."""
    cuts = sorted(torch.randint(min(1, R), R + 1, (E - 3,)).tolist())
    return torch.tensor([0, 0, min(1, R)] + cuts + [R]).int()


@pytest.mark.parametrize("shape", [(4, 128, 192), (7, 200, 64), (5, 262, 320), (4, 384, 1536), (16, 144, 2048)])
@pytest.mark.parametrize("R", [1, 17, 64, 129, 700, 3000])
def test_gated_and_fp32_products(R, shape):
    """Against 64-bit products.  fp32: K products of bf16 values summed in fp32, |error| <= K 2^-24 sum |x w| and in practice
    its root (4 sqrt(K) 2^-24 |x| |w| here); gated: the same error of both rows through silu(g) u (|silu'| <= 1.1, the
    exponential to 2^-20), and the rounding to bf16 (2^-8)."""
    E, N, K = shape
    print("expert_linear", R, shape, flush=True)
    torch.manual_seed(R + N)
    off = segments(E, R)
    x, W = torch.randn(R // 2 + 1, K).to(BF16), (torch.randn(E, 2 * N, K) * K ** -0.5).to(BF16)
    src = torch.randint(0, x.shape[0], (R,)).int()
    g, u = torch.zeros(R, N, dtype=torch.float64), torch.zeros(R, N, dtype=torch.float64)
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        p = x[src[a:b].long()].double() @ W[e].double().t()
        g[a:b], u[a:b] = p[:, :N], p[:, N:]
    norm = x.double().norm(dim=1).max() * W.double().norm(dim=2).max()
    eps = 4 * K ** 0.5 * 2.0 ** -24 * norm
    H = ops._hyb()
    xd, sd, Wd, od = x.cuda(), src.cuda(), W.cuda(), off.cuda()
    gate = Wd[:, :N].contiguous()
    want = g / (1 + torch.exp(-g)) * u
    bound = 2.0 ** -8 * want.abs() + 1.1 * eps * (g.abs() + u.abs()) + 2.0 ** -20 * want.abs() + 1e-30
    for impl in (1, 2, 3, -1):
        y = torch.full((R, N), 7.0, device="cuda")
        H.expert_linear(xd, sd, gate, od, y, False, impl)
        assert ((y.cpu().double() - g).abs() <= eps).all(), (impl, "fp32")
        z = torch.full((R + 1, N), 7.0, dtype=BF16, device="cuda")
        H.expert_linear(xd, sd, Wd, od, z[:R], False, impl, True)
        assert ((z[:R].cpu().double() - want).abs() <= bound).all(), (impl, "gated")
        assert (z[R] == 7.0).all()
        H.expert_linear(xd[src.cuda().long()], None, Wd, od, y2 := torch.empty_like(z[:R]), False, impl, True)
        assert torch.equal(y2, z[:R]), (impl, "gathered")


def test_refusals():
    """The gated and fp32-output products are bf16 MFMA forms; what they cannot take is an error before any launch."""
    H, off = ops._hyb(), torch.tensor([0, 4], dtype=torch.int32, device="cuda")
    x, W = torch.zeros(4, 40, dtype=BF16, device="cuda"), torch.zeros(1, 32, 40, dtype=BF16, device="cuda")
    with pytest.raises(RuntimeError):      # K % 32
        H.expert_linear(x, None, W, off, torch.zeros(4, 16, dtype=BF16, device="cuda"), False, -1, True)
    with pytest.raises(RuntimeError):
        H.expert_linear(x, None, W, off, torch.zeros(4, 32, device="cuda"), False)
    x, W = x[:, :32].contiguous(), W[:, :, :32].contiguous()
    with pytest.raises(RuntimeError):      # both epilogues
        H.expert_linear(x, None, W, off, torch.zeros(4, 16, dtype=BF16, device="cuda"), True, -1, True)
    with pytest.raises(RuntimeError):      # fp32 inputs have no gated form
        H.expert_linear(x.float(), None, W.float(), off, torch.zeros(4, 16, device="cuda"), False, -1, True)
    with pytest.raises(RuntimeError):      # no all-shapes form of it
        H.expert_linear(x, None, W, off, torch.zeros(4, 16, dtype=BF16, device="cuda"), False, 0, True)


@pytest.mark.parametrize("T", [1, 16, 17, 700])
@pytest.mark.parametrize("E,k,d", [(16, 4, 2048), (8, 2, 384), (10, 3, 512), (2, 1, 128)])
def test_router_in_runs(T, E, k, d):
    """``runs`` chooses and weighs as moe_router + moe_route do, to the bit, also where a token's logits are not numbers, and
    lays the segments out over them."""
    print("route_topk runs", T, E, k, d, flush=True)
    torch.manual_seed(T + E)
    x, Wr = torch.randn(T, d).to(BF16).cuda(), torch.zeros(16, d, dtype=BF16)
    Wr[:E] = torch.randn(E, d) * 2 * d ** -0.5
    Wr[E // 2] = Wr[0]                         # a tie in every row
    x[T // 2, 5] = float("nan")
    Wr, R, i32 = Wr.cuda(), T * k, dict(dtype=torch.int32, device="cuda")
    logits, ids0, w0 = torch.empty(T, 16, device="cuda"), torch.empty(R, **i32), torch.empty(R, device="cuda")
    ops.moe_router(x, Wr, logits)
    ops.moe_route(logits, T, k, E, ids0, w0)
    ids, w, off = torch.empty(R, **i32), torch.empty(R, device="cuda"), torch.empty(E + 1, **i32)
    dst, src = torch.empty(R, **i32), torch.empty(R, **i32)
    ops.route_topk(x, Wr[:E], None, k, ids, w, off, dst, src, runs=True)
    rows = torch.arange(T) != T // 2           # (a row without numbers: any valid experts, equal weights)
    assert torch.equal(ids.view(T, k)[rows], ids0.view(T, k)[rows]) and torch.equal(w, w0)
    assert int(ids.min()) >= 0 and int(ids.max()) < E
    assert torch.equal(src[dst.long()].cpu(), (torch.arange(R) // k).int())
    assert torch.equal(off.diff().cpu().long(), torch.bincount(ids.cpu().long(), minlength=E))


@pytest.mark.parametrize("dtype,E,runs", [(BF16, 8, False), (BF16, 8, True), (BF16, 100, False), (torch.float32, 8, False)])
@pytest.mark.parametrize("value", [-float("inf"), float("nan")])
def test_rows_without_a_finite_logit(dtype, E, runs, value):
    """Both routers give such a row its first k experts in equal parts, and the other rows what they had."""
    T, d, k = 20, 128, 3
    torch.manual_seed(E)
    x, Wr = torch.rand(T, d).to(dtype).cuda(), torch.rand(E, d).to(dtype).cuda()
    bad = [0, 7, 19]

    def route(x):
        ids, off, dst, src = (torch.full((n,), -1, dtype=torch.int32, device="cuda") for n in (T * k, E + 1, T * k, T * k))
        w = torch.empty(T * k, device="cuda")
        ops.route_topk(x, Wr, None, k, ids, w, off, dst, src, runs=runs)
        assert sorted(dst.tolist()) == list(range(T * k)) and int(off[E]) == T * k
        return ids.view(T, k).cpu(), w.view(T, k).cpu()

    want, share = route(x)
    x = x.clone()
    x[bad] = value                                   # (positive router weights: every logit of the row is this value)
    ids, w = route(x)
    for t in range(T):
        if t in bad:
            assert ids[t].tolist() == list(range(k)) and torch.allclose(w[t], torch.full((k,), 1 / k))
        else:
            assert torch.equal(ids[t], want[t]) and torch.equal(w[t], share[t])


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs a second GPU")
def test_a_device_that_is_not_the_current_one():
    """Routing and expert products launch on their operands' device (an engine on "cuda:1" of a process whose current device is 0)."""
    torch.manual_seed(3)
    T, d, E, N, k = 40, 256, 8, 64, 2
    x, Wr, W = torch.randn(T, d).to(BF16), torch.randn(E, d).to(BF16), (torch.randn(E, 2 * N, d) * d ** -0.5).to(BF16)
    got = []
    with torch.cuda.device(0):
        for dev in ("cuda:0", "cuda:1"):
            ids, off, dst, src = (torch.empty(n, dtype=torch.int32, device=dev) for n in (T * k, E + 1, T * k, T * k))
            w, y = torch.empty(T * k, device=dev), torch.empty(T * k, N, dtype=BF16, device=dev)
            xd = x.to(dev)
            ops.route_topk(xd, Wr.to(dev), None, k, ids, w, off, dst, src, runs=True)
            ops.expert_linear(xd, src, W.to(dev), off, y, glu=True)
            torch.cuda.synchronize(dev)
            got.append([t.cpu() for t in (ids, w, off, dst, src, y)])
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("N,K", [(300, 2048), (2048, 1536), (300, 4096), (300, 2560)])
def test_rows_of_tiles_sum_alike(N, K, glu):
    """A row's bits do not depend on the tile that it lies in, nor on how many rows its expert and the others have."""
    torch.manual_seed(N)
    rows, W = torch.randn(30, K).to(BF16).cuda(), (torch.randn(4, N * (2 if glu else 1), K) * K ** -0.5).to(BF16).cuda()
    H, seen = ops._hyb(), []
    for counts in ((30, 30, 30, 30), (0, 300, 30, 270), (700, 60, 330, 30), (129, 2580, 30, 30)):
        src = torch.cat([torch.arange(n) for n in counts]).remainder(30).int().cuda()
        off = torch.tensor((0,) + counts).cumsum(0).int().cuda()
        y = torch.empty(sum(counts), N, dtype=BF16 if glu else torch.float32, device="cuda")
        assert H.expert_linear(rows, src, W, off, y, False, 2, glu) == 2
        for e in range(4):
            part = y[int(off[e]):int(off[e + 1])]
            seen.append((e, part[:30]))
            assert torch.equal(part[30:], part[:-30])
    for e, part in seen:
        assert len(part) == 0 or torch.equal(part, seen[e][1])


@pytest.mark.parametrize("E,R,N,K", [(3, 700, 256, 512), (4, 1000, 300, 576), (5, 2600, 262, 1024), (2, 1, 512, 512),
                                     (16, 9000, 2048, 512), (7, 5000, 1028, 1088), (70, 9100, 260, 512), (130, 3000, 512, 576)])
def test_persistent_tiles(E, R, N, K):
    """The persistent form where its tiles end: segments around 128 and 256 rows, several tiles a workgroup, whole ones cut for the
    last round, more experts than lanes, odd stage counts, outputs that fill no tile.  Bounds as above; the squared ReLU of p
    with error eps is off by 2 |p| eps + eps^2."""
    print("persistent tiles", E, R, N, K, flush=True)
    torch.manual_seed(R + K)
    sizes = [0, 1, 127, 128, 129, 255, 256, 257, 384, 385][: E - 1]
    while sum(sizes) > R:
        sizes.pop()
    sizes += [0] * (E - 1 - len(sizes))
    rest = R - sum(sizes)
    sizes = [s + rest // E for s in sizes]
    off = torch.tensor([0] + sizes).cumsum(0).tolist() + [R]
    x, W = torch.randn(R // 2 + 1, K).to(BF16).cuda(), (torch.randn(E, 2 * N, K) * K ** -0.5).to(BF16).cuda()
    src = torch.randint(0, x.shape[0], (R,)).int().cuda()
    p = torch.empty(R, 2 * N, dtype=torch.float64, device="cuda")
    for e in range(E):
        a, b = off[e], off[e + 1]
        p[a:b] = x[src[a:b].long()].double() @ W[e].double().t()
    g, u = p[:, :N], p[:, N:]
    eps = 4 * K ** 0.5 * 2.0 ** -24 * x.double().norm(dim=1).max() * W.double().norm(dim=2).max()
    H, od = ops._hyb(), torch.tensor(off, dtype=torch.int32, device="cuda")
    half = W[:, :N].contiguous()
    y = torch.full((R + 1, N), 7.0, device="cuda")
    assert H.expert_linear(x, src, half, od, y[:R], False, 3) == 3
    assert ((y[:R].double() - g).abs() <= eps).all() and (y[R] == 7.0).all()
    z = torch.full((R + 1, N), 7.0, dtype=BF16, device="cuda")
    assert H.expert_linear(x, src, W, od, z[:R], False, 3, True) == 3
    want = g / (1 + torch.exp(-g)) * u
    assert ((z[:R].double() - want).abs() <= (2.0 ** -8 + 2.0 ** -20) * want.abs() + 1.1 * eps * (g.abs() + u.abs()) + 1e-30).all()
    assert (z[R] == 7.0).all()
    assert H.expert_linear(x[src.long()], None, half, od, z[:R], True, 3) == 3
    want = g.clamp(min=0) ** 2
    assert ((z[:R].double() - want).abs() <= 2.0 ** -8 * want + 2 * g.abs() * eps + eps ** 2).all()
    assert H.expert_linear(x, src, half, od, z[:R], False, 3) == 3
    assert ((z[:R].double() - g).abs() <= 2.0 ** -8 * g.abs() + 2 * eps).all()


@pytest.mark.parametrize("shape", [(1, 8, 512), (4, 132, 512), (7, 200, 1536), (5, 262, 2048), (64, 40, 2048), (16, 1536, 3072)])
@pytest.mark.parametrize("R", [1, 16, 17, 64, 130, 512])
def test_walk_over_the_experts(R, shape):
    """The persistent form: empty experts, more than 16 rows of one, outputs that fill no unit, fewer units than workgroups and many
    of each.  Bounds as above; the squared ReLU doubles the error times the value."""
    E, N, K = shape
    print("expert walk", R, shape, flush=True)
    torch.manual_seed(R + N)
    off = torch.tensor([0] + sorted(torch.randint(0, R + 1, (E - 1,)).tolist()) + [R]).int()
    x, W = torch.randn(R // 2 + 1, K).to(BF16), (torch.randn(E, 2 * N, K) * K ** -0.5).to(BF16)
    src = torch.randint(0, x.shape[0], (R,)).int()
    p = torch.zeros(R, 2 * N, dtype=torch.float64)
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        p[a:b] = x[src[a:b].long()].double() @ W[e].double().t()
    g, u = p[:, :N], p[:, N:]
    eps = 4 * K ** 0.5 * 2.0 ** -24 * x.double().norm(dim=1).max() * W.double().norm(dim=2).max()
    H = ops._hyb()
    xd, sd, Wd, od = x.cuda(), src.cuda(), W.cuda(), off.cuda()
    gate = Wd[:, :N].contiguous()
    y = torch.full((R + 1, N), 7.0, device="cuda")
    assert H.expert_linear(xd, sd, gate, od, y[:R], False, 4) == 4
    assert ((y[:R].cpu().double() - g).abs() <= eps).all() and (y[R] == 7.0).all()
    z = torch.full((R + 1, N), 7.0, dtype=BF16, device="cuda")
    assert H.expert_linear(xd, sd, Wd, od, z[:R], False, 4, True) == 4
    want = g / (1 + torch.exp(-g)) * u
    bound = 2.0 ** -8 * want.abs() + 1.1 * eps * (g.abs() + u.abs()) + 2.0 ** -20 * want.abs() + 1e-30
    assert ((z[:R].cpu().double() - want).abs() <= bound).all() and (z[R] == 7.0).all()
    assert H.expert_linear(xd[sd.long()], None, gate, od, z[:R], True, 4) == 4
    want = g.clamp(min=0) ** 2
    assert ((z[:R].cpu().double() - want).abs() <= 2.0 ** -8 * want + 2 * eps * g.abs() + eps ** 2).all() and (z[R] == 7.0).all()
    H.expert_linear(xd[sd.long()], None, gate, od, z[:R], False, 4)
    assert ((z[:R].cpu().double() - g).abs() <= 2.0 ** -8 * g.abs() + eps).all() and (z[R] == 7.0).all()


@pytest.mark.parametrize("R,N,K,glu,form", [(32, 1536, 2048, True, 4), (32, 2048, 1536, False, 4), (512, 512, 1536, True, 4),
                                            (32, 1024, 2048, False, 1), (32, 1536, 512, True, 1), (32, 1536, 1024, False, 1),
                                            (513, 512, 1536, True, 2), (8191, 512, 1024, False, 3), (8128, 512, 1024, False, 2)])
def test_who_walks(R, N, K, glu, form):
    x, W = torch.randn(R, K).to(BF16).cuda(), torch.randn(64, N * (2 if glu else 1), K).to(BF16).cuda()
    off = torch.arange(65).mul(R).div(64, rounding_mode="floor").int().cuda()
    y = torch.empty(R, N, dtype=BF16, device="cuda")
    assert ops._hyb().expert_linear(x, None, W, off, y, False, -1, glu) == form
    assert ops._hyb().expert_linear_choice(R, 64, N, K, R, glu, False) == form


@pytest.mark.parametrize("T", [1, 7, 16])
@pytest.mark.parametrize("E,k,d", [(16, 4, 2048), (8, 2, 512), (5, 5, 1536), (20, 3, 1024), (64, 8, 2048)])
def test_router_of_the_residual(T, E, k, d):
    """The norm inside the router: its rows are ops.rms_norm's but for sums in another order (fp32: a bf16 step, 2^-7 of a value, on
    a few), and from those rows the choices, weights and segments are route_topk's own, to the bit."""
    print("route_topk resid", T, E, k, d, flush=True)
    torch.manual_seed(T + E)
    resid, norm = torch.randn(T, d).cuda() * 3, torch.rand(d).to(BF16).cuda()
    Wr, R, i32 = (torch.randn(E, d) * 2 * d ** -0.5).to(BF16).cuda(), T * k, dict(dtype=torch.int32, device="cuda")
    xn, x = torch.empty(T, d, dtype=BF16, device="cuda"), torch.full((T + 1, d), 7.0, dtype=BF16, device="cuda")
    ops.rms_norm(resid, norm, 1e-5, xn)
    got, want = ([torch.empty(R, **i32), torch.empty(R, device="cuda")] + [torch.empty(n, **i32) for n in (E + 1, R, R)]
                 for _ in range(2))
    assert ops.route_norm_fits(T, d, E)
    ops.route_topk(x[:T], Wr, None, k, *got, runs=E <= 16, resid=resid, norm=norm, eps=1e-5)
    diff = (x[:T].float() - xn.float()).abs()
    assert bool((diff <= 2.0 ** -7 * xn.float().abs()).all()) and int((diff > 0).sum()) <= T * d // 100 and bool((x[T] == 7).all())
    ops.route_topk(x[:T], Wr, None, k, *want, runs=E <= 16)
    for a, b in zip(got[:3], want[:3]):
        assert torch.equal(a, b)
    assert torch.equal(got[4][got[3].long()].cpu(), (torch.arange(R) // k).int())
    with pytest.raises(RuntimeError):      # (17 rows are two workgroups' work)
        big = torch.empty(17, d, dtype=BF16, device="cuda")
        ops.route_topk(big, Wr, None, 1, *(torch.empty(99, dtype=t.dtype, device="cuda") for t in got), resid=big.float(), norm=norm, eps=1e-5)


def test_only_the_norming_router_writes_its_rows():
    """A router that reads its rows is declared to: one that writes them is recorded as a change of x, which a graph copies back."""
    for name, writes in (("route_topk", False), ("norm_route_topk", True)):
        x = getattr(ops._hyb(), name).default._schema.arguments[0]
        assert x.name == "x" and (x.alias_info is not None and x.alias_info.is_write) == writes


@pytest.mark.parametrize("R", [4, 60])
def test_choices_among_infinite_logits(R):
    """Infinite and missing logits keep their places: +inf first, ties to the lowest index, -inf and NaN never before a number."""
    d, E, k = 512, 16, 4
    bias = torch.zeros(E)
    bias[3], bias[5], bias[9] = float("inf"), float("-inf"), float("nan")
    x, Wr = torch.zeros(R, d, dtype=BF16).cuda(), torch.zeros(E, d, dtype=BF16).cuda()
    ids, off, dst, src = (torch.empty(n, dtype=torch.int32, device="cuda") for n in (R * k, E + 1, R * k, R * k))
    ops.route_topk(x, Wr, bias.cuda(), k, ids, torch.empty(R * k, device="cuda"), off, dst, src)
    assert ids.view(R, k).tolist() == [[3, 0, 1, 2]] * R
    bias[:] = float("-inf")
    bias[7] = 1.0
    w = torch.empty(R * k, device="cuda")
    ops.route_topk(x, Wr, bias.cuda(), k, ids, w, off, dst, src)
    assert ids.view(R, k).tolist() == [[7, 1, 2, 3]] * R and w.view(R, k).tolist() == [[1.0, 0.0, 0.0, 0.0]] * R


@pytest.mark.parametrize("M,N,K", [(2817, 1024, 1024), (1280, 2180, 1088), (400, 8192, 2048), (1025, 8192, 2048)])
def test_dense_gated_projection(M, N, K):
    """linear_glu of many rows: one expert's persistent tiles.  The gated product's bound from above."""
    torch.manual_seed(M)
    x, W = torch.randn(M, K, device="cuda").to(BF16), (torch.randn(2 * N, K, device="cuda") * K ** -0.5).to(BF16)
    out = torch.full((M + 1, N), 7.0, dtype=BF16, device="cuda")
    with torch.no_grad():
        assert ops.linear_glu(x, W, out[:M], None)
        p = x.double() @ W.double().t()
        g, u = p[:, :N], p[:, N:]
        want = g / (1 + torch.exp(-g)) * u
        eps = 4 * K ** 0.5 * 2.0 ** -24 * x.double().norm(dim=1).max() * W.double().norm(dim=1).max()
        bound = 2.0 ** -8 * want.abs() + 1.1 * eps * (g.abs() + u.abs()) + 2.0 ** -20 * want.abs() + 1e-30
        assert ((out[:M].double() - want).abs() <= bound).all() and (out[M] == 7.0).all()
        turned = torch.full_like(out, 7.0)                                          # eight gate rows, the eight up rows, the next ..
        eights = W.view(2, -1, 8, K).transpose(0, 1).reshape(2 * N, K) if N % 8 == 0 else W
        assert ops.linear_swiglu(x, eights, turned[:M]) == (N % 8 == 0)
        assert N % 8 or torch.equal(turned, out)
        wide = torch.empty(M, K + 64, device="cuda", dtype=BF16)
        assert not ops.linear_glu(wide[:, :K], W, out[:M], None)                    # rows of x apart
        assert not ops.linear_glu(x, W, torch.empty(M, N + 8, device="cuda", dtype=BF16)[:, :N], None)
        assert not ops.linear_glu(x[:300], W[:512], torch.empty(300, 256, device="cuda", dtype=BF16), None)      # the library's sizes
    x.requires_grad_(True)
    assert not ops.linear_glu(x, W, out[:M], None)

"""The prompt forms of the row kernels (short convolution, squared ReLU, residual + norm, gated
group norm) against 64-bit rows, on both sides of
the conditions that choose them."""
import pytest
import torch

from symmetry_amd import ops

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("C", [8, 24, 520, 1032, 13])
@pytest.mark.parametrize("taps", [4, 3])
@pytest.mark.parametrize("lens", [[300], [1, 2, 3, 4, 5, 250], [7, 130, 129], [255]])
def test_causal_conv(C, taps, lens):
    """Runs that begin anywhere in a group of 8 rows, with and without saved inputs; odd widths and other tap counts take the
    general kernel.  Four products in fp32 and one rounding to bf16 (2^-8 relative with silu's slope <= 1.1)."""
    print("causal_conv_silu", C, taps, lens, flush=True)
    torch.manual_seed(C + len(lens))
    T, S, i32 = sum(lens), len(lens), torch.int32
    z = torch.randn(T, C + 8).to(BF16)
    x, w, b = z[:, 8:], torch.randn(C, taps).to(BF16), torch.randn(C)
    state = torch.randn(S + 1, taps - 1, C).to(BF16)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist())
    prev = torch.full((T,), -1)
    want = torch.zeros(T, C, dtype=torch.float64)
    for s, n in enumerate(lens):
        old = state[s].double() if s % 2 == 0 else torch.zeros(taps - 1, C, dtype=torch.float64)
        prev[cu[s]] = -(s + 2) if s % 2 == 0 else -1
        seq = torch.cat([old, x[cu[s]:cu[s + 1]].double()])
        y = b.double() + sum(w[:, i].double() * seq[i:i + n] for i in range(taps))
        want[cu[s]:cu[s + 1]] = y / (1 + torch.exp(-y))
    zd = z.cuda()
    out = torch.full((T, C), 7.0, dtype=BF16, device="cuda")
    ops.causal_conv_silu(zd[:, 8:], w.cuda(), b.cuda(), state.cuda(), cu.to(i32).cuda(),
                         torch.repeat_interleave(torch.arange(S), torch.tensor(lens)).to(i32).cuda(), prev.to(i32).cuda(), S, out)
    err = (out.cpu().double() - want).abs()
    assert (err <= 2.0 ** -8 * want.abs() + 2e-5).all(), float(err.max())


@pytest.mark.parametrize("R,F,pad", [(1, 8, 0), (33, 264, 8), (257, 1032, 16), (40, 12, 0), (9, 64, 3)])
def test_relu_sq(R, F, pad):
    torch.manual_seed(F)
    z = torch.randn(R, F + pad).to(BF16).cuda()
    z[0, 0], z[R - 1, F - 1] = float("inf"), float("-inf")
    out = torch.empty(R, F, dtype=BF16, device="cuda")
    ops.relu_sq(z[:, :F], out)
    assert torch.equal(out, (z[:, :F].float().clamp_min(0) ** 2).to(BF16))


@pytest.mark.parametrize("T", [513, 512])
@pytest.mark.parametrize("d", [8, 264, 2048, 2056, 100])
@pytest.mark.parametrize("parts", ["a", "ab", "abc"])
def test_residual_mix(T, d, parts):
    """fp32 stream to 2^-22 of its summands; the norm's sum of d squares to 2^-20, its output rounded to bf16."""
    print("residual_mix_norm", T, d, parts, flush=True)
    torch.manual_seed(d)
    x, w, bias = torch.randn(T, d).cuda(), torch.randn(d).cuda(), torch.randn(d).cuda()
    a, b, c = torch.randn(T, d).to(BF16).cuda(), torch.randn(T, d).cuda(), torch.randn(T, d).to(BF16).cuda()
    b_, c_ = (b if "b" in parts else None), (c if "c" in parts else None)
    s = 0.5 * (a.double() + bias.double())
    size = 0.5 * (a.double().abs() + bias.double().abs()) + x.double().abs()
    if b_ is not None:
        s, size = s + 0.25 * b.double(), size + 0.25 * b.double().abs()
    if c_ is not None:
        s, size = s - 2.0 * c.double(), size + 2.0 * c.double().abs()
    want = x.double() + s
    out = torch.full((T, d), 7.0, dtype=BF16, device="cuda")
    ops.residual_mix_norm(x, a, 0.5, bias, b_, 0.25, c_, -2.0, w, 1e-5, 1.0, out)
    assert ((x.double() - want).abs() <= 2.0 ** -22 * size).all()
    n = want / (want.pow(2).mean(1, keepdim=True) + 1e-5).sqrt() * (1.0 + w.double())
    assert ((out.double() - n).abs() <= 2.0 ** -8 * n.abs() + 2e-5).all()


@pytest.mark.parametrize("T", [513, 512])
@pytest.mark.parametrize("groups,group,wlen", [(2, 264, 528), (1, 2048, 2048), (3, 2056, 2056), (1, 4096, 4096), (2, 300, 12),
                                               (1, 4104, 4104)])
@pytest.mark.parametrize("gate_first,sigmoid", [(True, False), (False, True)])
def test_gated_group_norm(T, groups, group, wlen, gate_first, sigmoid):
    """The norm's sum of a group's squares to 2^-20, the gate to 2^-20, the output rounded to bf16."""
    print("gated_group_norm", T, groups, group, gate_first, sigmoid, flush=True)
    torch.manual_seed(group)
    C = groups * group
    z = torch.randn(T, C + 8).to(BF16).cuda()
    y, w, gate = torch.randn(T, C).cuda(), torch.randn(wlen).cuda(), z[:, 8:]
    out = torch.full((T, C), 7.0, dtype=BF16, device="cuda")
    ops.gated_group_norm(y, gate, w, 1e-5, group, gate_first, out, sigmoid=sigmoid)
    g = gate.double().sigmoid()
    g = g if sigmoid else gate.double() * g
    v = y.double() * g if gate_first else y.double()
    n = v.view(T, groups, group)
    n = (n / (n.pow(2).mean(2, keepdim=True) + 1e-5).sqrt()).view(T, C) * w.double().repeat(C // wlen)
    n = n if gate_first else n * g
    assert ((out.double() - n).abs() <= 2.0 ** -8 * n.abs() + 2e-5).all()


@pytest.mark.parametrize("T", [513, 512])
@pytest.mark.parametrize("groups,group,wlen", [(8, 256, 256), (9, 256, 256), (5, 64, 320), (3, 8, 8), (40, 128, 128), (4, 96, 96)])
@pytest.mark.parametrize("gate_first,sigmoid", [(True, False), (False, True)])
def test_gated_group_norm_of_small_groups(T, groups, group, wlen, gate_first, sigmoid):
    """Groups of neighbouring lanes, rows that end inside a workgroup, and a width that keeps the general kernel; bounds as above."""
    test_gated_group_norm(T, groups, group, wlen, gate_first, sigmoid)


@pytest.mark.parametrize("T", [513, 512])
@pytest.mark.parametrize("d", [8, 264, 2048, 2056, 4096, 4104, 100])
def test_embed_norm(T, d):
    """A sum of d squares to 2^-20, the fp32 row to that as well; tokens from ids and from the step before."""
    print("embed_norm", T, d, flush=True)
    torch.manual_seed(d)
    table, w = torch.randn(50, d).to(BF16).cuda(), torch.randn(d).cuda()
    ids, prev = torch.randint(0, 50, (T,)).int().cuda(), torch.randint(0, 50, (9,)).int().cuda()
    src = torch.full((T,), -1).int().cuda()
    src[3], src[T - 1] = 5, 8
    x = torch.full((T + 1, d), 7.0, device="cuda")
    ops.embed_norm(ids, table, w, 1e-5, 1.0, x[:T], src, prev)
    tok = torch.where(src >= 0, prev[src.clamp_min(0).long()], ids).long()
    t = table[tok].double()
    want = t / (t.pow(2).mean(1, keepdim=True) + 1e-5).sqrt() * (1.0 + w.double())
    assert ((x[:T].double() - want).abs() <= 2.0 ** -19 * want.abs() + 1e-30).all() and (x[T] == 7.0).all()


@pytest.mark.parametrize("T", [513, 512])
@pytest.mark.parametrize("H,G,dk,dv,pairs,bias", [(16, 4, 128, 128, 32, True), (3, 1, 24, 40, 12, False), (2, 2, 8, 8, 0, True),
                                                  (5, 5, 64, 16, 32, True), (4, 2, 20, 16, 4, True), (4, 2, 16, 16, 3, True)])
def test_qkv_rope_cache(T, H, G, dk, dv, pairs, bias):
    """Pieces of eight entries: a head rotated in part, whole or not at all, rows without a place in the cache, and sizes that keep the
    general kernel.  Two products and a sum in fp32 of bf16 values, rounded to bf16."""
    print("qkv_rope_cache", T, H, G, dk, dv, pairs, flush=True)
    torch.manual_seed(T + dk)
    n, BS, NB = (H + G) * dk + G * dv, 16, 40
    z = torch.randn(T, n + 8).to(BF16).cuda()
    b = torch.randn(n).cuda() if bias else None
    pos = torch.randint(0, 200, (T,)).int().cuda()
    slots = torch.randperm(NB * BS)[:T].int().cuda()
    slots[2] = -1
    rope = torch.randn(200, pairs, 2).cuda() if pairs else None
    q = torch.full((T, H, dk), 7.0, dtype=BF16, device="cuda")
    k, v = (torch.full((NB, BS, G, e), 7.0, dtype=BF16, device="cuda") for e in (dk, dv))
    ops.qkv_rope_cache(z[:, 8:], b, H, G, dk, dv, pos, slots, rope, q, k, v)
    y = z[:, 8:].double() + (b.double() if bias else 0.0)
    qk, size = y[:, :(H + G) * dk].reshape(T, H + G, dk).clone(), y[:, :(H + G) * dk].reshape(T, H + G, dk).abs()
    if pairs:
        c, s = rope[pos.long()].double()[:, None, :, 0], rope[pos.long()].double()[:, None, :, 1]
        x0, x1 = qk[..., 0:2 * pairs:2].clone(), qk[..., 1:2 * pairs:2].clone()
        size = size.clone()
        size[..., 0:2 * pairs:2] = (x0 * c).abs() + (x1 * s).abs()
        size[..., 1:2 * pairs:2] = (x1 * c).abs() + (x0 * s).abs()
        qk[..., 0:2 * pairs:2], qk[..., 1:2 * pairs:2] = x0 * c - x1 * s, x1 * c + x0 * s
    kept = slots >= 0
    at = slots[kept].long()
    for got, want, room in ((q, qk[:, :H], size[:, :H]), (k.view(-1, G, dk)[at], qk[kept, H:], size[kept, H:]),
                            (v.view(-1, G, dv)[at], y[kept, (H + G) * dk:].view(-1, G, dv), y[kept, (H + G) * dk:].view(-1, G, dv).abs())):
        assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -21 * room).all()
    rest = torch.ones(NB * BS, dtype=torch.bool, device="cuda")
    rest[at] = False
    assert (k.view(-1, G, dk)[rest] == 7.0).all() and (v.view(-1, G, dv)[rest] == 7.0).all()

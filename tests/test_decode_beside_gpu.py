"""Launches of a decode step that do what several did: a token's recurrence with its norm and gate, beside attention; row work beside a
product; two products; sums that apply a norm's factor.  Against the references, or against the separate launches where the same code
runs in both (then bit for bit)."""
import pytest
import torch

from symmetry_amd import ops
from symmetry_amd.ops import reference

pytestmark = pytest.mark.gpu
B16, F32, I32 = torch.bfloat16, torch.float32, torch.int32


def rnd(*shape, dtype=B16, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (torch.randn(shape, generator=g) * scale).to(dtype)


def slots_of(T, slots):
    """Row r starts from slot r (every fourth from zero) and ends in slot T + r, the first in place, the last nowhere."""
    prev = torch.tensor([-1 if r % 4 == 3 else -(r + 2) for r in range(T)], dtype=I32)
    save = torch.tensor([0 if r == 0 else -1 if r == T - 1 and T > 1 else T + r for r in range(T)], dtype=I32)
    assert 2 * T <= slots
    return prev, save


def token_inputs(mode, T, H, N, P, rank=0):
    hpg = 1 if mode == 0 else H
    G = H // hpg
    width = G * N * 2 + H * P * 2 + (rank or (H * N if mode == 0 else H)) + 24
    wide = rnd(T, width - width % 8, seed=3)   # (views of a wider matrix)
    at = 0

    def cols(n):
        nonlocal at
        at += n + (-n % 8)
        return wide[:, at - n - (-n % 8):at - (-n % 8)]

    q, k, v, gate = cols(G * N), cols(G * N), cols(H * P), cols(H * P)
    dz = cols(rank if rank else H * N if mode == 0 else H)
    low, dzw = (dz, rnd(H * N, rank, scale=rank ** -0.5, seed=4)) if rank else (None, dz)
    dbias = rnd(H * N if mode == 0 else H, dtype=F32, seed=5) + (2.0 if mode == 0 else -2.0)
    dparam = 16.0 if mode == 0 else rnd(H, dtype=F32, seed=6)
    skip = None if mode == 0 else rnd(H, dtype=F32, seed=7)
    state = rnd(2 * T + 1, H, N, P, dtype=F32, seed=8)
    w = 1 + 0.1 * rnd(P if mode == 0 else H * P, dtype=F32, seed=9)
    return q, k, v, gate, low, dzw, dbias, dparam, skip, state, w, hpg


def gpu(t):
    if t is None or not torch.is_tensor(t):
        return t
    if t.dim() == 2 and not t.is_contiguous():      # a view keeps its place in the wider matrix
        base = t._base.cuda()
        return base.as_strided(t.size(), t.stride(), t.storage_offset())
    return t.cuda()


@pytest.mark.parametrize("mode,T,H,N,P,rank", [
    (0, 1, 8, 128, 256, 16), (0, 5, 8, 128, 256, 0), (0, 3, 3, 128, 128, 24), (0, 8, 4, 64, 64, 8), (0, 2, 2, 64, 256, 0),
    (1, 8, 64, 128, 64, 0), (1, 1, 16, 64, 64, 0), (1, 3, 5, 128, 256, 0), (1, 17, 16, 64, 128, 0)])
def test_decay_token(mode, T, H, N, P, rank):
    q, k, v, gate, low, dz, dbias, dparam, skip, state, w, hpg = token_inputs(mode, T, H, N, P, rank)
    prev, save = slots_of(T, state.shape[0])
    dzr = dz if low is None else (low.float() @ dz.float().t()).to(B16)
    st, y = state.clone(), torch.zeros(T, H, P)
    reference.decay_scan(mode, q, k, v, dzr, dbias, dparam, skip, N ** -0.5, H, N, P, hpg, st, None, prev, save, T, y)
    y = y.view(T, H * P)
    gst, out = state.cuda(), torch.empty(T, H * P, dtype=B16, device="cuda")
    ss = torch.empty(T, H, device="cuda") if mode == 1 else None
    done = ops.decay_token(mode, gpu(q), gpu(k), gpu(v), gpu(dz), gpu(low), gpu(dbias), gpu(dparam), gpu(skip), N ** -0.5, H, N, P, hpg,
                           gst, prev.cuda(), save.cuda(), gpu(gate), gpu(w), 1e-5, out, ss)
    assert done
    if mode == 0:
        want = torch.empty(T, H * P)
        reference.gated_group_norm(y, gate, w, 1e-5, P, False, want)
    else:
        s = y * torch.nn.functional.silu(gate.float())
        want = s * w
        assert torch.allclose(ss.cpu(), (s * s).view(T, H, P).sum(2), rtol=2e-5)
    # fp32 up to the one rounding to bf16; where the low-rank sums' order turns that rounding, an ulp of a pre-activation on the decays
    assert torch.allclose(out.float().cpu(), want, rtol=2 ** -7, atol=2e-3 if rank else 2e-5)
    tol = dict(rtol=2e-3, atol=2e-3) if rank else dict(rtol=1e-5, atol=1e-5)
    assert torch.allclose(gst.cpu(), st, **tol)


def test_decay_token_refuses():
    for N, P in ((96, 64), (128, 32), (128, 512)):
        q, k, v, gate, low, dz, dbias, dparam, skip, state, w, hpg = token_inputs(0, 2, 2, N, P)
        prev, save = slots_of(2, state.shape[0])
        out = torch.empty(2, 2 * P, dtype=B16, device="cuda")
        done = ops.decay_token(0, gpu(q), gpu(k), gpu(v), gpu(dz), None, gpu(dbias), dparam, None, 1.0, 2, N, P, 1, state.cuda(),
                               prev.cuda(), save.cuda(), gpu(gate), gpu(w), 1e-5, out)
        assert not done


@pytest.mark.parametrize("T,D,window,P", [(1, 128, 1024, 256), (9, 128, 300, 256), (16, 64, 1 << 30, 128), (40, 128, 64, 64)])
def test_attn_beside_decay(T, D, window, P):
    H, G, BS, HR, N = 8, 4, 64, 4, 128
    ctx = [1 + (97 * r) % 700 for r in range(T)]
    per = [-(-c // BS) for c in ctx]
    tables = torch.zeros(T, max(per), dtype=I32)
    at = 1
    for r in range(T):
        tables[r, :per[r]] = torch.arange(at, at + per[r])
        at += per[r]
    kc, vc = rnd(at, BS, G, D, seed=1).cuda(), rnd(at, BS, G, D, seed=2).cuda()
    q, hg = rnd(T, H, D, seed=3).cuda(), rnd(T, H, seed=4).cuda()
    pos = torch.tensor([c - 1 for c in ctx], dtype=I32).cuda()
    rows, tables = torch.arange(T, dtype=I32).cuda(), tables.cuda()
    keys, parts = ops.window_attn_split(T, G, min(tables.shape[1] * BS, window + 31))
    split = (torch.empty(T, H, parts, D, device="cuda"), torch.empty(T, H, parts, 2, device="cuda"),
             torch.zeros(T * G, dtype=I32, device="cuda"), keys)
    dq, dk, dv, gate, low, dz, dbias, tau, _, state, w, _ = token_inputs(0, T, HR, N, P, 16)
    dq, dk, dv, gate, low, dz, dbias, w = map(gpu, (dq, dk, dv, gate, low, dz, dbias, w))
    prev, save = (t.cuda() for t in slots_of(T, state.shape[0]))
    s1, s2 = state.cuda(), state.cuda()
    o1, o2 = torch.empty_like(q), torch.empty_like(q)
    g1, g2 = (torch.empty(T, HR * P, dtype=B16, device="cuda") for _ in range(2))
    assert ops.window_attn(q, kc, vc, tables, rows, pos, window, D ** -0.5, hg, o1, split=split) == 3
    done = ops.decay_token(0, dq, dk, dv, dz, low, dbias, tau, None, 0.1, HR, N, P, 1, s1, prev, save, gate, w, 1e-5, g1)
    assert done
    for _ in range(2):       # (the arrival counters are zero again)
        s2.copy_(state)
        done = ops.window_attn_decay(q, kc, vc, tables, rows, pos, window, D ** -0.5, hg, o2, split, dq, dk, dv, dz, low, dbias, tau, 0.1,
                                     HR, N, P, s2, prev, save, gate, w, 1e-5, g2)
        assert done
        assert torch.equal(o1, o2) and torch.equal(g1, g2) and torch.equal(s1, s2)


@pytest.mark.parametrize("M,N,K", [(1, 2048, 8192), (8, 2048, 8192), (9, 264, 3072), (16, 4096, 2048), (5, 10240, 2048)])
def test_row_work_beside_a_product(M, N, K):
    x, w = rnd(M, K, seed=1).cuda(), rnd(N, K, scale=K ** -0.5, seed=2).cuda()
    want = torch.empty(M, N, dtype=B16, device="cuda")
    ops.row_linear(x, w, want, relu2=True)
    # rotation and cache rows
    H, G, D, T = 6, 2, 64, M
    z, bias = rnd(T, (H + 2 * G) * D + 8, seed=3).cuda(), rnd((H + 2 * G) * D, dtype=F32, seed=4).cuda()
    pos, slot = torch.arange(T, dtype=I32).cuda() + 5, torch.tensor([-1 if r == 2 else 3 * r + 1 for r in range(T)], dtype=I32).cuda()
    rope = rnd(64, D // 4, 2, dtype=F32, seed=5).cuda()
    got = []
    for side in range(2):
        q = torch.zeros(T, H, D, dtype=B16, device="cuda")
        kc, vc = (torch.zeros(4, 16, G, D, dtype=B16, device="cuda") for _ in range(2))
        out = torch.empty_like(want)
        args = (z, bias, H, G, D, D, pos, slot, rope, q, kc, vc)
        if side:
            done = ops.row_linear_rope(x, w, out, *args)
            assert done
            assert torch.equal(out, want)
        else:
            ops.qkv_rope_cache(*args)
        got.append((q, kc, vc))
    assert all(torch.equal(a, b) for a, b in zip(*got))
    # convolution
    C, taps = 1000, 4
    xin, cw, cb = rnd(T, C + 8, seed=6).cuda()[:, 8:], rnd(C, taps, seed=7).cuda(), rnd(C, dtype=F32, seed=8).cuda()
    prev, save = (t.cuda() for t in slots_of(T, 2 * T + 1))
    got = []
    for side in range(2):
        st, co = rnd(2 * T + 1, taps - 1, C, seed=9).cuda(), torch.empty(T, C, dtype=B16, device="cuda")
        out = torch.empty_like(want)
        if side:
            done = ops.row_linear_conv(x, w, out, xin, cw, cb, st, prev, save, co)
            assert done
            assert torch.equal(out, want)
        else:
            ops.causal_conv_silu(xin, cw, cb, st, None, None, prev, T, co, save)
        got.append((st, co))
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("N,K", [(64, 128), (16400, 4096)])      # low-rank factors and walks over many tiles go without
def test_row_work_beside_refuses(N, K):
    x, w = rnd(2, K).cuda(), rnd(N, K).cuda()
    out, st = torch.empty(2, N, dtype=B16, device="cuda"), torch.zeros(4, 3, 64, dtype=B16, device="cuda")
    xin, cw, cb = rnd(2, 64).cuda(), rnd(64, 4).cuda(), torch.zeros(64, device="cuda")
    prev = torch.full((2,), -1, dtype=I32, device="cuda")
    done = ops.row_linear_conv(x, w, out, xin, cw, cb, st, prev, prev, torch.empty(2, 64, dtype=B16, device="cuda"))
    assert not done


@pytest.mark.parametrize("M,N,K", [(1, 2048, 2048), (8, 2048, 2048), (16, 2048, 4096), (3, 4096, 2048), (7, 64, 64), (24, 2048, 2048)])
def test_two_products(M, N, K):
    x, w = [rnd(M, K, seed=s).cuda() for s in (1, 2)], [rnd(N, K, seed=s, scale=K ** -0.5).cuda() for s in (3, 4)]
    out, want = ([torch.empty(M, N, dtype=B16, device="cuda") for _ in range(2)] for _ in range(2))
    ops.linear_two(x[0], w[0], out[0], x[1], w[1], out[1])
    for i in range(2):
        ops.linear(x[i], w[i], want[i])
        assert torch.equal(out[i], want[i])


@pytest.mark.parametrize("T,d,n", [(1, 2048, 64), (8, 2048, 5), (3, 5000, 130), (700, 2048, 64)])
def test_sum_applies_a_norms_factor(T, d, n):
    x, a, b = rnd(T, d, dtype=F32, seed=1), rnd(T, d, seed=2), rnd(T, d, seed=3)
    ss, w = rnd(T, n, dtype=F32, seed=4).abs(), rnd(d, dtype=F32, seed=5, scale=0.1)
    want, out = x.clone(), torch.empty(T, d, dtype=B16)
    ops.residual_mix_norm(want, a, 0.5, None, b, 2.0, None, 0.0, w, 1e-5, 1.0, out, ss, 4096, 1e-5)
    gx, go = x.cuda(), torch.empty(T, d, dtype=B16, device="cuda")
    ops.residual_mix_norm(gx, a.cuda(), 0.5, None, b.cuda(), 2.0, None, 0.0, w.cuda(), 1e-5, 1.0, go, ss.cuda(), 4096, 1e-5)
    assert torch.allclose(gx.cpu(), want, rtol=1e-5, atol=1e-5)
    assert torch.allclose(go.float().cpu(), out.float(), rtol=2 ** -7, atol=1e-5)


@pytest.mark.parametrize("T,d", [(1, 2048), (7, 1000), (600, 2048), (600, 4096), (600, 1001)])
def test_embedding_with_the_first_norm(T, d):
    ids = torch.randint(0, 50, (T,), dtype=I32, generator=torch.Generator().manual_seed(1)).cuda()
    table, w, w2 = rnd(50, d, seed=2).cuda(), rnd(d, dtype=F32, seed=3, scale=0.1).cuda(), rnd(d, dtype=F32, seed=4, scale=0.1).cuda()
    x, y = torch.empty(T, d, device="cuda"), torch.empty(T, d, device="cuda")
    h, want = torch.empty(T, d, dtype=B16, device="cuda"), torch.empty(T, d, dtype=B16, device="cuda")
    ops.embed_norm(ids, table, w, 1e-5, 1.0, x, w2=w2, out=h)
    ops.embed_norm(ids, table, w, 1e-5, 1.0, y)
    ops.rms_norm_rows(y, None, w2, 1e-5, 1.0, want)
    assert torch.equal(x, y)
    assert torch.allclose(h.float(), want.float(), rtol=2 ** -7, atol=1e-6)      # (the sums of squares in another order)


@pytest.mark.parametrize("T,H,P,rank,grank", [(1, 8, 256, 0, 0), (6, 3, 128, 0, 0), (16, 8, 64, 0, 0), (65, 2, 256, 0, 0),
                                              (1, 8, 256, 128, 128), (5, 3, 128, 32, 64), (9, 4, 64, 96, 160)])
def test_delta_token(T, H, P, rank, grank):
    N, d, taps, channel = 128, 2048 if H == 8 else 264, 4, rank > 0
    C = 2 * H * N + H * P
    wide = rnd(T, C + (rank + grank if channel else H * P) + 8, seed=1)
    z = wide[:, :C]
    x, gw = rnd(T, d, seed=2), rnd(H if channel else 2 * H, d, scale=d ** -0.5, seed=3)
    cw, conv = rnd(C, taps, scale=0.5, seed=4), rnd(2 * T + 1, taps - 1, C, seed=5)
    bias, alog = rnd(H * N if channel else H, dtype=F32, seed=6) - 2, rnd(H, dtype=F32, seed=7)
    state, w = rnd(2 * T + 1, H, N, P, dtype=F32, scale=0.3, seed=8), 1 + 0.1 * rnd(P, dtype=F32, seed=9)
    prev, save = slots_of(T, state.shape[0])
    gates = x.float() @ gw.float().t()
    if channel:
        a1, g1 = wide[:, C:C + rank], wide[:, C + rank:C + rank + grank]
        a2, g2 = rnd(H * N, rank, scale=rank ** -0.5, seed=10), rnd(H * P, grank, scale=grank ** -0.5, seed=11)
        dz, gate, low, gin = a1.float() @ a2.float().t(), (g1.float() @ g2.float().t()).to(B16), (a1, a2, g2), g1
    else:
        dz, gate, low = gates[:, H:], wide[:, C:C + H * P], None
        gin = gate
    st, cs = state.clone(), conv.clone()
    q, k, v, y = torch.empty(T, H, N), torch.empty(T, H, N), torch.empty(T, H, P, dtype=B16), torch.empty(T, H * P)
    reference.conv_silu_qkv(z, cw, cs, None, prev, T, H, N, H, P, N ** -0.5, 1e-6, q, k, v)
    reference.conv_state_update(z, cs, None, prev, save, T)
    reference.delta_rule(channel, q, k, v, dz, bias, alog, gates[:, :H], st, None, prev, save, T, y)
    want = torch.empty(T, H * P)
    reference.gated_group_norm(y, gate, w, 1e-5, P, False, want, channel)
    gz, gcs, gst, out = gpu(z), conv.cuda(), state.cuda(), torch.empty(T, H * P, dtype=B16, device="cuda")
    done = ops.delta_token(gz, cw.cuda(), gcs, prev.cuda(), save.cuda(), H, N, P, N ** -0.5, 1e-6, (x.cuda(), gw.cuda()),
                           tuple(map(gpu, low)) if low else None, bias.cuda(), alog.cuda(), gst, gpu(gin), w.cuda(), 1e-5, out)
    assert done
    assert torch.equal(gcs.cpu(), cs)
    # fp32 but for the roundings to bf16 of the values (an ulp where a sum's order turns one), the gate's factor and the result
    assert torch.allclose(gst.cpu(), st, rtol=1e-4, atol=2e-3)
    assert (gst.cpu() - st).norm() < 1e-4 * st.norm()
    err = (out.float().cpu() - want).norm() / want.norm()
    assert err < 2.5e-3, err            # (one rounding to bf16: 2^-9 / sqrt(3) of a value uniform in its binade, 1.7e-3 with the gate's)
    assert torch.allclose(out.float().cpu(), want, rtol=2 ** -6, atol=2e-2)


@pytest.mark.parametrize("T,d", [(1, 2048), (7, 1000), (300, 4096), (600, 1001)])
def test_embedding_with_the_first_layer_norm(T, d):
    ids = torch.randint(0, 50, (T,), dtype=I32, generator=torch.Generator().manual_seed(1)).cuda()
    src = torch.tensor([r % 3 - 1 for r in range(T)], dtype=I32).cuda()
    prev = torch.tensor([7, 9], dtype=I32).cuda()
    table, w, b = rnd(50, d, seed=2).cuda(), rnd(d, dtype=F32, seed=3).cuda(), rnd(d, dtype=F32, seed=4).cuda()
    x, y = torch.empty(T, d, device="cuda"), torch.empty(T, d, device="cuda")
    h, want = torch.empty(T, d, dtype=B16, device="cuda"), torch.empty(T, d, dtype=B16, device="cuda")
    ops.embed_layer_norm(ids, table, 8.0, x, w, b, 1e-6, h, src, prev)
    ops.embed_scale(ids, table, 8.0, y, src, prev)
    ops.residual_layer_norm(y, w=w, bias=b, eps=1e-6, out=want)
    assert torch.equal(x, y) and torch.equal(h, want)


@pytest.mark.parametrize("M", [1, 16, 40, 256, 257, 700])
def test_padded_weights_leave_the_same_columns(M):
    n, K = 3664, 2048
    x, w = rnd(M, K, seed=1).cuda(), rnd(n, K, scale=K ** -0.5, seed=2).cuda()
    wide = ops.pad_wide(w)
    assert wide.shape[0] == 3840 and torch.equal(wide[:n], w) and not wide[n:].any()
    got = ops.linear_wide(x, wide, wide[:n], lambda c: torch.empty(M, c, dtype=B16, device="cuda"))
    want = x.float() @ w.float().t()
    assert got.shape == (M, n)
    assert torch.allclose(got.float(), want, rtol=2 ** -7, atol=1e-3)


@pytest.mark.parametrize("M,H,N,K", [(1, 16, 512, 128), (16, 16, 128, 512), (9, 3, 100, 1024), (17, 16, 128, 512), (64, 5, 512, 128),
                                     (40, 2, 4096, 2048), (65, 4, 128, 512), (3, 2, 64, 24)])
def test_products_a_head(M, H, N, K):
    wide = rnd(M, H, K + 64, seed=1).cuda()
    x, w = wide[:, :, :K], rnd(H, N, K, scale=K ** -0.5, seed=2).cuda()
    out = torch.zeros(M, H, N + 64, dtype=B16, device="cuda")
    with torch.no_grad():
        ops.linear_heads(x, w.transpose(1, 2).contiguous(), w, out[:, :, :N])
    want = torch.einsum("mhk,hnk->mhn", x.float().cpu(), w.float().cpu())
    assert torch.allclose(out[:, :, :N].float().cpu(), want, rtol=2 ** -7, atol=1e-3)
    assert not out[:, :, N:].any()


@pytest.mark.parametrize("T", [1, 40])
def test_latent_prep_turns_the_queries(T):
    H, r, rot = 5, 512, 64
    z, q = rnd(T, r + rot + 8, seed=1).cuda()[:, :r + rot], rnd(T, H, 200, seed=2).cuda()
    pos, slot = torch.arange(T, dtype=I32).cuda() + 3, torch.arange(T, dtype=I32).cuda()
    rope, w = rnd(64, rot // 2, 2, dtype=F32, seed=3).cuda(), rnd(r, seed=4).cuda()
    got = []
    for side in range(2):
        plane, dst = torch.zeros(2, 64, r + rot, dtype=B16, device="cuda"), torch.zeros(T, H, r + rot, dtype=B16, device="cuda")
        if side:
            ops.latent_prep(z, 0, r, rot, None, w, 1e-6, pos, slot, rope, None, plane, q_rot=(q[:, :, 136:], dst[:, :, r:]))
        else:
            ops.latent_prep(z, 0, r, rot, None, w, 1e-6, pos, slot, rope, None, plane)
            ops.rope_pairs(q[:, :, 136:], dst[:, :, r:], pos, rope)
        got.append((plane, dst))
    assert all(torch.equal(a, b) for a, b in zip(*got))

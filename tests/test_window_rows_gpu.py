"""Single rows of the windowed attention's wave kernel in bf16, as decode steps call it, against attention in 64 bits."""
import math

import pytest
import torch

from symmetry_amd import ops

pytestmark = pytest.mark.gpu
BS = 64

# query heads, key / value heads, head size, rows, window: waves a workgroup and query heads a workgroup that take them
FORMS = [
    (16, 4, 128, 8, 1024),          # 16 waves
    (16, 4, 64, 8, 1024),
    (4, 4, 128, 3, 1 << 30),        # 16 waves, no window
    (6, 2, 128, 5, 1100),           # 16 waves, groups of 3 heads
    (16, 4, 128, 31, 600),          # 8 waves; one row short of four heads a workgroup
    (16, 4, 128, 32, 600), (16, 4, 64, 33, 1024),                           # 8 waves, 4 heads
    (16, 2, 128, 64, 600), (16, 2, 64, 65, 1024),                           # 8 waves, 8 heads
    (8, 4, 128, 32, 513), (8, 4, 64, 32, 600),                              # 8 waves, 2 heads
    (8, 8, 128, 17, 600), (4, 4, 64, 40, 520),                              # 8 waves, 1 head
    (16, 4, 128, 63, 512), (16, 4, 128, 64, 500), (32, 4, 64, 64, 129),     # 4 waves: 1, 4 and 8 heads
    (8, 4, 128, 255, 128), (8, 4, 128, 256, 100), (16, 2, 64, 512, 65), (2, 2, 128, 9, 1),      # one wave
    (16, 4, 96, 8, 1024),           # a head size that is scored lane by lane
]
EDGES = [0, 1, 62, 63, 64, 65, 127, 128, 129, 255, 300, 511, 512, 600, 703, 704, 1022, 1023, 1024, 1087, 1151, 1300, 1471]


@pytest.mark.parametrize("keep", [0, 70])
@pytest.mark.parametrize("H,G,D,T,window", FORMS)
def test_window_rows(gpu, H, G, D, T, window, keep):
    _check(H, G, D, T, window, keep, 0)


@pytest.mark.parametrize("H,G,D,T,window", [(16, 4, 128, 8, 1024), (16, 4, 64, 33, 600), (16, 2, 128, 64, 600)])
def test_keys_off_16_bytes(gpu, H, G, D, T, window):
    """A key cache 8 bytes off its 16: rows are scored lane by lane."""
    _check(H, G, D, T, window, 0, 4)


@pytest.mark.parametrize("H,G,D,T,window", [(16, 4, 128, 23, 1024), (16, 4, 64, 40, 600), (16, 2, 32, 23, 1), (6, 2, 96, 23, 33),
                                            (16, 1, 128, 30, 128), (5, 5, 112, 23, 97), (16, 4, 128, 300, 513)])
def test_window_ranges(gpu, H, G, D, T, window):
    """The key ranges of a window that ends, over every place of its first key in a step, and rows that end in their first range;
    whatever a row may not see is not finite.  The weights' three parts hold their 24 bits: the bounds are the wave kernel's."""
    _check(H, G, D, T, window, 0, 0, ranges=True)


def _check(H, G, D, T, window, keep, off, ranges=False):
    """Scores, weights and sums are fp32.  A score of D products of |q k| scale ~ 7 in all is within D 2^-24 7 < 2^-14 of the
    exact one and so a weight, the exponential's own 2^-22 aside; numerator and denominator both have them: 2^-13 of the sum of
    p |v|, and the result is rounded to bf16, at most 2^-8 of it (seven fraction bits).  Rows that p may not see, and the cache's first row, hold large values."""
    print("window_attn", H, G, D, T, window, keep, off, flush=True)
    g = torch.Generator(device="cuda").manual_seed(H * D + T)

    def rnd(*s):
        return torch.randn(*s, device="cuda", generator=g).bfloat16()

    short = window <= 128
    pos = [EDGES[(7 * i + T) % (11 if short else len(EDGES))] for i in range(T)]
    need = [p // BS + 1 for p in pos]
    mb = max(need) + 1 if short else 1536 // BS
    order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(T)).add_(1).tolist()
    bt = torch.zeros(T, mb, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        bt[i, :n] = torch.tensor(order[at:at + n])
        at += n
    bt = bt.cuda()
    shape = (at + 1, BS, G, D)
    k = torch.empty(math.prod(shape) + off, device="cuda", dtype=torch.bfloat16)[off:].view(shape)
    k.fill_(math.nan if ranges else 60.0)
    v = torch.full(shape, math.nan if ranges else -900.0, device="cuda", dtype=torch.bfloat16)
    rows = []
    for i, p in enumerate(pos):
        j0 = max(0, p - window + 1)
        j = torch.cat([torch.arange(min(keep, j0)), torch.arange(j0, p + 1)]).cuda()
        b, o = bt[i][j // BS].long(), j % BS
        k[b, o], v[b, o] = rnd(len(j), G, D), rnd(len(j), G, D)
        rows.append((b, o))
    q = rnd(T, H, D)
    out = torch.full((T + 1, H, D), 7.0, device="cuda", dtype=torch.bfloat16)
    i32 = dict(device="cuda", dtype=torch.int32)
    split = None
    if ranges:
        keys, parts = ops.window_attn_split(T, G, min(window + 31, mb * BS))
        split = (torch.empty(T, H, parts, D, device="cuda"), torch.empty(T, H, parts, 2, device="cuda"),
                 torch.zeros(T * G, **i32), keys)
    used = ops.window_attn(q, k, v, bt, torch.arange(T, **i32), torch.tensor(pos, **i32), window, D ** -0.5, None, out[:-1],
                           impl=1 if ranges else 0, keep_first=keep, split=split)
    assert used == (3 if ranges else 0) and bool((out[-1] == 7.0).all())
    assert split is None or not bool(split[2].any())
    for i, (b, o) in enumerate(rows):
        ks, vs = k[b, o].double(), v[b, o].double()
        p = torch.einsum("grd,cgd->grc", q[i].double().view(G, H // G, D), ks).mul_(D ** -0.5).softmax(-1)
        want, room = torch.einsum("grc,cgd->grd", p, vs), torch.einsum("grc,cgd->grd", p, vs.abs())
        err = (out[i].double().view(G, H // G, D) - want).abs()
        assert bool((err <= 2.0 ** -13 * room + 2.0 ** -8 * (want.abs() + 2.0 ** -13 * room)).all()), (i, pos[i], float(err.max()))


@pytest.mark.parametrize("H,G,D,block", [(4, 2, 128, 64), (3, 3, 64, 16), (4, 1, 32, 48), (2, 1, 80, 128)])
@pytest.mark.parametrize("window", [1, 31, 64, 65, 129, 300])
def test_window_prompts(gpu, H, G, D, block, window):
    """Prompt runs behind a window that ends: runs that start and end anywhere in a tile of 64 keys and in one of 128 rows, with and
    without cached rows, blocks that hold a tile and others.  Rows in front of a run's first window are not finite.  The weights are
    rounded to bf16 for their product: 2^-8 of the sum of p |v|, their scores' 2^-13 beside it, and the result's own rounding."""
    print("window prompts", H, G, D, block, window, flush=True)
    g = torch.Generator(device="cuda").manual_seed(D + window)
    runs = [(0, 1), (0, 200), (37, 130), (64, 64), (300, 65), (511, 3), (190, 129)]         # (cached, new)
    need = [-(-(c + n) // block) for c, n in runs]
    order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(D)).add_(1).tolist()
    bt = torch.zeros(len(runs), max(need), dtype=torch.int32)
    k = torch.full((sum(need) + 1, block, G, D), math.nan, device="cuda", dtype=torch.bfloat16)
    v = torch.full_like(k, math.nan)
    at, places = 0, []
    for i, (c, n) in enumerate(runs):
        bt[i, :need[i]] = torch.tensor(order[at:at + need[i]])
        at += need[i]
        j = torch.arange(max(0, c - window + 1), c + n)
        b, o = bt[i][j // block].long().cuda(), (j % block).cuda()
        k[b, o] = torch.randn(len(j), G, D, device="cuda", generator=g).bfloat16()
        v[b, o] = torch.randn(len(j), G, D, device="cuda", generator=g).bfloat16()
        places.append((j.cuda(), b, o))
    T, i32 = sum(n for _, n in runs), dict(device="cuda", dtype=torch.int32)
    q = torch.randn(T, H, D, device="cuda", generator=g).bfloat16()
    gate = torch.randn(T, H, device="cuda", generator=g).bfloat16()
    sink = torch.randn(H, device="cuda", generator=g)
    out = torch.full((T + 1, H, D), 7.0, device="cuda", dtype=torch.bfloat16)
    pos = torch.cat([torch.arange(c, c + n) for c, n in runs])
    rs = torch.repeat_interleave(torch.arange(len(runs)), torch.tensor([n for _, n in runs]))
    cu = [0]
    for _, n in runs:
        cu.append(cu[-1] + n)
    tiles = [(i, r) for i, (_, n) in enumerate(runs) for r in range(0, n, 64)]
    used = ops.window_attn(q, k, v, bt.cuda(), rs.to(**i32), pos.to(**i32), window, D ** -0.5, gate, out[:-1], torch.tensor(tiles, **i32),
                           torch.tensor(cu, **i32), sink=sink)
    assert used == 1 and bool((out[-1] == 7.0).all())
    for i, (c, n) in enumerate(runs):
        j, b, o = places[i]
        p = torch.arange(c, c + n, device="cuda")[:, None]
        hidden = (j[None] > p) | (j[None] <= p - window)
        qs = q[cu[i]:cu[i + 1]].double().view(n, G, H // G, D)
        s = torch.einsum("ngrd,cgd->ngrc", qs, k[b, o].double()).mul_(D ** -0.5).masked_fill_(hidden[:, None, None], -math.inf)
        s = torch.cat([s, sink.double().view(1, G, H // G, 1).expand(n, -1, -1, 1)], -1).softmax(-1)[..., :-1]
        f = gate[cu[i]:cu[i + 1]].double().sigmoid().view(n, G, H // G, 1)
        want = torch.einsum("ngrc,cgd->ngrd", s, v[b, o].double()) * f
        room = torch.einsum("ngrc,cgd->ngrd", s, v[b, o].double().abs()) * f
        err = (out[cu[i]:cu[i + 1]].double().view(n, G, H // G, D) - want).abs()
        assert bool((err <= (2.0 ** -8 + 2.0 ** -12) * room + 2.0 ** -8 * want.abs() + 1e-30).all()), (i, float(err.max()))

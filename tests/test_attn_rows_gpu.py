"""Prompt attention of few query rows behind cached contexts, on both sides of its dispatch line."""
import math

import pytest
import torch

from symmetry_amd import ops

pytestmark = pytest.mark.gpu
D = 128

# (query rows, context) of the sequences; 64-row tiles x kv heads = workgroups of the 64-row kernel
STEPS = [
    [(1, 1)],
    [(1, 33), (2, 2), (31, 40), (32, 257)],
    [(33, 33), (64, 700), (65, 300)],
    [(137, 1200)],
    [(3, 5000), (60, 60)],
    [(64 * 8, 800)],            # 64 workgroups at 8 kv heads: the last of the row kernel
    [(64 * 8 + 1, 800)],        # one tile more: the 64-row kernel
]


@pytest.mark.parametrize("BS", [32, 64, 256])
@pytest.mark.parametrize("heads", [(8, 1), (32, 8), (16, 4)])
@pytest.mark.parametrize("step", range(len(STEPS)))
def test_prompt_rows(step, heads, BS):
    """Against 64-bit attention.  P is rounded to bf16 (2^-8 of a term at most, not all one way), the result once more; the rest is
    fp32 (scores of |q| |k| ~ 30 to 2^-20, the exponential to 2^-20): 2^-8 (sum p |v| + |o|) bounds it.  Places past a
    context hold large values, which no row may see."""
    H, Hkv = heads
    runs = STEPS[step]
    print("attn_prefill", runs, heads, BS, flush=True)
    torch.manual_seed(step)
    mb = max(-(-c // BS) for _, c in runs) + 1
    bt = (torch.randperm(len(runs) * mb) + 1).view(len(runs), mb).int()
    k = torch.full((len(runs) * mb + 1, Hkv, BS, D), 60.0, dtype=torch.bfloat16)
    v = torch.full((len(runs) * mb + 1, Hkv, D, BS), -900.0, dtype=torch.bfloat16)
    ks, vs = [], []
    for s, (_, c) in enumerate(runs):
        a, b = torch.randn(Hkv, c, D).bfloat16(), torch.randn(Hkv, c, D).bfloat16()
        for i in range(0, c, BS):
            n = min(BS, c - i)
            k[bt[s, i // BS], :, :n], v[bt[s, i // BS], :, :, :n] = a[:, i:i + n], b[:, i:i + n].transpose(1, 2)
        ks.append(a.double()), vs.append(b.double())
    lens = torch.tensor([n for n, _ in runs])
    cu = torch.tensor([0] + lens.cumsum(0).tolist()).int()
    tiles = torch.tensor([(s, r) for s, (n, _) in enumerate(runs) for r in range(0, n, 64)]).int()
    q = torch.randn(int(lens.sum()), H, D).bfloat16()
    out = torch.full((q.shape[0] + 1, H, D), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.attn_prefill(q.cuda(), k.cuda(), v.cuda(), bt.cuda(), torch.tensor([c for _, c in runs]).int().cuda(), cu.cuda(),
                     tiles.cuda(), out[:-1], D ** -0.5)
    got = out.cpu().double()
    assert (got[-1] == 7.0).all()
    for s, (n, c) in enumerate(runs):
        rep = H // Hkv
        qs = q[cu[s]:cu[s + 1]].double().transpose(0, 1)
        sc = qs @ ks[s].repeat_interleave(rep, 0).transpose(1, 2) * D ** -0.5
        sc = sc.masked_fill((torch.arange(c)[None] > (c - n + torch.arange(n))[:, None])[None], -math.inf)
        p, vv = sc.softmax(-1), vs[s].repeat_interleave(rep, 0)
        want, room = (p @ vv).transpose(0, 1), (p @ vv.abs()).transpose(0, 1)
        err = (got[cu[s]:cu[s + 1]] - want).abs()
        assert (err <= 2.0 ** -8 * (room + want.abs())).all(), (s, float(err.max()))

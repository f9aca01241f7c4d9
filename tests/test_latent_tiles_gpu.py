"""Latent attention of 512 + 64 entries over cache blocks of whole tiles: prompt tiles, single rows and their partitions against the
one-wave kernel and a plain softmax; the merge of many and of few partitions."""
import pytest
import torch

from symmetry_amd import ops

pytestmark = pytest.mark.gpu


def setup(H, bs, runs, seed):
    g = torch.Generator().manual_seed(seed)
    Dk = 576
    per = [-(-(p0 + n) // bs) for p0, n in runs]
    cache = torch.randn(sum(per) + 1, bs, Dk, generator=g).bfloat16()
    order, at = torch.randperm(sum(per), generator=g).int() + 1, 0
    table = torch.zeros(len(runs), max(per), dtype=torch.int32)
    for i, k in enumerate(per):
        table[i, :k] = order[at:at + k]
        # what lies behind a sequence's last key is another's: large numbers there are seen if a tile takes them along
        end = sum(runs[i]) - (k - 1) * bs
        cache[order[at + k - 1], end:] = float("nan")
        at += k
    pos = torch.cat([torch.arange(p0, p0 + n) for p0, n in runs]).int()
    seq = torch.cat([torch.full((n,), i) for i, (_, n) in enumerate(runs)]).int()
    q = (torch.randn(pos.numel(), H, Dk, generator=g) * 0.5).bfloat16()
    sink, gate = torch.randn(H, generator=g), torch.randn(pos.numel(), H, generator=g).bfloat16()
    return cache, table, pos, seq, q, sink, gate


def want_of(cache, table, pos, seq, q, sink, gate, scale):
    out = torch.zeros(q.shape[0], q.shape[1], 512, device="cuda")
    for t in range(q.shape[0]):
        rows = cache[table[seq[t]].long()].reshape(-1, 576)[:int(pos[t]) + 1].float()
        s = torch.cat([q[t].float() @ rows.t() * scale, sink[:, None]], 1)
        out[t] = torch.softmax(s, 1)[:, :-1] @ rows[:, :512] * torch.sigmoid(gate[t].float())[:, None]
    return out


def close(got, want):
    # weights and result are rounded to bf16: 2^-9 of a value uniform in its binade each, 1.1e-3 of the norm; four times that
    err = float((got.float() - want).norm() / want.norm())
    assert err < 5e-3, err
    assert float((got.float() - want).abs().max()) < 3e-2


@pytest.mark.parametrize("H,bs", [(16, 64), (2, 32), (40, 128), (3, 64), (5, 256)])
def test_prompt_tiles_and_rows(H, bs):
    runs = [(300, 130), (0, 70), (517, 1), (64, 64), (0, 31), (0, 33)]
    cache, table, pos, seq, q, sink, gate = (t.cuda() for t in setup(H, bs, runs, H))
    cu = torch.tensor([0] + list(torch.tensor([n for _, n in runs]).cumsum(0)), dtype=torch.int32).cuda()
    tiles = torch.tensor([(i, o) for i, (_, n) in enumerate(runs) for o in range(0, n, 64)] + [(0, 1 << 24)], dtype=torch.int32).cuda()
    want = want_of(cache, table, pos, seq, q, sink, gate, 0.2)
    for kw in (dict(tiles=tiles, cu_q=cu), {}):
        out = torch.zeros(q.shape[0], H, 512, dtype=torch.bfloat16, device="cuda")
        assert ops.latent_attn(q, cache, table, seq, pos, 0.2, 512, out, impl=0, sink=sink, gate=gate, **kw) == 0
        close(out, want)


@pytest.mark.parametrize("H,bs,parts", [(16, 64, 2), (16, 64, 5), (16, 64, 32), (16, 64, 40), (40, 32, 3), (3, 128, 7)])
def test_rows_in_partitions(H, bs, parts):
    runs = [(n - 1, 1) for n in (1, 31, 32, 33, 64, 127, 128, 129, 300, 700, 1280)]
    cache, table, pos, seq, q, sink, gate = (t.cuda() for t in setup(H, bs, runs, H + parts))
    want = want_of(cache, table, pos, seq, q, sink, gate, 0.2)
    T = q.shape[0]
    po, ml = torch.full((T, H, parts, 512), float("nan"), device="cuda"), torch.full((T, H, parts, 2), float("nan"), device="cuda")
    out = torch.zeros(T, H, 512, dtype=torch.bfloat16, device="cuda")
    assert ops.latent_attn(q, cache, table, seq, pos, 0.2, 512, out, po, ml, impl=0, sink=sink, gate=gate) == 0
    close(out, want)

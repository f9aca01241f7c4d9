"""Decode attention within the rounding of every element: contexts around the edges of groups, steps and partitions, and batches
whose contexts differ widely, on both sides of the rules that cut them into partitions."""
import pytest
import torch

from symmetry_amd import ops

pytestmark = pytest.mark.gpu
D = 128


class _Batch:
    """One query row per context over a paged cache of scattered blocks; places past a context hold large values, which no row
    may see."""

    def __init__(self, ctx, heads, BS, width=None, seed=0):
        print("attn_decode", len(ctx), max(ctx), heads, BS, flush=True)
        self.H, self.G = heads
        self.BS, S = BS, len(ctx)
        g = torch.Generator(device="cuda").manual_seed(seed)

        def rnd(*s):
            return torch.randn(*s, device="cuda", generator=g).bfloat16()

        need = [-(-c // BS) for c in ctx]
        self.width = width or max(need) + 1
        order = torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed)) + 1
        bt = torch.zeros(S, self.width, dtype=torch.int32)
        at = 0
        for s, n in enumerate(need):
            bt[s, :n] = order[at:at + n]
            at += n
        self.tables, self.bt = bt, bt.cuda()
        self.k, self.v = rnd(at + 1, self.G, BS, D), rnd(at + 1, self.G, D, BS)
        self.q = rnd(S, self.H, D)
        self.k0, self.v0 = self.k.clone(), self.v.clone()
        self.ctx = torch.zeros(S, dtype=torch.int32, device="cuda")
        parts = -(-self.width * BS // ops.ATTN_DECODE_PART)
        self.tmp_o = torch.empty(S, self.H, parts, D, device="cuda")
        self.tmp_ml = torch.empty(S, self.H, parts, 2, device="cuda")
        self.counters = torch.zeros(S * self.G, dtype=torch.int32, device="cuda")
        self.out = torch.empty(S + 1, self.H, D, dtype=torch.bfloat16, device="cuda")
        self.cut(ctx)

    def cut(self, ctx):
        """Other contexts, no longer than the first ones."""
        self.lens = ctx
        self.ctx.copy_(torch.tensor(ctx, dtype=torch.int32))
        self.k.copy_(self.k0)
        self.v.copy_(self.v0)
        self.k[0], self.v[0] = 60.0, -900.0
        for s, c in enumerate(ctx):
            for i in range(c // self.BS, int((self.tables[s] > 0).sum())):
                b = int(self.tables[s, i])
                at = max(0, c - i * self.BS)
                self.k[b, :, at:], self.v[b, :, :, at:] = 60.0, -900.0
        self.out.fill_(7.0)
        self.tmp_o.fill_(float("nan"))
        self.tmp_ml.fill_(float("nan"))

    def run(self):
        ops.attn_decode(self.q, self.k, self.v, self.bt, self.ctx, self.out[:-1], self.tmp_o, self.tmp_ml, self.counters, D ** -0.5)

    def check(self):
        """Against 64-bit attention.  P is rounded to bf16 (2^-8 of a term at most, not all one way), the result once more; the rest is
        fp32 (scores of |q| |k| ~ 30 to 2^-20, the exponential to 2^-20): 2^-8 (sum p |v| + |o|) bounds it."""
        assert not self.counters.any() and bool((self.out[-1] == 7.0).all())
        rep = self.H // self.G
        for s, c in enumerate(self.lens):
            if not c:
                assert bool((self.out[s] == 7.0).all())       # (an empty context writes nothing)
                continue
            b = self.bt[s, :-(-c // self.BS)].long()
            k = self.k0[b].transpose(1, 2).reshape(-1, self.G, D)[:c].double()
            v = self.v0[b].permute(0, 3, 1, 2).reshape(-1, self.G, D)[:c].double()
            p = torch.einsum("grd,cgd->grc", self.q[s].double().view(self.G, rep, D), k).mul_(D ** -0.5).softmax(-1)
            want, room = torch.einsum("grc,cgd->grd", p, v), torch.einsum("grc,cgd->grd", p, v.abs())
            err = (self.out[s].double().view(self.G, rep, D) - want).abs()
            assert bool((err <= 2.0 ** -8 * (room + want.abs())).all()), (s, c, float(err.max()))


EDGES = [1, 17, 31, 32, 33, 64, 200, 255, 256, 257, 511, 512, 513, 700, 767, 769, 1000, 1025, 2049, 2300, 4100, 4700]


def _edges(n):
    return [EDGES[(5 * i + n) % len(EDGES)] for i in range(n)]


@pytest.mark.parametrize("ctx,heads", [
    (EDGES, (32, 8)), (EDGES, (64, 8)), (EDGES, (8, 1)), (EDGES, (16, 16)),
    (_edges(65), (32, 8)),                                  # units past a third of the chip: one partition of several steps
    (_edges(40), (32, 8)), (_edges(30), (32, 8)),           # two and three partitions, steps that do not divide by them
    (_edges(7), (16, 16)), (_edges(3), (64, 8)),
    (EDGES, (32, 2)), (_edges(70), (60, 5)), (_edges(6), (27, 3)), (_edges(40), (20, 4)), (_edges(9), (6, 2)),   # 16, 12, 9, 5 and 3 queries a head
    ([4700], (32, 4)), ([4673], (32, 4)), ([33], (8, 2)),   # one sequence: a partition for every step
])
@pytest.mark.parametrize("BS", [32, 64])
def test_contexts_around_the_edges(gpu, ctx, heads, BS):
    b = _Batch(ctx, heads, BS)
    b.run()
    b.check()
    first = b.out.clone()
    b.run()                                                 # (finds the counters re-armed)
    assert torch.equal(first, b.out)


def _at(n, short, *longs):
    """n contexts around ``short``, the long ones spread over the batch."""
    ctx = [max(0, short - 40 + 7 * (i % 12)) for i in range(n)]
    for i, c in enumerate(longs):
        ctx[(i + 1) * n // (len(longs) + 1)] = c
    return ctx


@pytest.mark.parametrize("ctx,heads", [
    ([7000] + _at(60, 300), (32, 8)),                       # the long one first, last, within
    (_at(60, 300) + [7000], (32, 8)),
    (_at(65, 200, 2000), (32, 8)),                          # one more than a wave's lanes
    (_at(130, 100, 5000, 4097, 30, 4096), (16, 4)),
    (_at(300, 60, 3500, 0, 3333), (8, 1)),                  # lengths past four a lane, one kv head, an empty context
    (_at(40, 250, 6000, 6000, 6000, 6000), (12, 12)),       # a number of heads that is no power of two; one query column
    (_at(70, 30, 4000), (64, 4)),                           # 16 query columns
    ([0, 3000], (16, 16)), ([1] * 63 + [1537], (8, 8)), ([0] * 64 + [1536] * 2, (16, 8)),     # either side of six steps
    ([6000, 6100, 5900] * 22, (8, 8)),                      # long ones throughout: nobody is above the others
])
@pytest.mark.parametrize("BS", [32, 64])
def test_contexts_of_very_different_lengths(gpu, ctx, heads, BS):
    b = _Batch(ctx, heads, BS)
    for _ in range(2):                                      # (the second call finds the counters re-armed)
        b.run()
        b.check()
        first = b.out.clone()
    b.run()
    assert torch.equal(first, b.out)


def test_a_long_context_is_cut_by_its_share(gpu):
    """60 short contexts and one of 8000 tokens: 152 steps of 256 tokens, shares of 3, so the long one's 32 steps are 11
    partitions, each of which leaves its partial result, and the short ones (one partition) leave none."""
    ctx = _at(61, 300, 8000)
    b = _Batch(ctx, (32, 8), 64, width=128)
    b.run()
    b.check()
    steps = sum(-(-c // 256) for c in ctx)
    want = -(-32 // -(-steps // 64))
    wrote = b.tmp_ml[..., 0].isfinite().sum(-1)             # [S, H]
    assert want >= 10
    for s, c in enumerate(ctx):
        assert bool((wrote[s] == (want if c == 8000 else 0)).all()), (s, c, wrote[s].tolist())


def test_replays_follow_the_lengths(gpu):
    """The grid of a captured step knows the tables' width only: lengths change between replays."""
    n = 66
    b = _Batch([3000] * n, (16, 8), 64, width=128)
    b.run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        b.run()
    for ctx in ([300] * n, _at(n, 60, 3000), [3000] * n, _at(n, 260, 2900, 1, 3000), [0] * (n - 1) + [2999]):
        b.cut(ctx)
        for _ in range(2):
            graph.replay()
        torch.cuda.synchronize()
        b.check()

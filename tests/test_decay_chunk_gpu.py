"""The chunked recurrence (csrc/kernels/decay_chunk.hip) against the recurrence in 64 bits, and beside the token-by-token
kernel (the same values as fp32 operands take that one).

Bound: every term of an output passes a handful of fp32 roundings (2^-24 each) and at most a run's chunks of decays and sums,
whose errors add up like a random walk: sqrt(200) 2^-24 = 8e-7 of the result's 2-norm at the longest run here; 2e-6 is asked
for.  The largest single error is asked to stay under 4e-6 of the largest output."""
import pytest
import torch

from symmetry_amd import ops

pytestmark = pytest.mark.gpu


def _walk(q, k, v, a, b, S0, lens, skip):
    o, ends, r = torch.zeros_like(v), [], 0
    for i, n in enumerate(lens):
        S = S0[i].clone()
        for t in range(r, r + n):
            S = a[t][:, :, None] * S + (b[t][:, None] * k[t])[:, :, None] * v[t][:, None, :]
            o[t] = (S * q[t][:, :, None]).sum(1) + skip[:, None] * v[t]
        ends.append(S)
        r += n
    return o, torch.stack(ends)


SHAPES = [(3, 128, 80, 3, [33, 64, 5, 97, 1, 32]), (4, 64, 64, 2, [100, 31]), (2, 24, 16, 1, [40, 41]), (2, 8, 70, 2, [8]),
          (2, 72, 70, 2, [200]), (2, 32, 130, 1, [63, 65])]


class _Case:
    """Runs of the given lengths whose q, k and v are column ranges of one projection; every third run is a sequence's first."""

    def __init__(self, gpu, mode, H, N, P, G, lens, tau=16.0):
        g = torch.Generator(device=gpu).manual_seed(H * N + P)
        T, R = sum(lens), len(lens)

        def rnd(*s):
            return torch.randn(*s, device=gpu, generator=g)

        z = rnd(T, 2 * G * N + H * P).bfloat16()
        self.q, self.k, self.v = z[:, :G * N], z[:, G * N:2 * G * N], z[:, 2 * G * N:]
        cols = H * N if mode == ops.DECAY_CHANNEL_GATE else H
        self.dz, self.db = rnd(T, cols).bfloat16(), rnd(cols) + (3.0 if mode == ops.DECAY_CHANNEL_GATE else -2.0)
        self.par = tau if mode == ops.DECAY_CHANNEL_GATE else torch.log(0.05 + 0.5 * torch.rand(H, device=gpu, generator=g))
        self.skip, self.scale = rnd(H), 0.37
        self.state = rnd(2 * R, H, N, P)
        self.fresh = [i for i in range(R) if i % 3 == 2]
        prev, save = [], []
        for i, n in enumerate(lens):
            prev += [-1 if i in self.fresh else -(i + 2)] + [0] * (n - 1)
            save += [-1] * (n - 1) + [R + i]
        i32 = dict(device=gpu, dtype=torch.int32)
        self.prev, self.save = torch.tensor(prev, **i32), torch.tensor(save, **i32)
        self.cu = torch.tensor([sum(lens[:i]) for i in range(R + 1)], **i32)
        self.tiles = torch.tensor([(i, r) for i, n in enumerate(lens) for r in range(0, n, 64)] + [(0, 1 << 24)], **i32)
        self.ws = torch.full((T, H, ops.decay_ws_cols(N)), float("nan"), device=gpu)
        self.mode, self.H, self.N, self.P, self.G, self.lens, self.T, self.R = mode, H, N, P, G, lens, T, R

    def exact(self):
        H, N, P, G, T = self.H, self.N, self.P, self.G, self.T
        head = torch.arange(H, device=self.q.device) // (H // G)
        y = self.dz.double().view(T, H, -1) + self.db.double().view(H, -1)
        if self.mode == ops.DECAY_CHANNEL_GATE:
            a, b = torch.exp(torch.nn.functional.logsigmoid(y) / self.par), torch.ones_like(y[..., 0])
        else:
            b = torch.nn.functional.softplus(y[..., 0], threshold=1e9)
            a = torch.exp(-torch.exp(self.par.double()) * b)[:, :, None].expand(T, H, N)
        S0 = self.state[:self.R].double().clone()
        S0[self.fresh] = 0
        return _walk(self.q.double().view(T, G, N)[:, head] * self.scale, self.k.double().view(T, G, N)[:, head],
                     self.v.double().reshape(T, H, P), a, b, S0, self.lens, self.skip.double())

    def run(self, chunked):
        """-> (out [T, H, P], final states)"""
        x = [t if chunked else t.float() for t in (self.q, self.k, self.v, self.dz)]
        out = torch.empty(self.T, self.H * self.P, device=self.q.device)
        ops.decay_scan(self.mode, *x, self.db, self.par, self.skip, self.scale, self.H, self.N, self.P, self.H // self.G, self.state,
                       self.cu, self.prev, self.save, self.R, out, tiles=self.tiles, ws=self.ws)
        return out.view(self.T, self.H, self.P), self.state[self.R:]

    def check(self):
        want, ends = self.exact()
        for chunked in (True, False):
            out, state = self.run(chunked)
            d = out.double() - want
            assert float(d.norm() / want.norm()) <= 2e-6, chunked
            assert float(d.abs().max() / want.abs().max()) <= 4e-6, chunked
            assert float((state.double() - ends).norm() / ends.norm()) <= 2e-6, chunked


@pytest.mark.parametrize("mode", [ops.DECAY_CHANNEL_GATE, ops.DECAY_STEP_SIZE])
@pytest.mark.parametrize("shift", [0.0, -40.0, 15.0])       # decays of a few hundred tokens, of one, of none
@pytest.mark.parametrize("H,N,P,G,lens", SHAPES)
def test_decay_chunks(gpu, mode, shift, H, N, P, G, lens):
    c = _Case(gpu, mode, H, N, P, G, lens)
    c.dz = (c.dz.float() + shift).bfloat16()
    c.check()


@pytest.mark.parametrize("mode,tau,share,hard", [
    (ops.DECAY_CHANNEL_GATE, 16.0, 0.1, -40.0), (ops.DECAY_CHANNEL_GATE, 16.0, 0.25, -100.0),
    (ops.DECAY_CHANNEL_GATE, 16.0, 0.1, -400.0), (ops.DECAY_CHANNEL_GATE, 1.0, 0.1, -40.0),
    (ops.DECAY_CHANNEL_GATE, 1.0, 0.1, -100.0), (ops.DECAY_STEP_SIZE, 0.0, 0.1, 100.0)])
@pytest.mark.parametrize("H,N,P,G,lens", SHAPES)
def test_tokens_that_forget_hard_among_others(gpu, mode, tau, share, hard, H, N, P, G, lens):
    """A few tokens of a chunk forget almost everything, so the chunk's running decay grows to hundreds, and the tokens behind
    them remember: their mutual decays are small differences of large sums.  The same bounds."""
    c = _Case(gpu, mode, H, N, P, G, lens, tau)
    pick = torch.rand(c.dz.shape, device=gpu, generator=torch.Generator(device=gpu).manual_seed(7)) < share
    c.dz = torch.where(pick, torch.full_like(c.dz, hard), c.dz)
    c.check()


@pytest.mark.parametrize("mode", [ops.DECAY_CHANNEL_GATE, ops.DECAY_STEP_SIZE])
@pytest.mark.parametrize("H,N,P,G,lens", SHAPES)
def test_decays_of_exactly_zero(gpu, mode, H, N, P, G, lens):
    """A gate of -inf, from the projection or as a channel's bias (or a head's infinite rate), forgets all there was: 0 x S + k v."""
    c = _Case(gpu, mode, H, N, P, G, lens)
    if mode == ops.DECAY_CHANNEL_GATE:
        pick = torch.rand(c.dz.shape, device=gpu, generator=torch.Generator(device=gpu).manual_seed(9)) < 0.1
        c.dz = torch.where(pick, torch.full_like(c.dz, -float("inf")), c.dz)
        c.db[::5] = -float("inf")
    else:
        c.par[0] = 100.0
    c.check()


@pytest.mark.parametrize("mode", [ops.DECAY_CHANNEL_GATE, ops.DECAY_STEP_SIZE])
@pytest.mark.parametrize("what,value", [("v", float("inf")), ("v", float("nan")), ("k", -float("inf")), ("q", float("nan")),
                                        ("q", float("inf")), ("dz", float("nan"))])
@pytest.mark.parametrize("H,N,P,G,lens", [(3, 128, 80, 3, [33, 64, 5, 97, 1, 32]), (4, 64, 64, 2, [100, 31]), (2, 24, 16, 1, [40, 41])])
def test_values_that_are_not_finite(gpu, mode, what, value, H, N, P, G, lens):
    """They reach what the token-by-token kernel lets them reach, and nothing else: no earlier token, no other column."""
    c = _Case(gpu, mode, H, N, P, G, lens)
    clean, state = (t.clone() for t in c.run(True))
    x = getattr(c, what).clone()
    for r in (5, 21, 60):                                     # (a chunk's first tile, its second, another chunk)
        x[r, (7 * r) % x.shape[1]] = value
    setattr(c, what, x)
    walk, walk_state = (t.clone() for t in c.run(False))
    out, ends = c.run(True)
    assert 0 < int((~walk.isfinite()).sum()) < walk.numel()
    assert torch.equal(out.isfinite(), walk.isfinite()) and torch.equal(ends.isfinite(), walk_state.isfinite())
    assert torch.equal(out[out.isfinite()], clean[out.isfinite()]) and torch.equal(ends[ends.isfinite()], state[ends.isfinite()])


@pytest.mark.parametrize("mode", [ops.DECAY_CHANNEL_GATE, ops.DECAY_STEP_SIZE])
@pytest.mark.parametrize("value", [3.4e38, -3.4e38])
def test_states_past_the_largest_bf16(gpu, mode, value):
    """A state between bf16's largest and fp32's is a number like others: the bounds relative to the columns that it scales."""
    c = _Case(gpu, mode, 4, 64, 64, 2, [100, 31])
    c.state[0, 1, 5, 3] = value
    c.k[:, 5] = 0                              # (nothing is added to it, and what is read of it stays below fp32's largest)
    c.q[:, 5] *= 0.125
    want, ends = c.exact()
    out, state = c.run(True)
    for got, w in ((out.double(), want), (state.double(), ends)):
        assert bool(((got - w).abs() <= 4e-6 * w.abs().amax(0 if w is want else 2, keepdim=True)).all())


@pytest.mark.parametrize("form", ["odd channels", "odd stride", "unaligned", "no scratch", "short runs", "wide"])
def test_forms_that_walk_token_by_token(gpu, form):
    """What the chunked form does not take gives the same recurrence (channel gate, one run from zero)."""
    g = torch.Generator(device=gpu).manual_seed(11)
    H, P, T = 2, 48, 40
    N = {"odd channels": 12, "wide": 136}.get(form, 16)
    lens = [4] * 10 if form == "short runs" else [T]

    def rnd(*s):
        return torch.randn(*s, device=gpu, generator=g)

    pad = 1 if form in ("odd stride", "unaligned") else 0
    z = rnd(T, 2 * H * N + (3 if form == "odd stride" else 8)).bfloat16()
    q, k = z[:, pad:pad + H * N], z[:, pad + H * N:pad + 2 * H * N]
    v, dz, db = rnd(T, H * P).bfloat16(), rnd(T, H * N).bfloat16(), rnd(H * N) + 2
    state = torch.zeros(len(lens), H, N, P, device=gpu)
    i32 = dict(device=gpu, dtype=torch.int32)
    cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], **i32)
    prev = torch.tensor([-1 if r in cu.tolist() else r - 1 for r in range(T)], **i32)
    save = torch.full((T,), -1, **i32)
    tiles = torch.tensor([(i, 0) for i in range(len(lens))], **i32)
    ws = None if form == "no scratch" else torch.empty(T, H, ops.decay_ws_cols(N), device=gpu)
    out = torch.empty(T, H * P, device=gpu)
    ops.decay_scan(ops.DECAY_CHANNEL_GATE, q, k, v, dz, db, 16.0, None, 0.25, H, N, P, 1, state, cu, prev, save, len(lens), out,
                   tiles=tiles, ws=ws)
    a = torch.exp(torch.nn.functional.logsigmoid((dz.double() + db.double()).view(T, H, N)) / 16)
    want, _ = _walk(q.double().reshape(T, H, N) * 0.25, k.double().reshape(T, H, N), v.double().view(T, H, P), a,
                    torch.ones(T, H, device=gpu).double(), torch.zeros(len(lens), H, N, P, device=gpu).double(), lens,
                    torch.zeros(H, device=gpu).double())
    assert float((out.double() - want.reshape(T, -1)).norm() / want.norm()) <= 2e-6


@pytest.mark.parametrize("mode", [ops.DECAY_CHANNEL_GATE, ops.DECAY_STEP_SIZE])
@pytest.mark.parametrize("step", [0, 16, 40])
def test_value_rows_that_overlap(gpu, mode, step):
    """Rows closer to each other than they are long, or all one row: what lies behind the last token is no token's, an infinity
    there reaches only the columns of the rows that hold it.  40 tokens end in the middle of a chunk."""
    H, N, P, T = 1, 16, 48, 40
    c = _Case(gpu, mode, H, N, P, 1, [T])
    flat = torch.randn(T * 48 + P, device=gpu).bfloat16()
    if step:
        flat[(T - 1) * step + P - 1] = float("inf")          # the last column of the last token alone
    c.v = flat.as_strided((T, P), (step, 1))
    out, state = c.run(True)
    want, end = out.clone(), state.clone()
    c.v = c.v.float().contiguous()
    c.q, c.k, c.dz = c.q.float(), c.k.float(), c.dz.float()
    out, state = c.run(False)
    assert torch.equal(want.isfinite(), out.isfinite()) and torch.equal(end.isfinite(), state.isfinite())
    assert bool(state[..., :P - 1].isfinite().all()) and bool(out[:-1].isfinite().all())
    for a, b in ((want, out), (end, state)):
        ok = b.isfinite()
        assert float((a[ok] - b[ok]).norm() / b[ok].norm()) <= 4e-6       # (both within 2e-6 of the exact ones)


@pytest.mark.parametrize("H,N,P,G,lens", SHAPES)
def test_scratch_of_its_own_or_the_callers(gpu, H, N, P, G, lens):
    """A scratch too small for the chunks' blocks is taken and stands for one of the walk's own: the same numbers."""
    c = _Case(gpu, ops.DECAY_CHANNEL_GATE, H, N, P, G, lens)
    start = c.state.clone()
    out, state = (t.clone() for t in c.run(True))
    c.state.copy_(start)
    c.ws = torch.full((ops.decay_scratch(c.mode, c.T, c.R, H, N, P),), float("nan"), device=gpu)
    assert c.ws.numel() >= c.T * H * ops.decay_ws_cols(N)
    for got, want in zip(c.run(True), (out, state)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("mode", [ops.DECAY_CHANNEL_GATE, ops.DECAY_STEP_SIZE])
@pytest.mark.parametrize("shift", [0.0, -40.0])
@pytest.mark.parametrize("H,N,P,G,lens", [(3, 128, 80, 3, [700]), (4, 64, 64, 2, [33, 1, 1000]), (2, 24, 16, 1, [257]), (8, 128, 256, 8, [1000, 64]),
                                          (20, 128, 64, 4, [800, 31, 500])])
def test_few_long_runs(gpu, mode, shift, H, N, P, G, lens):
    """Runs cut into segments: ends of segments inside and at the end of runs, runs shorter than one, a state saved where it came from.
    The bounds of whole runs: a segment's state passes the same roundings, one more for every segment."""
    c = _Case(gpu, mode, H, N, P, G, lens)
    c.dz = (c.dz.float() + shift).bfloat16()
    c.ws = torch.full((ops.decay_scratch(mode, c.T, c.R, H, N, P),), float("nan"), device=gpu)
    c.tiles = c.tiles if mode == ops.DECAY_CHANNEL_GATE else None
    assert ops.decay_scratch(ops.DECAY_STEP_SIZE, c.T, c.R, H, N, P) > 0      # (segments' states: they are cut)
    c.check()
    for i in range(c.R):      # run i's state: from slot i + .. into the same slot
        if i not in c.fresh:
            c.save[c.save == c.R + i] = i
    want, ends = c.exact()
    out, _ = c.run(True)
    assert float((out.double() - want).norm() / want.norm()) <= 2e-6
    for i in range(c.R):
        if i not in c.fresh:
            assert float((c.state[i].double() - ends[i]).norm() / ends[i].norm()) <= 2e-6

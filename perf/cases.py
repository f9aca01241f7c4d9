"""What is timed: engine steps of the model classes, as the serving engine gives them to ``model.forward``.

A case is one step of a stack of four layers with the layer shapes of the family benchmark (bench/families.py): a decode
step (one new token for each of ``seqs`` sequences whose contexts average ``context`` tokens, cache and carried states in
place) or a prompt step (``tokens`` new tokens split over ``seqs`` sequences that have about ``context`` tokens cached).
The step's metadata is on the device, as the model runner leaves it there.  As in serving, decode steps and the short
prompt steps of dense models replay a hipGraph that was captured beforehand; other prompt steps run eagerly.

Stacks: ``llama-w4096`` / ``llama-w2048`` (grouped-head attention, SwiGLU), ``mixtral-w2048`` (routed experts),
``lemunex-w2048`` (windowed attention beside gated linear attention, state-space layers), ``beletar-w2048`` (gated delta
rule, latent attention).  All in bfloat16, the dtype they are served in.
"""
from __future__ import annotations

import math
import random
import zlib

import torch

BLOCK = 64                               # tokens of a cache block (the engine's default)
MAX_POSITION = 8192
CONTEXT_BUCKETS = (512, 2048, 8192)      # block tables of decode steps are as wide as one of these (as in the engine)
GRAPH_PROMPT_TOKENS = 256                # prompt steps of dense models up to this size replay a hipGraph
VOCAB = 32768
LAYERS = 4
SPECIAL = dict(max_position=MAX_POSITION, bos_token_id=32000, eos_token_ids=(32001, 32002))
YARN = (4.0, 4096.0, 32.0, 1.0)          # factor, original positions, fast, slow

LLAMA = {
    "llama-w4096": dict(d=4096, ff=14336, heads=32, kv=8, experts=0, top=0),
    "llama-w2048": dict(d=2048, ff=8192, heads=16, kv=4, experts=0, top=0),
    "mixtral-w2048": dict(d=2048, ff=1536, heads=16, kv=4, experts=16, top=4),
}
LEMUNEX = dict(d=2048, ff=8192, pattern="pmmp", heads=16, kv=4, dim=128, window=1024, gla_heads=8, gla_dim=128, gla_vdim=256,
               rank=16, ssm_heads=64, ssm_vdim=64, state=128, conv=4, eps=1e-5, tau=16.0)
BELETAR = dict(d=2048, ff=8192, pattern="DCDL", heads=8, dim=128, vdim=256, rank=128, conv=4, att_heads=16, att_dim=128,
               rot=64, att_vdim=128, kv_rank=512, eps=1e-6, embed_scale=8.0)


# ---- the cases ----------------------------------------------------------------------------------------------------------
def listed():
    return [
        # one chat on a provider: the smallest step, bound by launches and the weight stream
        {"name": "llama-decode-1", "stack": "llama-w4096", "kind": "decode", "seqs": 1, "context": 700},
        # the default provider's full load (maxConnections: 10), short chats of different lengths
        {"name": "llama-decode-10", "stack": "llama-w4096", "kind": "decode", "seqs": 10, "context": 300},
        # a busy provider: many chats in one step
        {"name": "llama-decode-64", "stack": "llama-w4096", "kind": "decode", "seqs": 64, "context": 900},
        # a few long documents being discussed: attention over long contexts
        {"name": "llama-decode-long", "stack": "llama-w2048", "kind": "decode", "seqs": 5, "context": 5400},
        # the next turn of a chat: a short prompt behind a cached conversation
        {"name": "llama-prompt-turn", "stack": "llama-w4096", "kind": "prompt", "seqs": 1, "tokens": 137, "context": 1200},
        # a burst of long prompts: the largest step
        {"name": "llama-prompt-burst", "stack": "llama-w4096", "kind": "prompt", "seqs": 8, "tokens": 8100, "context": 0},
        # routed experts: chats, and a burst of prompts
        {"name": "mixtral-decode-8", "stack": "mixtral-w2048", "kind": "decode", "seqs": 8, "context": 1100},
        {"name": "mixtral-prompt-burst", "stack": "mixtral-w2048", "kind": "prompt", "seqs": 8, "tokens": 8100, "context": 0},
        # recurrent and windowed layers: chats, and prompts of different lengths
        {"name": "lemunex-decode-8", "stack": "lemunex-w2048", "kind": "decode", "seqs": 8, "context": 1100},
        {"name": "lemunex-prompt-burst", "stack": "lemunex-w2048", "kind": "prompt", "seqs": 8, "tokens": 8100, "context": 0},
        # delta rule and latent attention: chats, and a few prompts together
        {"name": "beletar-decode-16", "stack": "beletar-w2048", "kind": "decode", "seqs": 16, "context": 600},
        {"name": "beletar-prompt-3", "stack": "beletar-w2048", "kind": "prompt", "seqs": 3, "tokens": 1530, "context": 0},
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    stack = rng.choice(["llama-w4096", "llama-w2048", "mixtral-w2048", "lemunex-w2048", "beletar-w2048"])
    if rng.random() < 0.5:
        seqs = spread(1, 64)
        return {"stack": stack, "kind": "decode", "seqs": seqs, "context": spread(16, min(5400, 60000 // seqs))}
    tokens = spread(16, 8000)
    seqs = min(rng.randint(1, 8), tokens)
    context = spread(64, 1500) if rng.random() < 0.3 and tokens // seqs < 3000 else 0
    return {"stack": stack, "kind": "prompt", "seqs": seqs, "tokens": tokens, "context": context}


def _lengths(case):
    """(cached tokens, new tokens) of every sequence: part of the case, the same for every seed."""
    rng = random.Random("%(stack)s %(kind)s %(seqs)d %(context)d" % case)
    n, c = case["seqs"], case["context"]

    def around(mean):
        return mean if n == 1 else max(1, min(int(mean * rng.uniform(0.5, 1.5)), MAX_POSITION - 1))

    if case["kind"] == "decode":
        return [max(1, around(c) - 1) for _ in range(n)], [1] * n
    parts = [rng.uniform(0.5, 1.5) for _ in range(n)]
    new = [max(1, int(case["tokens"] * p / sum(parts))) for p in parts]
    new[0] += max(0, case["tokens"] - sum(new))
    return [min(around(c), MAX_POSITION - m) if c else 0 for m in new], new


# ---- weights: tensor name -> bfloat16 tensor, the same for every seed ------------------------------------------------------
def _tensors(stack):
    """The stack's checkpoint: matrices [out, in] of variance about 1 / in, those that write to the stream smaller (as after
    training, a sublayer changes the stream by a part of its size); norm weights around their neutral value; decays from a
    few to a few hundred tokens."""
    gen = torch.Generator(device="cuda")

    def rand(name, *shape):
        gen.manual_seed(zlib.crc32((stack + name).encode()))
        return torch.randn(shape, generator=gen, device="cuda", dtype=torch.bfloat16)

    def uniform(name, *shape):
        gen.manual_seed(zlib.crc32((stack + name).encode()))
        return torch.rand(shape, generator=gen, device="cuda", dtype=torch.float32)

    w = {}

    def matrix(name, *shape, gain=1.0):
        w[name] = rand(name, *shape) * (gain * shape[-1] ** -0.5)

    def vector(name, n, mean, std):
        w[name] = (mean + std * rand(name, n).float()).bfloat16()

    if stack in LLAMA:
        c = LLAMA[stack]
        d, ff, dq, dkv = c["d"], c["ff"], c["heads"] * 128, c["kv"] * 128
        w["embed"] = rand("embed", VOCAB, d)
        matrix("lm_head", VOCAB, d)
        vector("norm", d, 1.0, 0.1)
        for i in range(LAYERS):
            p = f"layers.{i}."
            vector(p + "ln1", d, 1.0, 0.1)
            vector(p + "ln2", d, 1.0, 0.1)
            matrix(p + "wqkv", dq + 2 * dkv, d)
            matrix(p + "wo", d, dq, gain=0.5)
            if c["experts"]:
                matrix(p + "router", c["experts"], d, gain=2.0)
                matrix(p + "w13", c["experts"], 2 * ff, d)
                matrix(p + "w2", c["experts"], d, ff, gain=0.5)
            else:
                matrix(p + "w_gu", 2 * ff, d)
                matrix(p + "w_down", d, ff, gain=0.5)
        return w
    if stack == "lemunex-w2048":
        c = LEMUNEX
        d, H, G, D = c["d"], c["heads"], c["kv"], c["dim"]
        nk, nv = c["gla_heads"] * c["gla_dim"], c["gla_heads"] * c["gla_vdim"]
        inner = c["ssm_heads"] * c["ssm_vdim"]
        chans = inner + 2 * c["state"]
        w["embed"] = rand("embed", VOCAB, d)
        vector("embed.norm", d, 0.0, 0.1)
        vector("final.norm", d, 0.0, 0.1)
        matrix("head", VOCAB, d)
        for i, kind in enumerate(c["pattern"]):
            p, q = f"l{i}.", f"l{i}.mix."
            vector(p + "norm1", d, 0.0, 0.1)
            if kind == "p":
                for nm, rows in (("q", H * D), ("k", G * D), ("v", G * D)):
                    matrix(f"{q}left.{nm}", rows, d)
                    vector(f"{q}left.{nm}.b", rows, 0.0, 0.1)
                matrix(q + "left.g", H, d)
                matrix(q + "left.o", d, H * D)
                vector(q + "left.o.b", d, 0.0, 0.1)
                for nm, rows in (("q", nk), ("k", nk), ("v", nv), ("g", nv), ("a1", c["rank"])):
                    matrix(f"{q}right.{nm}", rows, d)
                matrix(q + "right.a2", nk, c["rank"])
                vector(q + "right.a2.b", nk, 3.0, 1.0)
                vector(q + "right.norm", c["gla_vdim"], 1.0, 0.1)
                matrix(q + "right.o", d, nv)
            else:
                matrix(q + "in", 2 * inner + 2 * c["state"] + c["ssm_heads"], d)
                matrix(q + "conv", chans, c["conv"])
                vector(q + "conv.b", chans, 0.0, 0.1)
                w[q + "dt_bias"] = (uniform(q + "dt_bias", c["ssm_heads"]) - 2.0).bfloat16()
                w[q + "A_log"] = torch.log(0.05 + 0.5 * uniform(q + "A_log", c["ssm_heads"])).bfloat16()
                w[q + "D"] = (0.5 + uniform(q + "D", c["ssm_heads"])).bfloat16()
                vector(q + "norm", inner, 1.0, 0.1)
                matrix(q + "o", d, inner, gain=0.5)
            matrix(p + "mlp.up", c["ff"], d)
            matrix(p + "mlp.down", d, c["ff"], gain=0.5)
        return w
    c = BELETAR
    d, H, N, P = c["d"], c["heads"], c["dim"], c["vdim"]
    matrix("embed", VOCAB, d)
    vector("final.norm", d, 1.0, 0.1)
    vector("final.norm.b", d, 0.0, 0.2)
    for i, kind in enumerate(c["pattern"]):
        p, q = f"l{i}.", f"l{i}.mix."
        for nm in ("norm1", "norm2"):
            vector(p + nm, d, 1.0, 0.1)
            vector(p + nm + ".b", d, 0.0, 0.2)
        if kind == "L":
            A, dn, r = c["att_heads"], c["att_dim"], c["kv_rank"]
            matrix(q + "q", A * (dn + c["rot"]), d)
            matrix(q + "dkv", r + c["rot"], d)
            vector(q + "dkv.norm", r, 1.0, 0.1)
            matrix(q + "uk", A * dn, r)
            matrix(q + "uv", A * c["att_vdim"], r)
            vector(q + "sink", A, 0.0, 1.0)
            matrix(q + "g", A, d)
            matrix(q + "o", d, A * c["att_vdim"], gain=0.5)
        else:
            for nm, rows in (("q", H * N), ("k", H * N), ("v", H * P)):
                matrix(q + nm, rows, d)
                matrix(f"{q}{nm}.conv", rows, c["conv"])
            matrix(q + "b", H, d)
            w[q + "A_log"] = torch.log(0.02 + 0.5 * uniform(q + "A_log", H)).bfloat16()
            vector(q + "norm", P, 1.0, 0.1)
            if kind == "C":
                matrix(q + "a1", c["rank"], d)
                matrix(q + "a2", H * N, c["rank"])
                w[q + "dt_bias"] = (uniform(q + "dt_bias", H * N) - 2.0).bfloat16()
                matrix(q + "g1", c["rank"], d)
                matrix(q + "g2", H * P, c["rank"])
            else:
                matrix(q + "a", H, d)
                w[q + "dt_bias"] = (uniform(q + "dt_bias", H) - 2.0).bfloat16()
                matrix(q + "g", H * P, d)
            matrix(q + "o", d, H * P, gain=0.5)
        matrix(p + "mlp.gate", c["ff"], d)
        matrix(p + "mlp.up", c["ff"], d)
        matrix(p + "mlp.down", d, c["ff"], gain=0.5)
    return w


_MODELS = {}


def _model(stack):
    """The model a program loads once and keeps for all its requests."""
    if stack not in _MODELS:
        from symmetry_amd.models import model_class
        from symmetry_amd.models.config import ModelConfig, beletar_stack, lemunex_stack
        from symmetry_amd.models.weights import ModelWeights, ShardSpec

        if stack in LLAMA:
            c = LLAMA[stack]
            cfg = ModelConfig(stack, VOCAB, c["d"], c["ff"], LAYERS, c["heads"], c["kv"], num_experts=c["experts"],
                              top_k=c["top"] or 2, **SPECIAL)
        elif stack == "lemunex-w2048":
            c = LEMUNEX
            cfg = lemunex_stack(stack, VOCAB, c["d"], c["pattern"], heads=c["heads"], kv_heads=c["kv"], dim=c["dim"],
                                window=c["window"], gla_heads=c["gla_heads"], gla_dim=c["gla_dim"], gla_vdim=c["gla_vdim"],
                                ssm_heads=c["ssm_heads"], ssm_vdim=c["ssm_vdim"], ssm_state=c["state"], ff=c["ff"],
                                decay_rank=c["rank"], **SPECIAL)
        else:
            c = BELETAR
            cfg = beletar_stack(stack, VOCAB, c["d"], c["pattern"], heads=c["heads"], kv_heads=c["heads"], dim=c["dim"],
                                vdim=c["vdim"], ff=c["ff"], att_heads=c["att_heads"], embed_scale=c["embed_scale"],
                                scaling=YARN, **SPECIAL)
        device = torch.device("cuda", torch.cuda.current_device())
        _MODELS[stack] = model_class(cfg)(ModelWeights(cfg, ShardSpec(), _tensors(stack)), device, max_decode_ctx=MAX_POSITION)
    return _MODELS[stack]


# ---- one step's inputs ----------------------------------------------------------------------------------------------------
def _planes(stack, blocks, slots):
    """The cache's tensors: name -> (shape, dtype, standard deviation of the values that earlier steps left)."""
    b16, f32 = torch.bfloat16, torch.float32
    if stack in LLAMA:
        kv = LLAMA[stack]["kv"]
        return {"k": ((LAYERS, blocks, kv, BLOCK, 128), b16, 1.0), "v": ((LAYERS, blocks, kv, 128, BLOCK), b16, 1.0)}
    out = {}
    if stack == "lemunex-w2048":
        c = LEMUNEX
        for i, kind in enumerate(c["pattern"]):
            if kind == "p":
                out[f"k{i}"] = ((blocks, BLOCK, c["kv"], c["dim"]), b16, 1.0)
                out[f"v{i}"] = ((blocks, BLOCK, c["kv"], c["dim"]), b16, 1.0)
                out[f"rec{i}"] = ((slots, c["gla_heads"], c["gla_dim"], c["gla_vdim"]), f32, 3.0)
            else:
                out[f"rec{i}"] = ((slots, c["ssm_heads"], c["state"], c["ssm_vdim"]), f32, 0.2)
                out[f"conv{i}"] = ((slots, c["conv"] - 1, c["ssm_heads"] * c["ssm_vdim"] + 2 * c["state"]), b16, 1.0)
        return out
    c = BELETAR
    for i, kind in enumerate(c["pattern"]):
        if kind == "L":
            out[f"lat{i}"] = ((blocks, BLOCK, c["kv_rank"] + c["rot"]), b16, 1.0)
        else:
            out[f"rec{i}"] = ((slots, c["heads"], c["dim"], c["vdim"]), f32, 0.3)
            out[f"conv{i}"] = ((slots, c["conv"] - 1, c["heads"] * (2 * c["dim"] + c["vdim"])), b16, 1.0)
    return out


def _cache_tensors(cache, stack):
    """The model's cache by the names of _planes."""
    if stack in LLAMA:
        return {"k": cache.k, "v": cache.v}
    kinds = ("k", "v", "rec", "conv") if stack == "lemunex-w2048" else ("lat", "rec", "conv")
    return {f"{kind}{i}": t for kind in kinds for i, t in getattr(cache, kind).items()}


def _inputs(case, seed):
    """What earlier steps left and this step's tokens: every sequence's blocks are scattered over the pool; it reads its
    carried state from one slot and leaves the new one in another, so that a step can be run again."""
    cached, new = _lengths(case)
    rng = random.Random(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    n, T = len(new), sum(new)
    need = [-(-(c + m) // BLOCK) for c, m in zip(cached, new)]
    blocks = sum(need) + 2
    order = list(range(1, blocks))
    rng.shuffle(order)
    tables, at = [], 0
    for k in need:
        tables.append(order[at:at + k])
        at += k
    planes = {name: torch.randn(shape, generator=gen, device="cuda", dtype=dtype) * std
              for name, (shape, dtype, std) in _planes(case["stack"], blocks, 2 * n).items()}
    tokens = torch.randint(0, VOCAB, (T,), generator=gen, device="cuda", dtype=torch.int32)
    return cached, new, blocks, tables, planes, tokens


def prepare(case, seed):
    from symmetry_amd.models.transformer import ForwardBatch

    stack = case["stack"]
    model = _model(stack)
    cached, new, blocks, tables, planes, tokens = _inputs(case, seed)
    n, T, decode = len(new), sum(new), case["kind"] == "decode"
    cache = model.make_cache(blocks, BLOCK, 2 * n)
    outputs = _cache_tensors(cache, stack)
    for name, t in outputs.items():
        t.copy_(planes[name])
    del planes
    width = max(len(t) for t in tables)
    if decode:
        width = next(-(-c // BLOCK) for c in CONTEXT_BUCKETS if -(-c // BLOCK) >= width)

    def ints(v, dtype=torch.int32):
        return torch.tensor(v, dtype=dtype, device="cuda")

    pos, slots, prev, save, row_seq, cu, tiles = [], [], [], [], [], [0], []
    for i in range(n):
        for p in range(cached[i], cached[i] + new[i]):
            slots.append(tables[i][p // BLOCK] * BLOCK + p % BLOCK)
            prev.append(len(pos) - 1 if p > cached[i] else -(i + 2) if cached[i] else -1)
            pos.append(p)
        save += [-1] * (new[i] - 1) + [n + i]
        row_seq += [i] * new[i]
        cu.append(len(pos))
        tiles += [(i, r) for r in range(0, new[i], 64)]
    tiles.sort(key=lambda t: -(cached[t[0]] + min(t[1] + 64, new[t[0]])))
    batch = ForwardBatch(
        kind="decode" if decode else "prefill", input_ids=tokens, positions=ints(pos), slot_mapping=ints(slots),
        block_tables=ints([t + [0] * (width - len(t)) for t in tables]), ctx_lens=ints([c + m for c, m in zip(cached, new)]),
        temps=torch.zeros(n, device="cuda"), seeds=ints([seed + i for i in range(n)], torch.int64),
        step=ints([1], torch.int64), num_seqs=n, need_logits=True, src=ints([-1] * T), top_k=ints([0] * n),
        top_p=torch.ones(n, device="cuda"), prev_row=ints(prev), save_slot=ints(save), row_seq=ints(row_seq))
    if not decode:
        batch.cu_q, batch.tiles, batch.last_idx = ints(cu), ints(tiles), ints([e - 1 for e in cu[1:]], torch.int64)
    state = {"model": model, "batch": batch, "cache": cache, "outputs": outputs, "graph": None}
    if decode or (stack in LLAMA and not LLAMA[stack]["experts"] and T <= GRAPH_PROMPT_TOKENS):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model.forward(batch, cache)  # (workspaces are made here, outside the capture)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            model.forward(batch, cache)
        state["graph"] = graph
        outputs["logits"] = model.last_logits
    return state


def run(state):
    """One step: the logits of every sequence's last token, and the cache and carried states that it leaves.  (The sampled
    ids are left out: of two nearly equal logits either may win.)"""
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        state["model"].forward(state["batch"], state["cache"])
        state["outputs"]["logits"] = state["model"].last_logits
    return state["outputs"]


# ---- what a step cannot do without ------------------------------------------------------------------------------------------
def _shapes(stack):
    """(layer matrices as a list of (elements, whether per expert), width)."""
    if stack in LLAMA:
        c = LLAMA[stack]
        d, dq = c["d"], c["heads"] * 128
        mats = [d * (dq + c["kv"] * 256) + d * dq] * LAYERS
        per_expert = 3 * d * c["ff"]
        return sum(mats) + (0 if c["experts"] else LAYERS * per_expert), LAYERS * per_expert if c["experts"] else 0, d
    if stack == "lemunex-w2048":
        c = LEMUNEX
        d, inner = c["d"], c["ssm_heads"] * c["ssm_vdim"]
        nk, nv = c["gla_heads"] * c["gla_dim"], c["gla_heads"] * c["gla_vdim"]
        pair = d * (2 * c["heads"] * c["dim"] + 2 * c["kv"] * c["dim"] + c["heads"] + 2 * nk + 3 * nv + c["rank"]) + c["rank"] * nk
        ssm = d * (3 * inner + 2 * c["state"] + c["ssm_heads"])
        return sum(pair if k == "p" else ssm for k in c["pattern"]) + LAYERS * 2 * d * c["ff"], 0, d
    c = BELETAR
    d, H, N, P, r, A = c["d"], c["heads"], c["dim"], c["vdim"], c["kv_rank"], c["att_heads"]
    head = d * (2 * H * N + 3 * H * P + 2 * H)
    chan = d * (2 * H * N + 2 * H * P + H + 2 * c["rank"]) + c["rank"] * (H * N + H * P)
    lat = d * (A * (c["att_dim"] + c["rot"]) + r + c["rot"] + A + A * c["att_vdim"]) + r * A * (c["att_dim"] + c["att_vdim"])
    return sum({"D": head, "C": chan, "L": lat}[k] for k in c["pattern"]) + LAYERS * 3 * d * c["ff"], 0, d


def work(case):
    stack = case["stack"]
    cached, new = _lengths(case)
    n, T = len(new), sum(new)
    dense, routed, d = _shapes(stack)
    c = LLAMA.get(stack)
    weights = dense + VOCAB * d
    flops = 2.0 * T * dense + 2.0 * n * VOCAB * d
    if routed:
        weights += routed * c["experts"] * (1 - (1 - c["top"] / c["experts"]) ** T)
        flops += 2.0 * T * c["top"] * routed
    size = 2.0 * weights + 2.0 * T * d + 4.0 * n * VOCAB
    for a, m in zip(cached, new):
        def seen(window):  # keys that the new rows see, and cached rows that are read
            return sum(min(p + 1, window) for p in range(a, a + m)), min(a, window)

        if c:
            pairs, rows = seen(MAX_POSITION)
            flops += LAYERS * 4.0 * c["heads"] * 128 * pairs
            size += LAYERS * 2.0 * 256 * c["kv"] * (rows + m)
        elif stack == "lemunex-w2048":
            e = LEMUNEX
            pairs, rows = seen(e["window"])
            flops += 2 * 4.0 * e["heads"] * e["dim"] * pairs
            size += 2 * 2.0 * 2 * e["kv"] * e["dim"] * (rows + m)
            gla, ssm = e["gla_heads"] * e["gla_dim"] * e["gla_vdim"], e["ssm_heads"] * e["state"] * e["ssm_vdim"]
            flops += 2 * 5.0 * (gla + ssm) * m
            size += 2 * 4.0 * (gla + ssm) * (2 if a else 1)
        else:
            e = BELETAR
            pairs, rows = seen(MAX_POSITION)
            if m == 1:  # through the latents: one key / value row serves every head
                flops += 2.0 * e["att_heads"] * (2 * e["kv_rank"] + e["rot"]) * pairs
            else:
                flops += 2.0 * e["att_heads"] * (e["att_dim"] + e["rot"] + e["att_vdim"]) * pairs
            size += 2.0 * (e["kv_rank"] + e["rot"]) * (rows + m)
            rec = e["heads"] * e["dim"] * e["vdim"]
            flops += 3 * 7.0 * rec * m
            size += 3 * 4.0 * rec * (2 if a else 1)
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """Four times the distance from the 64-bit step that bfloat16 activations and weights show on the logits: 0.0024 to 0.003
    (Llama, Mixtral), 0.005 (Lemunex), 0.01 (Beletar).  Twice that for routed experts, where a near tie may fall either way."""
    rel = {"llama-w4096": 0.011, "llama-w2048": 0.011, "mixtral-w2048": 0.022, "lemunex-w2048": 0.021, "beletar-w2048": 0.03}
    return {"rel": rel[case["stack"]], "max": 0.8}


# ---- the same step in 64 bits ----------------------------------------------------------------------------------------------
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, w, b, eps):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w + b


def _silu(x):
    return x * torch.sigmoid(x)


def _attend(q, k, v, first, scale, window=MAX_POSITION, sink=None):
    """q [m, H, dk] at positions first .., k [S, G, dk], v [S, G, dv] at positions 0 .. -> [m, H, dv]."""
    m, H = q.shape[:2]
    S, G = k.shape[:2]
    i = torch.arange(first, first + m, device=q.device)[:, None]
    j = torch.arange(S, device=q.device)[None, :]
    hidden = (j > i) | (j <= i - window)
    out = q.new_zeros(m, H, v.shape[2])
    for h in range(H):
        g = h // (H // G)
        s = (q[:, h] @ k[:, g].T * scale).masked_fill_(hidden, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].expand(m, 1)], 1)
        out[:, h] = torch.softmax(s, 1)[:, :S] @ v[:, g]
    return out


def _angles(dims, base, scaling=None):
    i = torch.arange(dims // 2, dtype=torch.float64, device="cuda")
    f, mag = base ** (-2.0 * i / dims), 1.0
    if scaling:
        factor, original, fast, slow = scaling

        def at(turns):
            return dims * math.log(original / (2.0 * math.pi * turns)) / (2.0 * math.log(base))

        lo, hi = max(math.floor(at(fast)), 0), min(math.ceil(at(slow)), dims - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        f, mag = f / factor * ramp + f * (1.0 - ramp), 0.1 * math.log(factor) + 1.0
    return f, mag


def _turn(x, pos, f, mag, pairs):
    """x [T, heads, D]: entry 2 i turns with 2 i + 1 (``pairs``), else entry i with entry i + D / 2."""
    a = pos.double()[:, None, None] * f
    co, si = torch.cos(a) * mag, torch.sin(a) * mag
    out, n = x.clone(), f.numel()
    u, v = (slice(0, 2 * n, 2), slice(1, 2 * n, 2)) if pairs else (slice(0, n), slice(n, 2 * n))
    out[..., u], out[..., v] = x[..., u] * co - x[..., v] * si, x[..., v] * co + x[..., u] * si
    return out


def _padded(x, new):
    """[T, ...] rows -> [sequences, longest, ...], zeros behind a sequence's end."""
    return torch.nn.utils.rnn.pad_sequence(list(x.split(new)), batch_first=True)


def _packed(x, new):
    return torch.cat([x[i, :m] for i, m in enumerate(new)])


def _conv(x, w, hist, new):
    """Causal taps w [C, taps] over every sequence behind its carried rows hist [n, taps - 1, C] -> (rows, newest rows)."""
    out, keep = [], []
    for i, z in enumerate(x.split(new)):
        z = torch.cat([hist[i], z])
        taps = w.shape[1]
        out.append(sum(z[j:j + new[i]] * w[:, j] for j in range(taps)))
        keep.append(z[-(taps - 1):])
    return torch.cat(out), torch.stack(keep)


def _scan(S, new, decay, k, v, q, beta=None):
    """S <- decay S + k u^T with u = v, or beta (v - S^T k) with the decayed S; o = S^T q.  S [n, H, N, P]; decay [T, H, N],
    k and q [T, H, N], v [T, H, P] -> (o [T, H, P], S)."""
    n = len(new)
    log = _padded(torch.log(decay), new)  # (a padded row: decay 1, k 0)
    k, v, q = _padded(k, new), _padded(v, new), _padded(q, new)
    beta = None if beta is None else _padded(beta, new)
    out = v.new_zeros(v.shape)
    for t in range(max(new)):
        S = S * torch.exp(log[:, t])[..., None]
        u = v[:, t]
        if beta is not None:
            u = beta[:, t, :, None] * (u - torch.matmul(k[:, t, :, None], S)[:, :, 0])
        S = S + k[:, t, :, :, None] * u[:, :, None]
        out[:, t] = torch.matmul(q[:, t, :, None], S)[:, :, 0]
    return _packed(out, new), S


class _Exact:
    """One step's sequences, and the cache's planes in 64 bits as the step leaves them."""

    def __init__(self, case, seed):
        cached, new, blocks, tables, planes, tokens = _inputs(case, seed)
        self.cached, self.new, self.n = cached, new, len(new)
        self.planes = {k: v.double() for k, v in planes.items()}
        self.tokens = tokens.long()
        self.tables = [torch.tensor(t, device="cuda") for t in tables]
        self.pos = torch.cat([torch.arange(c, c + m, device="cuda") for c, m in zip(cached, new)])
        self.last = torch.tensor(new, device="cuda").cumsum(0) - 1
        self.w = _tensors(case["stack"])

    def __getitem__(self, name):
        return self.w[name].double()

    def rows(self, i, upto):
        """(block, offset) of a sequence's positions below ``upto``."""
        p = torch.arange(upto, device="cuda")
        return self.tables[i][p // BLOCK], p % BLOCK

    def state(self, name):
        """The carried states that the step starts from."""
        t = self.planes[name][:self.n].clone()
        for i, c in enumerate(self.cached):
            if not c:
                t[i] = 0
        return t

    def paged(self, plane, x):
        """Stores the new rows x [T, ...] in a token-major plane [blocks, BLOCK, ...]; yields every sequence's rows."""
        for i, z in enumerate(x.split(self.new)):
            b, o = self.rows(i, self.cached[i] + self.new[i])
            plane[b[self.cached[i]:], o[self.cached[i]:]] = z
            yield plane[b, o]


def _exact_llama(e, c):
    H, G = c["heads"], c["kv"]
    f, _ = _angles(128, 500000.0)
    x = e["embed"][e.tokens]
    for i in range(LAYERS):
        p = f"layers.{i}."
        h = _rms(x, 1e-5) * e[p + "ln1"]
        q, k, v = (h @ e[p + "wqkv"].T).split([H * 128, G * 128, G * 128], 1)
        q, k, v = _turn(q.unflatten(1, (H, 128)), e.pos, f, 1.0, False), k.unflatten(1, (G, 128)), v.unflatten(1, (G, 128))
        k = _turn(k, e.pos, f, 1.0, False)
        kp, vp = e.planes["k"][i].transpose(1, 2), e.planes["v"][i].permute(0, 3, 1, 2)  # token-major views
        o = [_attend(qs, ks, vs, a, 128 ** -0.5) for qs, ks, vs, a in zip(q.split(e.new), e.paged(kp, k), e.paged(vp, v), e.cached)]
        x = x + torch.cat(o).flatten(1) @ e[p + "wo"].T
        h = _rms(x, 1e-5) * e[p + "ln2"]
        if not c["experts"]:
            g, u = (h @ e[p + "w_gu"].T).chunk(2, 1)
            x = x + (_silu(g) * u) @ e[p + "w_down"].T
            continue
        value, chosen = (h @ e[p + "router"].T).topk(c["top"], 1)
        share, add = torch.softmax(value, 1), torch.zeros_like(x)
        for j in range(c["experts"]):
            row, at = (chosen == j).nonzero(as_tuple=True)
            g, u = (h[row] @ e.w[p + "w13"][j].double().T).chunk(2, 1)
            add.index_add_(0, row, share[row, at, None] * ((_silu(g) * u) @ e.w[p + "w2"][j].double().T))
        x = x + add
    return _rms(x[e.last], 1e-5) * e["norm"] @ e["lm_head"].T


def _exact_lemunex(e, c):
    eps, n = c["eps"], e.n
    H, G, D, gh, gk, gv = c["heads"], c["kv"], c["dim"], c["gla_heads"], c["gla_dim"], c["gla_vdim"]
    f, mag = _angles(D // 2, 10000.0, YARN)
    x = _rms(e["embed"][e.tokens], eps) * (1 + e["embed.norm"])
    for i, kind in enumerate(c["pattern"]):
        p, m = f"l{i}.", f"l{i}.mix."
        h = _rms(x, eps) * (1 + e[p + "norm1"])
        if kind == "p":
            q, k, v = ((h @ e[f"{m}left.{nm}"].T + e[f"{m}left.{nm}.b"]).unflatten(1, (-1, D)) for nm in "qkv")
            q, k = _turn(q, e.pos, f, mag, True), _turn(k, e.pos, f, mag, True)
            o = [_attend(qs, ks, vs, a, D ** -0.5, c["window"]) for qs, ks, vs, a in
                 zip(q.split(e.new), e.paged(e.planes[f"k{i}"], k), e.paged(e.planes[f"v{i}"], v), e.cached)]
            o = torch.cat(o) * torch.sigmoid(h @ e[m + "left.g"].T)[..., None]
            left = o.flatten(1) @ e[m + "left.o"].T + e[m + "left.o.b"]
            q, k, v = ((h @ e[f"{m}right.{nm}"].T).unflatten(1, (gh, -1)) for nm in "qkv")
            z = h @ e[m + "right.a1"].T @ e[m + "right.a2"].T + e[m + "right.a2.b"]
            decay = torch.sigmoid(z).pow(1 / c["tau"]).unflatten(1, (gh, gk))
            o, S = _scan(e.state(f"rec{i}"), e.new, decay, k, v, q * gk ** -0.5)
            e.planes[f"rec{i}"][n:] = S
            o = (_rms(o, eps) * e[m + "right.norm"]).flatten(1) * _silu(h @ e[m + "right.g"].T)
            mix = 0.5 * left + 0.5 * (o @ e[m + "right.o"].T)
        else:
            inner, st, sh = c["ssm_heads"] * c["ssm_vdim"], c["state"], c["ssm_heads"]
            z, y, dt = (h @ e[m + "in"].T).split([inner, inner + 2 * st, sh], 1)
            y, keep = _conv(y, e[m + "conv"], e.state(f"conv{i}"), e.new)
            e.planes[f"conv{i}"][n:] = keep
            v, B, C = _silu(y + e[m + "conv.b"]).split([inner, st, st], 1)
            v = v.unflatten(1, (sh, -1))
            dt = torch.log1p(torch.exp(dt + e[m + "dt_bias"]))
            decay = torch.exp(-torch.exp(e[m + "A_log"]) * dt)[..., None].expand(-1, -1, st)
            k, q = dt[..., None] * B[:, None], C[:, None].expand(-1, sh, -1)
            o, S = _scan(e.state(f"rec{i}"), e.new, decay, k, v, q)
            e.planes[f"rec{i}"][n:] = S
            o = (o + e[m + "D"][:, None] * v).flatten(1) * _silu(z)
            mix = _rms(o, eps) * e[m + "norm"] @ e[m + "o"].T
        x = x + mix + torch.relu(h @ e[p + "mlp.up"].T) ** 2 @ e[p + "mlp.down"].T
    return _rms(x[e.last], eps) * (1 + e["final.norm"]) @ e["head"].T


def _exact_beletar(e, c):
    eps, n = c["eps"], e.n
    H, N, P, A, dn, r = c["heads"], c["dim"], c["vdim"], c["att_heads"], c["att_dim"], c["kv_rank"]
    f, mag = _angles(c["rot"], 10000.0, YARN)
    x = e["embed"][e.tokens] * c["embed_scale"]

    def unit(v):
        return v / torch.sqrt((v * v).sum(-1, keepdim=True) + 1e-6)

    for i, kind in enumerate(c["pattern"]):
        p, m = f"l{i}.", f"l{i}.mix."
        h = _layer_norm(x, e[p + "norm1"], e[p + "norm1.b"], eps)
        if kind == "L":
            qn, qr = (h @ e[m + "q"].T).unflatten(1, (A, -1)).split([dn, c["rot"]], 2)
            z, kr = (h @ e[m + "dkv"].T).split([r, c["rot"]], 1)
            qr, kr = _turn(qr, e.pos, f, mag, True), _turn(kr[:, None], e.pos, f, mag, True)[:, 0]
            row = torch.cat([_rms(z, eps) * e[m + "dkv.norm"], kr], 1)
            o = []
            for a, qa, qb, rows in zip(e.cached, qn.split(e.new), qr.split(e.new), e.paged(e.planes[f"lat{i}"], row)):
                k = (rows[:, :r] @ e[m + "uk"].T).unflatten(1, (A, dn))
                k = torch.cat([k, rows[:, None, r:].expand(-1, A, -1)], 2)
                v = (rows[:, :r] @ e[m + "uv"].T).unflatten(1, (A, -1))
                o.append(_attend(torch.cat([qa, qb], 2), k, v, a, (dn + c["rot"]) ** -0.5, sink=e[m + "sink"]))
            o = (torch.cat(o) * torch.sigmoid(h @ e[m + "g"].T)[..., None]).flatten(1)
        else:
            y = torch.cat([h @ e[m + nm].T for nm in "qkv"], 1)
            y, keep = _conv(y, torch.cat([e[f"{m}{nm}.conv"] for nm in "qkv"]), e.state(f"conv{i}"), e.new)
            e.planes[f"conv{i}"][n:] = keep
            q, k, v = _silu(y).split([H * N, H * N, H * P], 1)
            q, k, v = unit(q.unflatten(1, (H, N))) * N ** -0.5, unit(k.unflatten(1, (H, N))), v.unflatten(1, (H, P))
            rate = torch.exp(e[m + "A_log"])[:, None]
            z = h @ e[m + "a1"].T @ e[m + "a2"].T if kind == "C" else h @ e[m + "a"].T
            z = torch.log1p(torch.exp(z + e[m + "dt_bias"])).unflatten(1, (H, -1))
            decay = torch.exp(-rate * z).expand(-1, -1, N)
            o, S = _scan(e.state(f"rec{i}"), e.new, decay, k, v, q, torch.sigmoid(h @ e[m + "b"].T))
            e.planes[f"rec{i}"][n:] = S
            gate = torch.sigmoid(h @ e[m + "g1"].T @ e[m + "g2"].T) if kind == "C" else _silu(h @ e[m + "g"].T)
            o = (_rms(o, eps) * e[m + "norm"]).flatten(1) * gate
        x = x + o @ e[m + "o"].T
        h = _layer_norm(x, e[p + "norm2"], e[p + "norm2.b"], eps)
        x = x + (_silu(h @ e[p + "mlp.gate"].T) * (h @ e[p + "mlp.up"].T)) @ e[p + "mlp.down"].T
    return _layer_norm(x[e.last], e["final.norm"], e["final.norm.b"], eps) @ e["embed"].T


@torch.no_grad()
def exact(case, seed):
    stack, e = case["stack"], _Exact(case, seed)
    if stack in LLAMA:
        logits = _exact_llama(e, LLAMA[stack])
    else:
        logits = _exact_lemunex(e, LEMUNEX) if stack == "lemunex-w2048" else _exact_beletar(e, BELETAR)
    return dict(e.planes, logits=logits)

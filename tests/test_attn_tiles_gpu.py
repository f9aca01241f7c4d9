"""Prompt attention over key tiles of 64 in LDS (csrc/kernels/attention.hip, attn_prefill_m32p_kernel) against attention in 64 bits, at the
ends of its tiles and subtiles, for blocks of half a tile (the entry takes no smaller ones) to two.

Bound: a weight is rounded to bf16 (8 bits: at most 2^-8 of it) in front of the product with the values, the result once more (2^-8 of
it); scores and sums are fp32 (2^-20 of the weights covers both)."""
import math

import pytest
import torch

from symmetry_amd import ops

pytestmark = pytest.mark.gpu
D = 128


@pytest.mark.parametrize("BS", [32, 64, 128])
@pytest.mark.parametrize("Hq,Hkv,copies", [(8, 2, 1), (16, 4, 4), (16, 2, 3)])
@pytest.mark.parametrize("slow", [False, True])
def test_tiles_of_keys(gpu, BS, Hq, Hkv, copies, slow):
    """Prompts of a row to a few tiles, alone and behind contexts; scores of every size (slow: growing along the keys, so that the running
    maximum moves in every subtile).  Keys past a context are NaN, values too from the next group of 8 on."""
    specs = [(1, 1), (31, 31), (32, 32), (33, 33), (63, 63), (64, 64), (65, 65), (128, 128), (129, 129), (7, 200), (70, 333), (40, 64), (300, 421)] * copies
    g = torch.Generator(device=gpu).manual_seed(BS + Hq)
    blocks = [(c + BS - 1) // BS for _, c in specs]
    kc = torch.randn(sum(blocks), Hkv, BS, D, device=gpu, generator=g).bfloat16()
    vc = torch.randn(sum(blocks), Hkv, D, BS, device=gpu, generator=g).bfloat16()
    order = torch.randperm(sum(blocks), generator=torch.Generator().manual_seed(BS))
    bt = torch.zeros(len(specs), max(blocks) + 1, dtype=torch.int32)
    T = sum(n for n, _ in specs)
    q = torch.randn(T, Hq, D, device=gpu, generator=g).bfloat16()
    at, r, want, weight = 0, 0, torch.empty(T, Hq, D, device=gpu, dtype=torch.float64), torch.empty(T, Hq, D, device=gpu, dtype=torch.float64)
    scale = 1 / math.sqrt(D)
    for s, ((n, c), b) in enumerate(zip(specs, blocks)):
        ids = order[at:at + b]
        bt[s, :b], at = ids.int(), at + b
        k, v = kc[ids].transpose(1, 2).reshape(-1, Hkv, D), vc[ids].permute(0, 3, 1, 2).reshape(-1, Hkv, D)
        if slow:
            k = k * (1 + torch.arange(len(k), device=gpu)[:, None, None] / 16).to(k.dtype)
        k[c:], v[(c + 7) // 8 * 8:] = float("nan"), float("nan")
        kc[ids], vc[ids] = k.view(b, BS, Hkv, D).transpose(1, 2), v.view(b, BS, Hkv, D).permute(0, 2, 3, 1)
        kd, vd = (t[:c].double().repeat_interleave(Hq // Hkv, 1) for t in (k, v))
        x = torch.einsum("qhd,khd->hqk", q[r:r + n].double().cpu(), kd.cpu()).to(gpu) * scale
        x = x.masked_fill(torch.arange(c, device=gpu)[None] > torch.arange(c - n, c, device=gpu)[:, None], -math.inf).softmax(-1)
        want[r:r + n] = torch.einsum("hqk,khd->qhd", x.cpu(), vd.cpu()).to(gpu)
        weight[r:r + n] = torch.einsum("hqk,khd->qhd", x.cpu(), vd.abs().cpu()).to(gpu)
        r += n
    i32 = dict(dtype=torch.int32, device=gpu)
    tiles = torch.tensor([(s, i) for s, (n, _) in enumerate(specs) for i in range(0, n, 64)] + [(0, 1 << 20)] * 40, **i32)
    cu = torch.tensor([sum(n for n, _ in specs[:i]) for i in range(len(specs) + 1)], **i32)
    out = torch.empty_like(q)
    ops.attn_prefill(q, kc, vc, bt.to(gpu), torch.tensor([c for _, c in specs], **i32), cu, tiles, out, scale)
    bound = 2 ** -8 * (weight + want.abs()) + 2 ** -20 * (1 + weight)
    worst = ((out.double() - want).abs() / bound).max()
    assert worst <= 1, float(worst)

"""The prompt form of the rotary embedding and K/V write against its row form (the same arithmetic: equal bits)."""
import pytest
import torch

from symmetry_amd import ops
from symmetry_amd.ops import reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [32, 63, 64, 65, 137])
@pytest.mark.parametrize("start", [0, 3, 40])
@pytest.mark.parametrize("dims", [(8, 2, 128, 64), (3, 1, 48, 16), (4, 3, 80, 12), (2, 1, 256, 32)])
@pytest.mark.parametrize("slabs", [0, 3])
def test_forms_agree(T, start, dims, slabs):
    """Two sequences (the second begins inside a 64-row tile), shuffled blocks, runs that begin anywhere, padding rows, block
    sizes that are and are not multiples of 8, column counts that leave a part of a tile."""
    H, G, D, BS = dims
    print("rope_cache", T, start, dims, slabs, flush=True)
    torch.manual_seed(T + start)
    N, cut = (H + 2 * G) * D, T // 3
    mb = (T + start) // BS + 1
    bt = torch.randperm(2 * mb)
    pos = torch.cat([torch.arange(cut) + start, torch.arange(T - cut)])
    slots = torch.cat([bt[(torch.arange(cut) + start) // BS] * BS + (torch.arange(cut) + start) % BS,
                       bt[mb + torch.arange(T - cut) // BS] * BS + torch.arange(T - cut) % BS])
    slots[T - 2:] = -1
    slots[cut // 2] = -1
    qkv = torch.randn(T, N).bfloat16() if slabs == 0 else torch.randn(slabs, T, N)
    qkv, pos, slots = qkv.cuda(), pos.int().cuda(), slots.int().cuda()
    cs = reference.rope_table(256, D, 1e4).cuda()
    got = []
    for decode in (False, True):
        q = torch.full((T + 1, H, D), 5.0, dtype=torch.bfloat16, device="cuda")
        k = torch.full((2 * mb, G, BS, D), 5.0, dtype=torch.bfloat16, device="cuda")
        v = torch.full((2 * mb, G, D, BS), 5.0, dtype=torch.bfloat16, device="cuda")
        ops.rope_cache(qkv, pos, slots, cs, q[:T], k, v, H, G, decode=decode)
        got.append((q, k, v))
    for a, b in zip(*got):
        assert torch.equal(a, b)

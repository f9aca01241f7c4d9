"""Partitions of decode steps over a latent cache: both sides of the line between 64 and 128 keys."""
from symmetry_amd import ops


def test_smallest_partition():
    def least(rows, span, heads=16, kv_rank=512, rot=64, block=64):
        return ops.latent_row_tokens(rows, heads, span, kv_rank, rot, block)

    assert [least(n, 512) for n in (1, 16, 32, 33, 64)] == [64, 64, 64, 128, 128]
    assert [least(n, 2048) for n in (1, 8, 9, 16)] == [64, 64, 128, 128]
    assert [least(n, 2048, heads) for n, heads in ((8, 17), (4, 32), (5, 17))] == [128, 64, 128]
    assert least(1, 4096) == 64 and least(1, 4097) == 128 and least(64, 64) == 64
    assert least(64, 2048, kv_rank=256) == least(64, 2048, rot=32) == least(64, 2048, block=16) == least(64, 2048, block=96) == 64
    assert ops.latent_attn_parts(16, 2048, min_tokens=128) == 16 and ops.latent_attn_parts(1, 8192, min_tokens=128) == 64

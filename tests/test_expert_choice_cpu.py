"""Which form a routed product takes (csrc/kernels/routed_ff.hip, expert_linear_form), on both sides of every line of the rule and
without the tensors: 0 all shapes, 1 weight stream, 2 / 3 tiles of 128 / 256, 4 the walk over the chosen experts' weights."""
import pytest

from symmetry_amd import ops


def form(R, E, N, K, glu=False, rows=None):
    return ops._hyb().expert_linear_choice(R, E, N, K, R if rows is None else rows, glu, False)


def test_rows_per_expert_part_streams_and_tiles():
    for glu in (False, True):
        assert [form(R, 16, 1024, 1024, glu) for R in (1, 128, 129)] == [1, 1, 2]
        assert [form(R, 16, 1024, 1056, glu) for R in (128, 129, 9000)] == [1, 1, 1]         # (widths in 64s have tiles)
        assert [form(R, 16, 2048, 2048, glu) for R in (128, 129)] == [4, 2]
    assert form(32, 16, 1024, 1000) == 0                                                     # (no width in 32s)


@pytest.mark.parametrize("K", [512, 1536, 2048, 3072])
def test_widths_that_walk(K):
    assert sorted(ops._walk_widths()) == [512, 1536, 2048, 3072]
    assert form(64, 32, 2048, K) == 4 and form(64, 32, 2048, K + 64) == 1 and form(64, 32, 1535, K) == 1
    assert form(64, 64, 2048, K) == 4 and form(64, 65, 2048, K) == 1                         # (a lane knows one expert's segment)
    assert form(512, 64, 2048, K) == 4 and form(513, 64, 2048, K) == 2
    assert form(64, 32, 1536, K, True) == (1 if K == 512 else 4)


def test_few_experts_stay_on_the_stream():
    """256 CUs: a unit is 16 outputs of an expert, gated 8."""
    assert [form(R, 8, 512, 2048, True) for R in (15, 16, 64)] == [4, 1, 1]                  # 512 units
    assert [form(64, E, 512, 2048, True) for E in (4, 8, 9, 16)] == [2, 1, 4, 4]             # (4 experts: 16 rows each)
    assert [form(32, E, 512, 2048, True) for E in (4, 5, 8, 9)] == [4, 1, 1, 4]              # 256, 320, 512, 576
    assert [form(R, 32, 2048, 512) for R in (4, 5)] == [1, 4]                                # 512, 640 of the chosen ones
    assert [form(R, 8, 2048, 2048) for R in (11, 12, 64)] == [4, 1, 1]                       # 1024
    assert [form(32, E, 2048, 2048) for E in (8, 9, 16)] == [1, 4, 4]
    assert [form(32, E, 2048, K) for E in (4, 8) for K in (1536, 3072)] == [4] * 4


def test_persistent_tiles_need_rows_and_rounds():
    assert [form(16 * per, 16, 2048, 1536) for per in (127, 128, 2025)] == [2, 3, 3]
    assert [form(16 * per, 16, 1536, 2048, True) for per in (127, 128, 2025)] == [2, 3, 3]
    assert form(16 * 128, 16, 255, 2048) == 2 and form(64 * 128, 64, 256, 2048) == 2         # (64 tiles)
    # below 0.3 rounds of 256 the small ones: 8 experts of 2048 outputs are 64 tiles up to 256 rows each
    assert [form(8 * per, 8, 2048, 1536) for per in (128, 256, 257)] == [2, 2, 3]
    assert [form(128 * E, E, 2048, 2048) for E in (9, 10)] == [2, 3]                         # 72, 80
    assert [form(8 * per, 8, 512, 2048) for per in (375, 500, 1024, 1025)] == [2, 2, 2, 3]   # 32, 32, 64, 80
    # gated, 0.7 to 1 round of whole tiles: 12 columns of 128
    assert [form(R, 16, 1536, 2048, True) for R in (14 * 256, 15 * 256, 21 * 256, 22 * 256)] == [3, 2, 2, 3]


def test_narrow_widths_need_more():
    assert [form(16 * per, 16, 2048, 960) for per in (1023, 1024)] == [2, 3] and form(16 * 128, 16, 2048, 1024) == 3
    assert form(16 * 4096, 16, 2048, 448) == 2 and form(16 * 4096, 16, 2048, 512) == 3       # (eight stages at least)
    assert form(16 * 4096, 16, 1023, 512) == 2 and form(16 * 4096, 16, 1024, 512) == 3
    assert [form(16 * per, 16, 1536, 768) for per in (1024, 1280, 1281)] == [2, 2, 3]        # 480 and 576 tiles: two rounds are 512
    assert [form(16 * per, 16, 512, 768, True) for per in (4096,)] == [2]                    # (outputs from 1024)
    assert [form(4 * per, 4, 1024, 512, True) for per in (1792, 2048)] == [2, 3]             # 224 and 256: one round


def test_operands_past_a_buffers_range():
    """x and an expert's weights are addressed by 32-bit offsets: what does not fit stays on the tiles of 128."""
    top = 0x7FFFFFFF
    K = 4096
    rows = top // (2 * K)
    assert form(16 * 256, 16, 4096, K, rows=rows) == 3 and form(16 * 256, 16, 4096, K, rows=rows + 1) == 2
    N = top // (2 * K) - 512
    assert form(16 * 256, 16, N, K) == 3 and form(16 * 256, 16, N + 1, K) == 2
    N = (top // (2 * K) - 512) // 2
    assert form(16 * 512, 16, N, K, True) == 3 and form(16 * 512, 16, N + 1, K, True) == 2


def test_sizes_that_are_none_are_refused():
    for bad in ((0, 16, 64, 64), (4, 0, 64, 64), (4, 16, 0, 64), (4, 16, 64, 0), (4, 16, 1 << 31, 64)):
        with pytest.raises(RuntimeError, match="sizes"):
            form(*bad, rows=4)


def test_dense_gated_projections_need_full_rounds():
    """256 CUs; whole tiles of 256 rows x 128 pairs, half ones 5 / 9 of their time: 0.6 of a round's work to be done, from 4096 wide 0.8."""
    pays = ops._hyb().dense_glu_pays
    assert [pays(M, 8192, 2048) for M in (256, 320, 400, 513, 600, 700, 1530, 8100)] == [False, False, True, False, False, True, True, True]
    assert [pays(M, 5632, 2048) for M in (700, 800, 1000)] == [False, False, True]
    assert [pays(M, 14336, 4096) for M in (400, 700, 1000, 1100)] == [False, False, True, True]
    assert [pays(4000, 8192, K) for K in (960, 1024)] == [False, True] and not pays(4000, 255, 2048)
    assert pays(1600, 2048, 2048, 64) and pays(400, 2048, 2048, 64) == pays(400, 8192, 2048, 256)

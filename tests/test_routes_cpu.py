"""Which kernel a launch takes, asked of the library's own rules without a GPU."""
import ctypes as C
import os

import pytest

from nerva_amd import abi

pytestmark = pytest.mark.skipif(not os.path.exists(abi.LIBRARY), reason="library not built")

PLAIN, RESIDUAL, SWIGLU, XIELU = range(4)
FEW, WIDE, DEEP = 2, 5, 6    # enum GemmKernel of gemm_rows.cuh


def route(epilogue, rows, cols, tokens, workspace=1 << 32, reader_adds=False):
    """(kernel, K slices) of nv::gemm_rows_route(int, uint32_t, uint32_t, uint32_t, uint64_t, bool)."""
    rule = getattr(abi.load(), "_ZN2nv15gemm_rows_routeEijjjmb")
    rule.restype, rule.argtypes = C.c_uint64, [C.c_int, C.c_uint32, C.c_uint32, C.c_uint32, C.c_uint64, C.c_bool]
    both = rule(epilogue, rows, cols, tokens, workspace, reader_adds)
    return both & 0xffffffff, both >> 32


def test_activated_projections_are_judged_by_the_tiles_they_launch():
    """The kernel with wave pairs has no xIELU launches of fewer than sixteen token tiles, so its time does not grow with the
    tokens from 129 to 256, and the other kernel's does not fall: where it is taken, it is taken for more tokens too."""
    for rows, cols, tokens in ((11136, 3584, 160), (12288, 3584, 160), (12288, 4096, 130), (12288, 4096, 160)):
        assert route(XIELU, rows, cols, tokens)[0] == DEEP    # (54 us in sixteen tiles against 33; 40 against 36)
    for cols in range(512, 4097, 128):
        for rows in range(2 * cols, 4 * cols + 1, 192):
            pairs = [route(XIELU, rows, cols, tokens)[0] == WIDE for tokens in (129, 160, 192, 224, 256)]
            assert pairs == sorted(pairs), (rows, cols)


def test_projections_of_few_tiles_leave_the_256_row_tiles_only_for_something_faster():
    """Long runs of K in few workgroups, and rows short of the last tiles: measured faster in 256-row tiles (46.9 against 52.0 us,
    47.0 and 52.2, 58.9 and 69.8, 31.5 and 32.9). The others gain by the tiles left out."""
    for epilogue, rows, cols, tokens in ((RESIDUAL, 3584, 14336, 189), (RESIDUAL, 3584, 14336, 139), (RESIDUAL, 4096, 14336, 185), (RESIDUAL, 4608, 18432, 194),
                                         (PLAIN, 9216, 3072, 208)):
        assert route(epilogue, rows, cols, tokens)[0] == DEEP, (rows, cols)
    for epilogue, rows, cols, tokens in ((PLAIN, 9216, 3072, 136), (RESIDUAL, 8192, 8192, 160), (RESIDUAL, 4096, 12288, 160), (PLAIN, 6144, 4096, 250)):
        assert route(epilogue, rows, cols, tokens)[0] == WIDE, (rows, cols)


def test_few_rows_leave_the_k_slices_only_for_something_faster():
    """More workgroups than CUs start twice, and 9 and more tokens are fetched more slowly: measured 17.4 us in slices against 19.8,
    12.4 and 13.4, 12.2 and 12.9, 16.6 and 17.3. Narrow matrices gain by the launch that they do without."""
    for epilogue, rows, cols, tokens in ((PLAIN, 7168, 5120, 9), (PLAIN, 7168, 5120, 16), (SWIGLU, 5120, 2048, 9), (RESIDUAL, 4096, 4096, 6),
                                         (RESIDUAL, 4096, 4096, 16), (SWIGLU, 8192, 2048, 24), (PLAIN, 6912, 3840, 16)):
        assert route(epilogue, rows, cols, tokens)[0] != FEW, (rows, cols)
    for epilogue, rows, cols, tokens in ((PLAIN, 4096, 1024, 6), (RESIDUAL, 1024, 2048, 6), (RESIDUAL, 1024, 3072, 16), (SWIGLU, 3072, 1024, 6), (PLAIN, 2688, 3328, 16),
                                         (SWIGLU, 2048, 512, 17)):
        assert route(epilogue, rows, cols, tokens)[0] == FEW, (rows, cols)


def test_slices_that_their_reader_adds_cost_less():
    """The q/k/v projection of a batch step, whose attention adds the slices: 9.1 us + 1 against 9.2 of a launch without slices, and
    11.8 with a launch that adds them."""
    assert route(PLAIN, 6144, 2560, 4)[0] == FEW
    assert route(PLAIN, 6144, 2560, 4, reader_adds=True)[0] != FEW and route(PLAIN, 6144, 2560, 4, reader_adds=True)[1] > 1
    assert route(PLAIN, 4096, 1024, 6, reader_adds=True)[0] == FEW


def test_long_batches_that_fill_the_chip_stay_with_the_block_kernel():
    """32 sequences, 32 heads of 128 on 8, one split each: the step kernel is the faster one up to about 2500 keys (18.1 against 20.8
    us at 767, 180 against 167 at 8250); with fewer workgroups, heads of 64 or eight query heads a key head it is at every length."""
    rule = getattr(abi.load(), "_ZN2nv18attn_batch_in_stepEjjjjjj")
    rule.restype, rule.argtypes = C.c_bool, [C.c_uint32] * 6

    def step(heads, kv_heads, head_dim, sequences, keys, splits=1):
        return rule(heads, kv_heads, head_dim, sequences, splits, (keys + 15) // 16)
    for heads in (8, 16, 32, 40, 56):
        assert step(heads, 8, 128, 32, 1) and step(heads, 8, 128, 32, 2048)
        assert not step(heads, 8, 128, 32, 2049) and not step(heads, 8, 128, 32, 8264)
    assert step(64, 8, 128, 32, 8264) and step(24, 8, 64, 32, 8264) and step(32, 8, 128, 24, 8264) and step(32, 4, 128, 32, 8264)
    assert not step(32, 8, 128, 33, 100) and not step(32, 8, 128, 16, 100, splits=2)
    assert not rule(32, 8, 128, 32, 1, 0)    # a launch that does not say how long its sequences are


def test_few_sequences_of_short_merges_split_earlier():
    """2 and 4 sequences of 16 heads of 128 on 8 read 628 to 760 keys faster in splits (12.1 to 12.4 and 12.8 to 12.9 us, in one 12.9 to
    13.8 and 13.0 to 13.6); more sequences, more query heads a key head and heads of 64 do not."""
    rule = getattr(abi.load(), "_ZN2nv23attn_batch_single_splitEjjjj")
    rule.restype, rule.argtypes = C.c_uint32, [C.c_uint32] * 4
    for heads, sequences in ((8, 4), (16, 2), (16, 4), (24, 4)):
        assert rule(heads, 8, 128, sequences) == 36
    for heads, kv_heads, head_dim, sequences in ((16, 8, 128, 6), (32, 8, 128, 4), (28, 4, 128, 4), (16, 8, 64, 4), (8, 2, 64, 9)):
        assert rule(heads, kv_heads, head_dim, sequences) == 48


def test_expert_routes_count_only_where_rounds_take_longer():
    """Counting who is ahead grows with the experts, rounds of an argmax with the chosen: measured 3.6 us against 3.2 for 1 of 32, 8.6
    and 5.1 for 2 of 128, 15.4 and 13.7 for 8 of 256; 4.5 and 10.7 for 8 of 48, 8.6 and 11.7 for 8 of 128."""
    rule = getattr(abi.load(), "_ZN2nv16moe_route_rankedEjj")
    rule.restype, rule.argtypes = C.c_bool, [C.c_uint32] * 2
    for experts, top in ((32, 1), (48, 2), (64, 2), (128, 1), (128, 2), (128, 4), (256, 1), (256, 8), (257, 64), (1024, 64)):
        assert not rule(experts, top), (experts, top)
    for experts, top in ((1, 1), (8, 1), (8, 2), (16, 1), (16, 4), (32, 2), (48, 8), (64, 4), (64, 8), (128, 8), (192, 8), (256, 64)):
        assert rule(experts, top), (experts, top)

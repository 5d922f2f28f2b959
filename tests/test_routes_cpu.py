"""Which kernel a launch takes, asked of the library's own rules without a GPU."""
import ctypes as C
import os

import pytest

from nerva_amd import abi

pytestmark = pytest.mark.skipif(not os.path.exists(abi.LIBRARY), reason="library not built")

PLAIN, RESIDUAL, XIELU = 0, 1, 3
WIDE, DEEP = 5, 6    # enum GemmKernel of gemm_rows.cuh


def route(epilogue, rows, cols, tokens, workspace=1 << 32):
    """(kernel, K slices) of nv::gemm_rows_route(int, uint32_t, uint32_t, uint32_t, uint64_t)."""
    rule = getattr(abi.load(), "_ZN2nv15gemm_rows_routeEijjjm")
    rule.restype, rule.argtypes = C.c_uint64, [C.c_int, C.c_uint32, C.c_uint32, C.c_uint32, C.c_uint64]
    both = rule(epilogue, rows, cols, tokens, workspace)
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

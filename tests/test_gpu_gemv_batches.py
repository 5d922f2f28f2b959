"""The lean GEMV where a wave's share is any small number of batches - none, one, the two asked for at once, up to twice as many and one
over -, in every variant of it."""
import numpy as np
import pytest

import nerva_amd as N
import oracle as O
from test_gpu_ops import BF16, F16, REL_L2, dev, rel_l2

pytestmark = pytest.mark.gpu

# rows, columns: one row a wave of one to seven batches (the last workgroup not full), one or two rows, two to four; rows of no whole
# batches, with the norm's row in registers and not
SHAPES = [(1030, 1024), (1030, 2048), (514, 3072), (514, 6144), (258, 8192), (130, 10240), (258, 12288), (66, 14336), (7001, 1024), (13003, 1024),
          (5125, 2048), (11003, 2048), (5005, 1088), (1030, 2624), (514, 3648), (514, 5184)]


@pytest.mark.parametrize("rows,cols", SHAPES)
def test_gemv_of_every_number_of_batches(rows, cols):
    dtype = BF16 if rows % 4 else F16
    rng = np.random.default_rng(rows + cols)
    w = O.synth_16(dtype, 5, 17, 2 * rows * cols, 0.0, 0.02).reshape(2 * rows, cols)
    xf = rng.normal(0, 1, cols).astype(np.float32)
    gamma = O.encode16(dtype, rng.normal(1, 0.1, cols).astype(np.float32))
    res = rng.normal(0, 1, rows).astype(np.float32)
    x16 = O.encode16(dtype, O.rms_norm(dtype, xf, gamma, 1e-6))
    both = O.gemv_x16(dtype, w, x16)
    g, u = both[:rows], both[rows:]
    dw, dx, dxf, dg, dres = dev(w), dev(x16), dev(xf), dev(gamma), dev(res)
    y, y16 = N.DeviceBuffer(rows * 4), N.DeviceBuffer(rows * 2)
    N.gemv(dtype, dw, rows, cols, input16=dx, residual=dres, out_f32=y, epilogue=1)
    assert rel_l2(y.numpy(np.float32), g + res) <= REL_L2
    N.gemv(dtype, dw, rows, cols, input16=dx, out_f32=y)
    assert rel_l2(y.numpy(np.float32), g) <= REL_L2
    if cols > 12288:
        return   # (the norm in front of such rows is the general kernel's)
    N.gemv(dtype, dw, rows, cols, input_f32=dxf, gamma=dg, eps=1e-6, out_f32=y)
    assert rel_l2(y.numpy(np.float32), g) <= REL_L2
    N.gemv(dtype, dw, rows, cols, input_f32=dxf, gamma=dg, eps=1e-6, out16=y16, epilogue=2)
    # one 16-bit rounding of the result, as in the plain 16-bit output
    assert rel_l2(O.decode16(dtype, y16.numpy(np.uint16, rows)), g / (1 + np.exp(-g)) * u) <= 4e-3


@pytest.mark.parametrize("rows,cols", [(1030, 4096), (1030, 6144), (514, 8192), (130, 12288)])
def test_forced_start_up_behind_a_norm_of_any_width(rows, cols):
    """With the exact start-up asked for everywhere, rows behind the norm that do not fit the registers (more than 4096 columns with four waves) are
    normalised whole all the same: bit for bit the launch's without."""
    rng = np.random.default_rng(rows + cols)
    w = O.synth_16(BF16, 5, 17, rows * cols, 0.0, 0.02).reshape(rows, cols)
    xf = rng.normal(0, 1, cols).astype(np.float32)
    gamma = O.encode16(BF16, rng.normal(1, 0.1, cols).astype(np.float32))
    dw, dxf, dg, y = dev(w), dev(xf), dev(gamma), N.DeviceBuffer(rows * 4)
    outs = {}
    try:
        for waves in (4, 16):
            for mode in (2, 1):
                N.Device.set_tuning("gemv_workgroup_waves", waves)
                N.Device.set_tuning("gemv_exact_start", mode)
                N.gemv(BF16, dw, rows, cols, input_f32=dxf, gamma=dg, eps=1e-6, out_f32=y)
                outs[waves, mode] = y.numpy(np.float32).copy()
    finally:
        N.Device.reset_tuning()
    ref = O.gemv_x16(BF16, w, O.encode16(BF16, O.rms_norm(BF16, xf, gamma, 1e-6)))
    for waves in (4, 16):
        assert np.array_equal(outs[waves, 1], outs[waves, 2]) and rel_l2(outs[waves, 1], ref) <= REL_L2

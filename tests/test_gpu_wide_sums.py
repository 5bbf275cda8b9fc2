"""What MFM_STAGE_AUTO moves from the separate kernels to the face sums (FP32
fluxes; boxes that do not fill 64 x 8 tiles) and the Hancock corrector keep
the flux differences in FP64, as the separate kernels form them.

A neutral fluid whose density alternates along x between 2^20 + 1 and 2^-6 at
the supersonic velocity 4: minmod's slopes vanish, so a face's mass flux is the
upwind density times 4, exact in FP32, while the difference over a cell has 27
bits and more.  No rounding but the sum's own can then separate the
structures: the densities agree to the last bit."""
import numpy as np
import pytest

import mfmhd
from helpers import GpuPatch, grid_shape
from test_gpu_parity import periodic_params

pytestmark = pytest.mark.gpu


def update(p, U, lo, vhi, mode, n=1):
    ctx = mfmhd.Context(p)
    ctx.set_stage_kernel(mode)
    ctx.set_timing(True)
    pats = [GpuPatch(U, lo) for _ in range(n)]
    ctx.update_level([(g.fab, mfmhd.Box.of((0, 0, 0), vhi)) for g in pats], 2.0 ** -9, 2.0 ** -4)
    summed = ctx.timing(1, mfmhd.KT_FSUM_PLASMA)[1] > 0
    out = pats[-1].numpy()
    ctx.close()
    return out, summed


@pytest.mark.parametrize("n,boxes,time,mode", [
    ((90, 100, 91), 1, mfmhd.TIME_FIRST_ORDER, mfmhd.STAGE_AUTO),
    ((16, 15, 14), 250, mfmhd.TIME_FIRST_ORDER, mfmhd.STAGE_AUTO),  # a level, blocks of 256
    ((90, 100, 90), 1, mfmhd.TIME_HANCOCK, mfmhd.STAGE_AUTO),
    ((20, 9, 7), 1, mfmhd.TIME_HANCOCK, mfmhd.STAGE_SUMMED),
])
def test_sums_hold_exact_differences(n, boxes, time, mode):
    print("wide sums", n, boxes, time, mode, flush=True)
    p = periodic_params(nf=2, time=time, prec=mfmhd.PREC_FP32_FLUX, gamma=2.0)
    ng, nc = mfmhd.num_ghost_cells(p), mfmhd.num_components(p)
    vhi = tuple(v - 1 for v in n)
    lo, hi, shape = grid_shape(nc, (0, 0, 0), vhi, ng)
    U = np.zeros(shape)
    U[0], U[4], U[5] = 1.0, 2.0, 1.0  # a uniform plasma at rest
    rho = np.where((np.arange(shape[3]) + lo[0]) % 2 == 0, 2.0 ** 20 + 1.0, 2.0 ** -6)
    U[8] = rho
    U[9] = 4.0 * rho
    U[12] = 8.0 * rho + 2.0 ** -10
    a, summed = update(p, U, lo, vhi, mode, boxes)
    b, other = update(p, U, lo, vhi, mfmhd.STAGE_SEPARATE, boxes)
    assert summed and not other
    assert not np.array_equal(b[8], U[8])
    assert np.array_equal(a[8], b[8])

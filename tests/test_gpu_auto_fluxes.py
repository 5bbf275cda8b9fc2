"""MFM_STAGE_AUTO by what a call asks for: with the caller's face fluxes an RK2
call (and an FP64 first-order one) keeps the separate kernels, which are the
faster ones there, whatever its size; without, the face sums from the sizes on
where those are."""
import numpy as np
import pytest

import mfmhd
from helpers import GpuPatch, grid_shape, periodic_fill, smooth_state
from test_gpu_parity import periodic_params

pytestmark = pytest.mark.gpu

RK2, FIRST, HAN = mfmhd.TIME_RK2, mfmhd.TIME_FIRST_ORDER, mfmhd.TIME_HANCOCK
F64, F32 = mfmhd.PREC_FP64, mfmhd.PREC_FP32_FLUX


def run(p, U, lo, vhi, boxes, mode, want_F):
    ctx = mfmhd.Context(p)
    ctx.set_stage_kernel(mode)
    ctx.set_timing(True)
    nc = U.shape[0]
    pats, F = [GpuPatch(U, lo) for _ in range(boxes)], []
    table = []
    for g in pats:
        rec = (g.fab, mfmhd.Box.of((0, 0, 0), vhi))
        if want_F:
            fabs = []
            for d in range(3):
                hi = [vhi[e] + (e == d) for e in range(3)]
                F.append(mfmhd.DeviceArray((nc, hi[2] + 1, hi[1] + 1, hi[0] + 1), zero=True))
                fabs.append(mfmhd.fab(F[-1].ptr, (0, 0, 0), hi, nc))
            rec += (fabs,)
        table.append(rec)
    ctx.update_level(table, 2e-3, 1.0 / 32)
    sums = ctx.timing(1, mfmhd.KT_FSUM_PLASMA)[1] > 0
    out = [pats[-1].numpy()] + [a.numpy() for a in F[-3:]]
    ctx.close()
    return sums, out


@pytest.mark.parametrize("prec,time,nf,n,boxes,sums,sums_F", [
    (F32, RK2, 2, (91, 75, 70), 1, True, False),
    (F32, RK2, 2, (12, 12, 12), 260, True, False),
    (F32, RK2, 4, (91, 75, 70), 1, False, False),
    (F32, RK2, 3, (32, 32, 32), 64, True, False),
    (F32, RK2, 1, (130, 130, 130), 1, False, False),
    (F32, RK2, 2, (64, 64, 64), 1, True, True),  # fills 64 x 8 tiles
    (F32, FIRST, 2, (91, 100, 91), 1, True, True),
    (F32, FIRST, 4, (130, 130, 130), 1, False, False),
    (F32, HAN, 2, (91, 100, 91), 1, True, True),
    (F32, HAN, 4, (130, 130, 130), 1, False, False),
    (F64, RK2, 3, (130, 130, 120), 1, True, False),
    (F64, FIRST, 3, (130, 130, 120), 1, True, False),
    (F64, HAN, 3, (130, 130, 120), 1, True, True),
    (F64, RK2, 2, (130, 130, 120), 1, False, False),
])
def test_structure_by_size_and_outputs(prec, time, nf, n, boxes, sums, sums_F):
    print("auto", prec, time, nf, n, boxes, flush=True)
    p = periodic_params(nf=nf, time=time, prec=prec)
    ng, nc = mfmhd.num_ghost_cells(p), mfmhd.num_components(p)
    vhi = tuple(v - 1 for v in n)
    lo, hi, shape = grid_shape(nc, (0, 0, 0), vhi, ng)
    U = periodic_fill(smooth_state(p, shape, lo, seed=nf), ng)
    assert run(p, U, lo, vhi, boxes, mfmhd.STAGE_AUTO, False)[0] == sums
    used, a = run(p, U, lo, vhi, boxes, mfmhd.STAGE_AUTO, True)
    assert used == sums_F
    if not used:
        for x, y in zip(a, run(p, U, lo, vhi, boxes, mfmhd.STAGE_SEPARATE, True)[1]):
            assert np.array_equal(x, y)

"""The default structure's choice costs a call next to nothing however long
its box is: a tube of a million cells by AUTO (which takes the separate
kernels in 2-D) against the separate kernels themselves."""
import time

import numpy as np
import pytest

import mfmhd
from helpers import GpuPatch, grid_shape
from test_gpu_parity import periodic_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [mfmhd.PREC_FP64, mfmhd.PREC_FP32_FLUX])
def test_choice_on_a_long_tube(prec):
    nx = 1000003
    print("long tube", prec, flush=True)
    p = periodic_params(dims=2, prec=prec)
    lo, hi, shape = grid_shape(8, (0, 0, 0), (nx - 1, 0, 0), 4, 2)
    U = np.zeros(shape)
    U[0], U[4], U[5] = 1.0, 2.0, 0.5
    best, out = {}, {}
    g = {}
    ctxs = {}
    for mode in (mfmhd.STAGE_AUTO, mfmhd.STAGE_SEPARATE):
        ctxs[mode] = mfmhd.Context(p)
        ctxs[mode].set_stage_kernel(mode)
        g[mode] = GpuPatch(U, lo)
        best[mode] = 1e9
    box = mfmhd.Box.of((0, 0, 0), (nx - 1, 0, 0))
    for _ in range(12):
        for mode, ctx in ctxs.items():
            t0 = time.perf_counter()
            ctx.update_state(g[mode].fab, box, 1e-9, 1e-6)
            best[mode] = min(best[mode], time.perf_counter() - t0)
    for mode in ctxs:
        out[mode] = g[mode].numpy()
        ctxs[mode].close()
    assert np.array_equal(out[mfmhd.STAGE_AUTO], out[mfmhd.STAGE_SEPARATE])
    # the search over a million columns took 1.1 to 3.6 ms; a step takes about 1
    assert best[mfmhd.STAGE_AUTO] <= best[mfmhd.STAGE_SEPARATE] + 3e-4, best

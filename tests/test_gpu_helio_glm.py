"""GLM cleaning in the heliospheric box (one fluid): the ghost value of psi is
a constant of the problem like the plasma's, the same in both RK2 stages, so
the three stage structures give the same bits next to the boundary."""
import numpy as np
import pytest

import mfmhd
from helpers import gpu_update, grid_shape
from test_gpu_parity import helio_setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("box", [((0, 0, 0), (15, 15, 15)), ((0, 5, 9), (7, 15, 15))])
@pytest.mark.parametrize("time", [mfmhd.TIME_RK2, mfmhd.TIME_FIRST_ORDER])
def test_psi_ghosts_of_both_stages(oracle_mod, time, box):
    print("helio glm", time, box, flush=True)
    n = 16
    p, dx = helio_setup(oracle_mod, n, 1)
    p.dedner, p.eight_wave, p.time_approx = 1, 0, time
    nc, ng = mfmhd.num_components(p), mfmhd.num_ghost_cells(p)
    lo, hi, shape = grid_shape(nc, (0, 0, 0), (n - 1,) * 3, ng)
    U = oracle_mod.init_problem(p, shape, lo, lo, hi, dx)
    z, y, x = np.meshgrid(*(np.arange(m) for m in shape[1:]), indexing="ij")
    U[8] = 0.1 * np.sin(0.7 * x + 0.4 * y - 0.5 * z)  # psi varies next to every side
    dt = 0.2 * oracle_mod.compute_dt(p, U, lo, (0, 0, 0), (n - 1,) * 3, dx)[0]
    res = []
    for mode in (mfmhd.STAGE_FUSED, mfmhd.STAGE_SEPARATE, mfmhd.STAGE_SUMMED):
        ctx = mfmhd.Context(p)
        ctx.set_dedner(1.3, 0.9)
        ctx.set_stage_kernel(mode)
        res.append(gpu_update(ctx, U, lo, *box, dt, dx, want_F=True))
        assert res[-1]["rc"] == 0
        ctx.close()
    for r in res[1:]:
        assert np.array_equal(r["U"], res[0]["U"])
        assert r["dt"] == res[0]["dt"]
        for a, b in zip(r["F"], res[0]["F"]):
            assert np.array_equal(a, b)

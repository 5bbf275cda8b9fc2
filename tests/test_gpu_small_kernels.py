"""The reduction of a large patch's CFL partials (more than 1024 blocks: the
1024-thread kernel), the periodic fill's component chunks, and the physical
ghost states that an RK2 stage takes over from the one before."""
import numpy as np
import pytest

import mfmhd
from helpers import GpuPatch, grid_shape, periodic_fill, smooth_state
from test_gpu_parity import check64, helio_setup, periodic_params, run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(128, 64, 32), (128, 64, 33), (131, 67, 61)])
@pytest.mark.parametrize("uniform", [False, True])
def test_dt_of_many_blocks(oracle_mod, n, uniform):
    """Below and above 1024 blocks of 256 cells; a uniform state's minimum is
    its first cell."""
    p = periodic_params(nf=1)
    lo, hi, shape = grid_shape(8, (0, 0, 0), tuple(v - 1 for v in n), 4)
    U = smooth_state(p, shape, lo, seed=sum(n))
    if uniform:
        U[:] = U[:, 5:6, 5:6, 5:6]
    vhi = tuple(v - 1 for v in n)
    ctx = mfmhd.Context(p)
    g = GpuPatch(U, lo)  # holds the device memory during the call
    dt, cell = ctx.compute_dt(g.fab, mfmhd.Box.of((0, 0, 0), vhi), 0.05)
    want, wcell = oracle_mod.compute_dt(p, U, lo, (0, 0, 0), vhi, 0.05)
    assert abs(dt - want) <= 1e-14 * want
    assert tuple(cell) == ((0, 0, 0) if uniform else tuple(wcell))
    ctx.close()


@pytest.mark.parametrize("nf,ded", [(1, False), (1, True), (2, False), (3, True), (4, False), (4, True)])
def test_periodic_fill_chunks(nf, ded):
    p = periodic_params(nf=nf, dedner=ded, eight=not ded)
    nc = mfmhd.num_components(p)
    lo, hi, shape = grid_shape(nc, (0, 0, 0), (6, 2, 8), 4)
    U = np.random.default_rng(nf).uniform(1, 2, shape)
    g = GpuPatch(U, lo)
    ctx = mfmhd.Context(p)
    ctx.fill_periodic(g.fab, mfmhd.Box.of((0, 0, 0), (6, 2, 8)))
    assert np.array_equal(g.numpy(), periodic_fill(U.copy(), 4))
    ctx.close()


@pytest.mark.parametrize("nf", [1, 2, 3, 4])
@pytest.mark.parametrize("time", [mfmhd.TIME_RK2, mfmhd.TIME_HANCOCK, mfmhd.TIME_FIRST_ORDER])
def test_ghosts_between_stages(oracle_mod, nf, time):
    """Patches on corners, edges and faces of the heliospheric box: constant
    ghosts (plasma, first population) and copied ones (the others), every
    scheme; after an update elsewhere the same context starts from its own
    ghosts again."""
    n = 16
    p, dx = helio_setup(oracle_mod, n, nf)
    p.time_approx = time
    ng, nc = mfmhd.num_ghost_cells(p), mfmhd.num_components(p)
    for vlo, vhi in (((0, 0, 0), (5, 6, 7)), ((9, 0, 4), (15, 15, 9)), ((4, 5, 11), (12, 9, 15))):
        lo, hi, shape = grid_shape(nc, vlo, vhi, ng)
        U = oracle_mod.init_problem(p, shape, lo, lo, hi, dx)
        U[:, ng:-ng, ng:-ng, ng:-ng] *= 1.01
        dt = 0.2 * oracle_mod.compute_dt(p, U, lo, vlo, vhi, dx)[0]
        g, o = run_pair(oracle_mod, p, U, lo, vlo, vhi, dt, dx)
        check64(g, o, lo, vlo, vhi, U_in=U)

"""The face kernels take the faces of every direction from one list: sizes
around their block sizes (64 boundary faces, 256 interior faces), patch
tables whose patches have boundary faces in some directions only, and the
limiter paths, against the oracle."""
import numpy as np
import pytest

import mfmhd
from helpers import GpuPatch, gpu_update, grid_shape, smooth_state
from test_gpu_parity import check64, helio_setup, periodic_params, run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vhi", [(62, 0, 0), (63, 1, 0), (64, 2, 2), (0, 64, 3), (2, 3, 63),
                                 (254, 0, 1), (255, 1, 0), (15, 16, 17)])
@pytest.mark.parametrize("lim", [mfmhd.LIM_MINMOD, mfmhd.LIM_VANLEER, mfmhd.LIM_MC])
def test_interior_faces_at_block_edges(oracle_mod, vhi, lim):
    print("faces", vhi, lim, flush=True)
    p = periodic_params(nf=3, flux=mfmhd.FLUX_ROE8, lim=lim)
    ng, nc = mfmhd.num_ghost_cells(p), mfmhd.num_components(p)
    lo, hi, shape = grid_shape(nc, (0, 0, 0), vhi, ng)
    U = smooth_state(p, shape, lo, seed=sum(vhi))
    g, o = run_pair(oracle_mod, p, U, lo, (0, 0, 0), vhi, 0.004, 0.05)
    check64(g, o, lo, (0, 0, 0), vhi, U_in=U)


@pytest.mark.parametrize("n", [8, 9, 16])
def test_boundary_faces_of_a_table(oracle_mod, n):
    """A 2 x 2 x 2 tiling of the heliospheric box (each patch on three of the
    six sides) with one inner patch more (no boundary face at all): the level
    call equals the single patches bit for bit, and those the oracle."""
    p, dx = helio_setup(oracle_mod, 2 * n, 4)
    ng, nc = mfmhd.num_ghost_cells(p), mfmhd.num_components(p)
    boxes = [(tuple(n * q for q in c), tuple(n * q + n - 1 for q in c))
             for c in np.ndindex(2, 2, 2)] + [((4, 4, 4), (n - 2, n - 1, n))]
    ctx = mfmhd.Context(p)
    dt = None
    want, pats = [], []
    for vlo, vhi in boxes:
        lo, hi, shape = grid_shape(nc, vlo, vhi, ng)
        U = oracle_mod.init_problem(p, shape, lo, lo, hi, dx)
        if dt is None:
            dt = 0.3 * oracle_mod.compute_dt(p, U, lo, vlo, vhi, dx)[0]
        g = gpu_update(ctx, U, lo, vlo, vhi, dt, dx)
        check64(g, oracle_mod.patch_update(p, U, lo, vlo, vhi, dt, dx), lo, vlo, vhi, U_in=U)
        want.append(g["U"])
        pats.append(GpuPatch(U, lo))
    ctx.update_level([(g.fab, mfmhd.Box.of(*b)) for g, b in zip(pats, boxes)], dt, dx)
    mfmhd.synchronize()
    for q, (g, w) in enumerate(zip(pats, want)):
        assert np.array_equal(g.numpy(), w), q
    ctx.close()

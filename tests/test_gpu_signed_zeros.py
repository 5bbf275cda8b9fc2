"""Quotients over a shared reciprocal keep the sign that a division gives a
zero: the zero face fluxes of a field-free, one-dimensional flow (HLLC: the
transverse momentum over the wave speed's distance to the contact, of either
sign) carry the oracle's signs."""
import numpy as np
import pytest

import mfmhd
from helpers import grid_shape, periodic_fill
from test_gpu_parity import periodic_params, run_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lim", [mfmhd.LIM_MINMOD, mfmhd.LIM_VANLEER])
def test_hllc_zero_fluxes(oracle_mod, lim):
    print("signed zeros", lim, flush=True)
    p = periodic_params(nf=2, flux=mfmhd.FLUX_HLLC, lim=lim, time=mfmhd.TIME_RK2)
    ng, nc = mfmhd.num_ghost_cells(p), mfmhd.num_components(p)
    vhi = (11, 9, 7)
    lo, hi, shape = grid_shape(nc, (0, 0, 0), vhi, ng)
    r = np.random.default_rng(3)
    U = np.zeros(shape)
    rho = r.uniform(0.5, 1.5, shape[1:])
    vx, by = (np.round(r.uniform(-1.4, 1.4, shape[1:])) for _ in range(2))
    U[0], U[1], U[5], U[6] = rho, rho * vx, 0.75, by
    U[2], U[7], U[10] = -0.0, -0.0, -0.0
    U[4] = 1.5 + 0.5 * rho * vx * vx + (U[5] ** 2 + by * by) / (8 * np.pi)
    U[8], U[9], U[12] = 0.5 * rho, 0.5 * rho * vx, 1.5 + 0.25 * rho * vx * vx
    periodic_fill(U, ng)
    g, o = run_pair(oracle_mod, p, U, lo, (0, 0, 0), vhi, 1e-3, 1.0 / 16, want_F=True)
    for a, b in zip(g["F"], o["F"]):
        zero = (a == 0) & (b == 0)
        assert zero.sum() > 500
        assert np.array_equal(np.signbit(a[zero]), np.signbit(b[zero]))

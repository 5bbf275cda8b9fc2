"""The FP32-flux build's plasma and neutral face fluxes where their selects
change sides: fluid at rest, no field, a field along one axis, flow faster than
the fast wave either way, a uniform state.  One first-order step's face
fluxes against the oracle's FP64 ones; states are of order one, so a flux
component's error is bounded by 2e-5 max(1, max |F|) (some 300 FP32
roundings).  A NaN in the second ghost layer reaches the same cells as in
the FP64 build."""
import numpy as np
import pytest

import mfmhd
from helpers import gpu_update, grid_shape, smooth_state
from test_gpu_parity import periodic_params

pytestmark = pytest.mark.gpu

KINDS = ["smooth", "rest", "hydro", "fast+", "fast-", "axial", "uniform"]


def state(p, shape, lo, kind):
    U = smooth_state(p, shape, lo, seed=5)
    g1 = p.gamma - 1.0
    rho = U[0]
    v = [U[1 + d] / rho for d in range(3)]
    B = [U[5 + d].copy() for d in range(3)]
    pr = g1 * (U[4] - 0.5 * rho * sum(q * q for q in v) - sum(b * b for b in B) / (8 * np.pi))
    if kind == "rest":
        v = [0.0 * q for q in v]
    elif kind == "hydro":
        B = [0.0 * b for b in B]
    elif kind in ("fast+", "fast-"):
        v[0] = v[0] + (12.0 if kind == "fast+" else -12.0)
    elif kind == "axial":
        v, B = [0.0 * v[0], v[1], 0.0 * v[2]], [B[0], 0.0 * B[1], 0.0 * B[2]]
    elif kind == "uniform":
        rho, pr = 0.0 * rho + 1.25, 0.0 * pr + 0.75
        v = [0.0 * rho + q for q in (0.5, -0.25, 0.0)]
        B = [0.0 * rho + q for q in (1.0, 0.5, -2.0)]
    U[0] = rho
    for d in range(3):
        U[1 + d], U[5 + d] = rho * v[d], B[d]
    U[4] = pr / g1 + 0.5 * rho * sum(q * q for q in v) + sum(b * b for b in B) / (8 * np.pi)
    return U


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("flux,lim", [(mfmhd.FLUX_ROE8, mfmhd.LIM_MINMOD),
                                      (mfmhd.FLUX_ROE8_ROEAVG, mfmhd.LIM_VANLEER),
                                      (mfmhd.FLUX_ROE7, mfmhd.LIM_MINMOD),
                                      (mfmhd.FLUX_RUSANOV_ROEAVG, mfmhd.LIM_VANLEER),
                                      (mfmhd.FLUX_HLLC, mfmhd.LIM_MINMOD)])
def test_fluxes_in_fp32(oracle_mod, kind, flux, lim):
    print("flux32", kind, flux, lim, flush=True)
    p = periodic_params(nf=2, flux=flux, lim=lim, time=mfmhd.TIME_FIRST_ORDER,
                        prec=mfmhd.PREC_FP32_FLUX)
    vlo, vhi = (0, 0, 0), (17, 8, 6)
    ng, nc = mfmhd.num_ghost_cells(p), mfmhd.num_components(p)
    lo, hi, shape = grid_shape(nc, vlo, vhi, ng)
    U = state(p, shape, lo, kind)
    o = oracle_mod.patch_update(p, U, lo, vlo, vhi, 1e-3, 0.05, 0.0, want_F=True)
    for mode in (mfmhd.STAGE_SEPARATE, mfmhd.STAGE_SUMMED):
        ctx = mfmhd.Context(p)
        ctx.set_stage_kernel(mode)
        g = gpu_update(ctx, U, lo, vlo, vhi, 1e-3, 0.05, 0.0, want_F=True)
        ctx.close()
        assert g["rc"] == 0 and o["rc"] == 0
        for d in range(3):
            for c in range(nc):
                a, b = g["F"][d][c], o["F"][d][c]
                assert np.abs(a - b).max() <= 2e-5 * max(1.0, np.abs(b).max()), (mode, d, c)


@pytest.mark.parametrize("lim", [mfmhd.LIM_MINMOD, mfmhd.LIM_VANLEER])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("side", [-1, 1])
def test_nan_ghosts_are_not_limited_away(lim, axis, side):
    print("nan ghost", lim, axis, side, flush=True)
    vlo, vhi = (0, 0, 0), (9, 8, 7)
    seen = []
    for prec in (mfmhd.PREC_FP64, mfmhd.PREC_FP32_FLUX):
        p = periodic_params(nf=2, lim=lim, time=mfmhd.TIME_FIRST_ORDER, prec=prec)
        ng, nc = mfmhd.num_ghost_cells(p), mfmhd.num_components(p)
        lo, hi, shape = grid_shape(nc, vlo, vhi, ng)
        U = smooth_state(p, shape, lo, seed=9)
        at = [4 - lo[2], 4 - lo[1], 4 - lo[0]]
        at[2 - axis] = (vlo[axis] - 2 if side < 0 else vhi[axis] + 2) - lo[axis]
        for c in (1, 2, 3, 9, 10, 11):
            U[(c,) + tuple(at)] = np.nan
        for mode in (mfmhd.STAGE_SEPARATE, mfmhd.STAGE_SUMMED):
            ctx = mfmhd.Context(p)
            ctx.set_stage_kernel(mode)
            g = gpu_update(ctx, U, lo, vlo, vhi, 1e-3, 0.05)
            ctx.close()
            inner = g["U"][:, ng:-ng, ng:-ng, ng:-ng]
            seen.append((g["rc"], np.isnan(inner)))
    for rc, bad in seen[1:]:
        assert rc == seen[0][0]
        assert np.array_equal(bad, seen[0][1])

"""The face-sum tile kernels beyond their 64-wide tiles: any box shape, the
FP64 build and the Hancock corrector, against the separate kernels.

FP64: the tile kernels apply the directions in the separate kernels' order
with the same arithmetic per face, so states, fluxes, div(B), dt and its cell
agree to the last bit.  FP32 fluxes: they add the directions' differences
first and store the sum in FP32 (agree's 1e-6 per component on smooth
states)."""
import numpy as np
import pytest

import mfmhd
from helpers import GpuPatch, gpu_update, grid_shape, periodic_fill, smooth_state
from test_gpu_fused import agree, both
from test_gpu_parity import helio_setup, periodic_params

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (8, 8, 8), (12, 11, 5), (20, 21, 9), (31, 17, 3), (33, 16, 2), (36, 37, 4),
          (64, 9, 3), (65, 8, 7), (130, 3, 2), (17, 70, 1), (256, 2, 2), (300, 1, 3)]


def state(p, shape3, seed):
    nc, ng = mfmhd.num_components(p), mfmhd.num_ghost_cells(p)
    vhi = tuple(v - 1 for v in shape3)
    lo, hi, shape = grid_shape(nc, (0, 0, 0), vhi, ng)
    return periodic_fill(smooth_state(p, shape, lo, seed=seed), ng), lo, vhi


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("time", [mfmhd.TIME_RK2, mfmhd.TIME_HANCOCK])
@pytest.mark.parametrize("prec", [mfmhd.PREC_FP64, mfmhd.PREC_FP32_FLUX])
def test_tile_shapes(shape, time, prec):
    print("tile", shape, time, prec, flush=True)
    p = periodic_params(nf=3, time=time, prec=prec)
    U, lo, vhi = state(p, shape, sum(shape))
    a, b = both(p, U, lo, (0, 0, 0), vhi, 2e-3, 1.0 / 32, tz=3, mode=mfmhd.STAGE_SUMMED)
    agree(a, b, prec == mfmhd.PREC_FP64)


@pytest.mark.parametrize("lim", [mfmhd.LIM_VANLEER, mfmhd.LIM_KOREN])
@pytest.mark.parametrize("flux,ded", [(mfmhd.FLUX_ROE8, False), (mfmhd.FLUX_RUSANOV, False),
                                      (mfmhd.FLUX_HLLC, True), (mfmhd.FLUX_ROE8, True)])
def test_tile_solvers_fp64(lim, flux, ded):
    p = periodic_params(nf=2, flux=flux, lim=lim, dedner=ded, eight=not ded)
    U, lo, vhi = state(p, (37, 22, 6), 4)
    a, b = both(p, U, lo, (0, 0, 0), vhi, 2e-3, 1.0 / 32, tz=4, ch=(1.3, 0.9) if ded else None,
                mode=mfmhd.STAGE_SUMMED)
    agree(a, b, True)


@pytest.mark.parametrize("time", [mfmhd.TIME_RK2, mfmhd.TIME_HANCOCK])
def test_tiles_with_boundary_faces_fp64(oracle_mod, time):
    """Every side of the heliospheric box, and sub-patches on some of them."""
    n = 22
    p, dx = helio_setup(oracle_mod, n, 4)
    p.time_approx = time
    nc, ng = mfmhd.num_components(p), mfmhd.num_ghost_cells(p)
    vlo, vhi = (0, 0, 0), (n - 1,) * 3
    lo, hi, shape = grid_shape(nc, vlo, vhi, ng)
    U = oracle_mod.init_problem(p, shape, lo, lo, hi, dx)
    dt = 0.2 * oracle_mod.compute_dt(p, U, lo, vlo, vhi, dx)[0]
    for box in ((vlo, vhi), ((3, 0, 9), (21, 17, 21)), ((0, 10, 12), (7, 21, 21))):
        a, b = both(p, U, lo, *box, dt, dx, tz=5, mode=mfmhd.STAGE_SUMMED)
        agree(a, b, True)


def test_auto_takes_small_tiles_for_a_level():
    """A level of 12^3 boxes with 2/3 million cells: the default takes the
    tile kernels (in blocks of 256 threads), within 1e-6 of the separate
    ones."""
    p = periodic_params(nf=2, prec=mfmhd.PREC_FP32_FLUX)
    U, lo, vhi = state(p, (12, 12, 12), 8)
    n = 390
    res = {}
    for mode in (mfmhd.STAGE_AUTO, mfmhd.STAGE_SEPARATE):
        ctx = mfmhd.Context(p)
        ctx.set_stage_kernel(mode)
        ctx.set_timing(True)
        pats = [GpuPatch(U * (1.0 + 1e-3 * (q % 7)), lo) for q in range(n)]
        ctx.update_level([(g.fab, mfmhd.Box.of((0, 0, 0), vhi)) for g in pats], 2e-3, 1.0 / 32)
        used = ctx.timing(1, mfmhd.KT_FSUM_PLASMA)[1]
        assert (used > 0) == (mode == mfmhd.STAGE_AUTO)
        res[mode] = [pats[q].numpy() for q in (0, 5, 191, n - 1)]
        ctx.close()
    for x, y in zip(res[mfmhd.STAGE_AUTO], res[mfmhd.STAGE_SEPARATE]):
        for c in range(y.shape[0]):
            assert np.max(np.abs(x[c] - y[c])) <= 1e-6 * np.max(np.abs(y[c])), c

"""Characteristic slopes on large patches walk the faces of y and z per thread
and pass the x faces' states between lanes; the same update cut into slabs
small enough for the face-per-thread kernel gives the same bits."""
import numpy as np
import pytest

import mfmhd
from helpers import GpuPatch, grid_shape, periodic_fill, smooth_state
from test_gpu_parity import periodic_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,time,ded,flux", [
    ((131, 97, 65), mfmhd.TIME_HANCOCK, False, mfmhd.FLUX_ROE8),   # 4 faces per thread
    ((64, 131, 97), mfmhd.TIME_RK2, True, mfmhd.FLUX_ROE8),
    ((63, 127, 101), mfmhd.TIME_RK2, False, mfmhd.FLUX_HLLC),
    ((190, 149, 145), mfmhd.TIME_HANCOCK, False, mfmhd.FLUX_RUSANOV),  # 8
    ((1100, 733, 1), mfmhd.TIME_RK2, True, mfmhd.FLUX_HLLC),       # 2-D
])
@pytest.mark.parametrize("tvd", [0, 1])
def test_walked_faces_equal_single_ones(n, time, ded, flux, tvd):
    print("walk", n, time, ded, flux, tvd, flush=True)
    dims = 3 if n[2] > 1 else 2
    p = periodic_params(nf=1, flux=flux, lim=mfmhd.LIM_VANLEER, dims=dims, dedner=ded,
                        eight=not ded, time=time)
    p.char_reconstruction = 1
    p.check_tvd = tvd
    ng, nc = mfmhd.num_ghost_cells(p), mfmhd.num_components(p)
    vhi = tuple(v - 1 for v in n)
    lo, hi, shape = grid_shape(nc, (0, 0, 0), vhi, ng, dims)
    U = periodic_fill(smooth_state(p, shape, lo, seed=sum(n)), ng, dims)
    ctx = mfmhd.Context(p)
    if ded:
        ctx.set_dedner(1.3, 0.9)
    g = GpuPatch(U, lo)
    dt, cell = ctx.update_state(g.fab, mfmhd.Box.of((0, 0, 0), vhi), 1e-3, 1.0 / 32)
    whole = g.numpy()
    top = dims - 1
    per = n[0] * n[1] if dims == 3 else n[0]
    thick = max(1, int(2.4e5 // per))
    dts = []
    for k in range(0, n[top], thick):
        a, b = [0, 0, 0], list(vhi)
        a[top], b[top] = k, min(k + thick, n[top]) - 1
        s = GpuPatch(U, lo)
        d, _ = ctx.update_state(s.fab, mfmhd.Box.of(a, b), 1e-3, 1.0 / 32)
        dts.append(d)
        part = s.numpy()
        cut = [slice(None)] * 4
        cut[3 - top] = slice(a[top] - lo[top], b[top] - lo[top] + 1)
        inner = [slice(None)] * 4
        for d2 in range(dims):
            if d2 != top:
                inner[3 - d2] = slice(ng, -ng)
        x, y = whole[tuple(cut)], part[tuple(cut)]
        assert np.array_equal(x[tuple(inner)], y[tuple(inner)])
    assert dt == min(dts)
    ctx.close()

"""Host buffers of more than 4 MB go through the pinned copy pipeline (chunks
of 2 MB over four threads) and only the planes of the valid box come back:
the same bits as the device entry point, ghost cells and buffers around the
state untouched, several calls and sizes through one context."""
import numpy as np
import pytest

import mfmhd
from helpers import gpu_update, grid_shape, smooth_state
from test_gpu_parity import periodic_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,n,nf,time", [
    (3, (49, 33, 41), 1, mfmhd.TIME_RK2),        # 7.3 MB, chunks cut components
    (3, (64, 60, 24), 4, mfmhd.TIME_HANCOCK),    # 28 MB
    (3, (120, 120, 1), 2, mfmhd.TIME_FIRST_ORDER),
    (2, (700, 90, 1), 1, mfmhd.TIME_RK2),        # 2-D: rows instead of planes
    (3, (20, 20, 20), 1, mfmhd.TIME_RK2),        # below the pipeline's size
])
def test_pipeline_equals_device(dims, n, nf, time):
    print("host pipeline", dims, n, nf, time, flush=True)
    p = periodic_params(nf=nf, dims=dims, time=time)
    ng, nc = mfmhd.num_ghost_cells(p), mfmhd.num_components(p)
    vhi = tuple(v - 1 for v in n)
    lo, hi, shape = grid_shape(nc, (0, 0, 0), vhi, ng, dims)
    ctx, ref = mfmhd.Context(p), mfmhd.Context(p)
    guard = 4096
    for call in range(3):
        U = smooth_state(p, shape, lo, seed=10 * sum(n) + call)
        room = np.full(U.size + 2 * guard, 7.0)
        V = room[guard:guard + U.size].reshape(shape)
        V[...] = U
        dt, cell = ctx.update_state_host(V, lo, mfmhd.Box.of((0, 0, 0), vhi), 2e-3, 1.0 / 32)
        want = gpu_update(ref, U, lo, (0, 0, 0), vhi, 2e-3, 1.0 / 32)
        assert np.array_equal(V, want["U"])
        assert dt == want["dt"] and cell == want["cell"]
        assert np.all(room[:guard] == 7.0) and np.all(room[-guard:] == 7.0)
    ctx.close()
    ref.close()

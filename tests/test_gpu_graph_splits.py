"""Replayed launches (mfm_ctx_set_graphs) over boxes whose lists have the same
lengths but begin their directions elsewhere: a box and its permutations in
turn through one context, each against eager launches."""
import numpy as np
import pytest

import mfmhd
from helpers import gpu_update, grid_shape, periodic_fill, smooth_state
from test_gpu_parity import periodic_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [mfmhd.PREC_FP64, mfmhd.PREC_FP32_FLUX])
@pytest.mark.parametrize("time", [mfmhd.TIME_RK2, mfmhd.TIME_HANCOCK])
def test_permuted_boxes(time, prec):
    print("graph splits", time, prec, flush=True)
    p = periodic_params(nf=2, time=time, prec=prec)
    nc, ng = mfmhd.num_components(p), mfmhd.num_ghost_cells(p)
    graph, eager = mfmhd.Context(p), mfmhd.Context(p)
    graph.set_graphs(True)
    for ctx in (graph, eager):
        ctx.set_stage_kernel(mfmhd.STAGE_SEPARATE)
    for turn, n in enumerate([(16, 32, 64), (64, 32, 16), (64, 32, 16), (32, 64, 16), (16, 32, 64)]):
        vhi = tuple(v - 1 for v in n)
        lo, hi, shape = grid_shape(nc, (0, 0, 0), vhi, ng)
        U = periodic_fill(smooth_state(p, shape, lo, seed=turn), ng)
        a = gpu_update(graph, U, lo, (0, 0, 0), vhi, 2e-3, 1.0 / 32)
        b = gpu_update(eager, U, lo, (0, 0, 0), vhi, 2e-3, 1.0 / 32)
        assert np.array_equal(a["U"], b["U"]), n
        assert a["dt"] == b["dt"] and a["cell"] == b["cell"]
    graph.close()
    eager.close()

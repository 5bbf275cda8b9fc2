"""Ghost copies of large boxes: rectangles whose mean size takes the exchange
in large blocks, and periodic fills of more than 2048 blocks, where a thread
takes the component chunks one after the other; one and several chunks, in 3-D
and 2-D."""
import numpy as np
import pytest

import mfmhd
from fill_layouts import grown, level_params, split
from helpers import GpuPatch, grid_shape, periodic_fill
from test_gpu_fill import same, to_dev
from test_gpu_parity import periodic_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,n,parts,nf", [
    (3, (128, 64, 64), (2, 1, 1), 4),   # two boxes of 64^3
    (3, (71, 67, 69), (1, 1, 1), 2),    # one box, periodic onto itself
    (2, (4096, 2050, 1), (1, 1, 1), 1),  # rows of 4096 cells
    (3, (96, 48, 48), (2, 1, 1), 1),    # just below: small blocks
])
def test_exchange_of_large_boxes(oracle_mod, dims, n, parts, nf):
    print("large exchange", dims, n, parts, nf, flush=True)
    boxes = split(n, parts, dims)
    p = level_params(n, dims, (1, 1, 1), nfluids=nf)
    nc, ng = mfmhd.num_components(p), 4
    rng = np.random.default_rng(sum(n))
    arrs, los = [], []
    for b in boxes:
        lo, hi = grown(b, ng, dims)
        arrs.append(rng.uniform(1, 2, (nc, hi[2] - lo[2] + 1, hi[1] - lo[1] + 1, hi[0] - lo[0] + 1)))
        los.append(lo)
    devs, fabs = to_dev(arrs, los, nc)
    ctx = mfmhd.Context(p)
    plan = mfmhd.FillPlan(p, boxes, interp_radius=ng)
    for _ in range(2):
        ctx.exchange(plan, fabs)
    oracle_mod.level_exchange(p, boxes, arrs, los, ng)
    for d, a in zip(devs, arrs):
        assert same(d.numpy(), a)
    plan.close()
    ctx.close()


@pytest.mark.parametrize("dims,n,nf,ded", [
    (3, (83, 79, 71), 4, True),       # 24 components, below 2048 blocks
    (3, (91, 83, 89), 4, True),       # above
    (3, (91, 83, 89), 1, False),
    (2, (1021, 701, 1), 3, False),
])
def test_periodic_fill_of_large_boxes(dims, n, nf, ded):
    print("large periodic fill", dims, n, nf, flush=True)
    p = periodic_params(nf=nf, dims=dims, dedner=ded, eight=not ded)
    nc = mfmhd.num_components(p)
    vhi = tuple(v - 1 for v in n)
    lo, hi, shape = grid_shape(nc, (0, 0, 0), vhi, 4, dims)
    U = np.random.default_rng(nf).uniform(1, 2, shape)
    g = GpuPatch(U, lo)
    ctx = mfmhd.Context(p)
    ctx.fill_periodic(g.fab, mfmhd.Box.of((0, 0, 0), vhi))
    assert np.array_equal(g.numpy(), periodic_fill(U.copy(), 4, dims))
    ctx.close()

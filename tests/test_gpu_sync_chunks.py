"""The synchronisation and ghost-fill kernels take the components in chunks
(4 per thread in the register and average, 8 in the copies): every component
count, both refinement ratios' paths and 2-D, against the oracle or the exact
average."""
import numpy as np
import pytest

import mfmhd
from fill_layouts import level_params, split
from sync_layouts import COARSE, FINE, R, cell_fabs, face_fabs, params
from test_gpu_sync import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nf", [1, 2, 3, 4])
def test_register_chunks(oracle_mod, nf):
    p = params(nf)
    nc = mfmhd.num_components(p)
    rng = np.random.default_rng(nf)
    ctx = mfmhd.Context(p)
    reg = mfmhd.FluxRegister(p, FINE, COARSE, R)
    oreg = oracle_mod.FluxRegister(p, FINE, COARSE, R, nc)
    cfab, clos = cell_fabs(COARSE, rng.uniform(1, 2, (nc, 16, 16, 16)))
    ffab, flos = cell_fabs(FINE, rng.uniform(1, 2, (nc, 32, 32, 32)))
    dUc, fUc = to_dev(cfab, clos, nc)
    dUf, fUf = to_dev(ffab, flos, nc)
    reg.set_zero(ctx)
    oreg.R[:] = 0.0
    fc, fclos = face_fabs(COARSE, [rng.standard_normal((nc, 16, 16, 16)) for _ in range(3)])
    ff, fflos = face_fabs(FINE, [rng.standard_normal((nc, 32, 32, 32)) for _ in range(3)])
    dC, fC = to_dev(fc, fclos, nc)
    dF, fF = to_dev(ff, fflos, nc)
    reg.increment_coarse(ctx, fC, 0.013)
    oreg.increment_coarse(fc, fclos, 0.013)
    reg.increment_fine(ctx, fF, 0.007)
    oreg.increment_fine(ff, fflos, 0.007)
    reg.reflux(ctx, fUc, -1.0, 1.0 / 16)
    oreg.reflux(cfab, clos, -1.0, 1.0 / 16)
    reg.average_down(ctx, fUc, fUf, 1.0 / 32)
    oreg.average_down(cfab, clos, ffab, flos, 1.0 / 32)
    for d, a in zip(dUc, cfab):
        assert np.array_equal(d.numpy(), a)


@pytest.mark.parametrize("dims,r,nf", [(3, 2, 1), (3, 2, 4), (3, 4, 2), (2, 2, 1), (2, 2, 4),
                                       (2, 4, 3)])
def test_average_down_ratios(dims, r, nf):
    """The average of r^dims children, formed as sum(vol x) / sum(vol) with
    vol a power of two: within (r^dims + 2) rounding errors of the mean."""
    nz = 8 if dims == 3 else 1
    n = (8, 8, nz)
    cb = split(n, (2, 2, 1), dims) if dims == 3 else [((0, 0, 0), (3, 7, 0)), ((4, 0, 0), (7, 7, 0))]
    fhi = tuple((v * r - 1) if d < dims else 0 for d, v in enumerate((6, 5, 4)))
    flo = tuple(r if d < dims else 0 for d in range(3))
    fine = [(flo, fhi)]
    fn = tuple(n[d] * r if d < dims else 1 for d in range(3))
    p = level_params(fn, dims, (1, 1, 1), nfluids=nf)
    nc = mfmhd.num_components(p)
    rng = np.random.default_rng(10 * r + nf)
    Uc = rng.uniform(1, 2, (nc, n[2], n[1], n[0]))
    Uf = rng.uniform(1, 2, (nc, fn[2], fn[1], fn[0]))
    cfab, clos = cell_fabs(cb, Uc)
    ffab, flos = cell_fabs(fine, Uf)
    dUc, fUc = to_dev(cfab, clos, nc)
    dUf, fUf = to_dev(ffab, flos, nc)
    ctx = mfmhd.Context(p)
    reg = mfmhd.FluxRegister(p, fine, cb, r)
    reg.average_down(ctx, fUc, fUf, 1.0 / 64)
    rz = r if dims == 3 else 1
    want = Uf.reshape(nc, n[2], rz, n[1], r, n[0], r).mean(axis=(2, 4, 6))
    inside = np.zeros((n[2], n[1], n[0]), bool)
    lo = [1 if d < dims else 0 for d in range(3)]
    hi = [(v + 1) // r - 1 if d < dims else 0 for d, v in enumerate(fhi)]
    inside[lo[2]:hi[2] + 1, lo[1]:hi[1] + 1, lo[0]:hi[0] + 1] = True
    ref = np.where(inside, want, Uc)
    for d, (blo, bhi) in zip(dUc, cb):
        got = d.numpy()
        w = ref[:, blo[2]:bhi[2] + 1, blo[1]:bhi[1] + 1, blo[0]:bhi[0] + 1]
        m = inside[blo[2]:bhi[2] + 1, blo[1]:bhi[1] + 1, blo[0]:bhi[0] + 1]
        assert np.array_equal(got[:, ~m], w[:, ~m])
        np.testing.assert_allclose(got, w, rtol=(r ** dims + 2) * 2.3e-16)

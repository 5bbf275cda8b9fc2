"""Requests with different plasma limiters on one server: each keeps its own
limiter, alone and in any mix, bit for bit, in every stage structure (a launch
of the tile kernels has one limiter instance for all its patches); and what an
FP64 or Hancock request is charged does not grow with the summed structure,
which runs the separate kernels there."""
import numpy as np
import pytest

import mfmhd
from test_serve import req_params, request_charge, run_until_done, swlism_req

pytestmark = pytest.mark.gpu

LIMS = (mfmhd.LIM_MINMOD, mfmhd.LIM_VANLEER, mfmhd.LIM_MC)


def request(kind, n, lim, prec):
    if kind == "swlism":
        p, dx = swlism_req(n, prec=prec)
    else:
        p, dx = req_params(n // 4, prec=prec)
        if kind == "hancock":
            p.time_approx = mfmhd.TIME_HANCOCK
    for v in range(8):
        p.limiter[v] = lim
    return p, dx


def serve(mode, reqs):
    srv = mfmhd.Server(reqs[0][0], 8 << 30)
    srv.set_stage_kernel(mode)
    ids = [srv.submit(p, dx, 3, 0.25) for p, dx in reqs]
    run_until_done(srv, lambda: ids)
    out = []
    for q in ids:
        assert srv.info(q)["state"] == mfmhd.REQ_DONE, srv.error(q)
        out.append((srv.fetch(q), srv.info(q)["t"]))
    srv.close()
    return out


@pytest.mark.parametrize("mode", [mfmhd.STAGE_SUMMED, mfmhd.STAGE_FUSED, mfmhd.STAGE_SEPARATE])
@pytest.mark.parametrize("kind,prec", [("swlism", mfmhd.PREC_FP32_FLUX), ("swlism", mfmhd.PREC_FP64),
                                       ("helio", mfmhd.PREC_FP32_FLUX),
                                       ("hancock", mfmhd.PREC_FP32_FLUX)])
def test_limiters_stay_with_their_requests(kind, prec, mode):
    print("limiters", kind, prec, mode, flush=True)
    reqs = [request(kind, 48 + 8 * q, lim, prec) for q, lim in enumerate(LIMS)]
    alone = [serve(mode, [r])[0] for r in reqs]
    # the limiters act: another limiter is another result
    other = serve(mode, [request(kind, 48, mfmhd.LIM_VANLEER, prec)])[0]
    assert not np.array_equal(other[0], alone[0][0])
    for order in ((0, 1, 2), (1, 2, 0), (2, 0, 1)):
        for q, (U, t) in zip(order, serve(mode, [reqs[q] for q in order])):
            assert np.array_equal(U, alone[q][0]), (order, q)
            assert t == alone[q][1]


def test_summed_structure_keeps_the_charge_of_fp64_requests():
    """Room for two FP64 requests by the separate kernels' charge: two run."""
    p, dx = req_params(16)
    srv = mfmhd.Server(p, 2.02 * request_charge(16, mfmhd.num_components(p)))
    srv.set_stage_kernel(mfmhd.STAGE_SUMMED)
    ids = [srv.submit(p, dx, 2, 0.5) for _ in range(2)]
    na, npd, _ = srv.step()
    assert (na, npd) == (2, 0)
    run_until_done(srv, lambda: ids)
    srv.close()

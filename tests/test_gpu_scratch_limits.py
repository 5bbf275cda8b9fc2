"""The face sums where their scratch finds no device memory: the call runs the
separate kernels, and the context does not ask for that memory again on every
call (it would free and allocate its scratch each time) until its stage kernel
is set again."""
import ctypes as C

import numpy as np
import pytest

import mfmhd
from helpers import GpuPatch, grid_shape, periodic_fill, smooth_state
from test_gpu_parity import periodic_params

pytestmark = pytest.mark.gpu

N, NF = (130, 130, 120), 3


def free_bytes():
    f, t = C.c_size_t(), C.c_size_t()
    assert mfmhd.load().hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


class Held:
    """Device memory taken so that about `leave` bytes stay free."""

    def __init__(self, leave):
        self.arrays = []
        size = 32 << 30
        while size >= 4 << 20:
            if free_bytes() - size < leave:
                size //= 2
                continue
            self.arrays.append(mfmhd.DeviceArray((size // 8,)))

    def free(self):
        for a in self.arrays:
            a.free()
        self.arrays = []


def scratch(nc, sums):
    """Scratch of an FP64 RK2 call on N: U*, W, faces of the box + 2, the sums
    when asked for, as the context allocates it (an eighth more); the tables
    come to under 8 MB."""
    a256 = lambda x: (x + 255) // 256 * 256
    cells = np.prod([n + 8 for n in N])
    b = 2 * a256(cells * nc * 8) + (a256(cells * (nc + 1) * 8) if sums else 0)
    for d in range(3):
        f = np.prod([N[e] + 4 + (e == d) for e in range(3)])
        b += a256(f * nc * 8) + a256(f * 8)
    return int(b) * 9 // 8


def test_refused_sums():
    p = periodic_params(nf=NF)
    nc = mfmhd.num_components(p)
    vhi = tuple(n - 1 for n in N)
    lo, hi, shape = grid_shape(nc, (0, 0, 0), vhi, 4)
    U = periodic_fill(smooth_state(p, shape, lo, seed=1), 4)
    box = mfmhd.Box.of((0, 0, 0), vhi)

    def step(ctx, g):
        ctx.set_timing(True)
        r = ctx.update_state(g.fab, box, 2e-3, 1.0 / 32)
        return ctx.timing(1, mfmhd.KT_FSUM_PLASMA)[1] > 0, r

    patches = [GpuPatch(U, lo) for _ in range(4)]
    want = {}
    for q, mode in enumerate((mfmhd.STAGE_AUTO, mfmhd.STAGE_SEPARATE)):  # all kernels have run
        ctx = mfmhd.Context(p)
        ctx.set_stage_kernel(mode)
        sums, want[mode] = step(ctx, patches[q])
        assert sums == (mode == mfmhd.STAGE_AUTO)
        ctx.close()
    first = patches[0].numpy()
    small, large = scratch(nc, False), scratch(nc, True)
    held = Held((small + large) // 2)
    try:
        assert small + (32 << 20) < free_bytes() < large
        for q, mode in ((2, mfmhd.STAGE_AUTO), (3, mfmhd.STAGE_SUMMED)):
            print("refused sums, mode", mode, flush=True)
            ctx = mfmhd.Context(p)
            ctx.set_stage_kernel(mode)
            sums, r = step(ctx, patches[q])
            assert not sums and r == want[mfmhd.STAGE_SEPARATE]
            assert np.array_equal(patches[q].numpy(), first)
            if mode == mfmhd.STAGE_AUTO:
                ctx.close()
    finally:
        held.free()
    # there is memory again: not asked for, until the stage kernel is set
    assert not step(ctx, patches[3])[0]
    ctx.set_stage_kernel(mfmhd.STAGE_AUTO)
    assert step(ctx, patches[3])[0]
    ctx.close()


def test_failed_host_call_keeps_no_memory():
    """U finds device memory, its scratch does not: the call's U is given back,
    and a smaller call fits."""
    p = periodic_params(nf=NF)
    nc = mfmhd.num_components(p)
    vhi = tuple(n - 1 for n in N)
    lo, hi, shape = grid_shape(nc, (0, 0, 0), vhi, 4)
    U = periodic_fill(smooth_state(p, shape, lo, seed=1), 4)
    slo, _, sshape = grid_shape(nc, (0, 0, 0), (19, 19, 19), 4)
    V = periodic_fill(smooth_state(p, sshape, slo, seed=2), 4)
    ctx = mfmhd.Context(p)
    ctx.update_state_host(V, slo, mfmhd.Box.of((0, 0, 0), (19, 19, 19)), 2e-3, 1.0 / 32)
    held = Held(U.nbytes + (512 << 20))
    try:
        before = free_bytes()
        assert U.nbytes + (64 << 20) < before < scratch(nc, False)
        with pytest.raises(mfmhd.MfmError):
            ctx.update_state_host(U, lo, mfmhd.Box.of((0, 0, 0), vhi), 2e-3, 1.0 / 32)
        assert free_bytes() > before - U.nbytes // 2
        ctx.update_state_host(V, slo, mfmhd.Box.of((0, 0, 0), (19, 19, 19)), 2e-3, 1.0 / 32)
    finally:
        held.free()
        ctx.close()

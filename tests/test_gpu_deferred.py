"""Particles that leave their segment's window since the sort: the passes that
complete them in the block against the chunk kernels on unsorted particles."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("state", [0, 1])
@pytest.mark.parametrize("shape", range(5))
@pytest.mark.parametrize("far", [0.02, 1.0])
@pytest.mark.parametrize("bz", [False, True])
def test_far_particles(gpu, state, shape, far, bz):
    """Two fused passes, a pass without a deposit: `far` of the particles move
    60 cells a pass.  Particles bit for bit (both kernels do the reference's
    arithmetic per particle from the same field); charge within 1e-12 (FP64
    sums) or a fixed-point quantum (2^-30 of a block's charge, FP32)."""
    pic = gpu
    L = pic._lib
    nx, ny, n = 128, 128, 30_011
    rng = np.random.default_rng(shape)
    p = np.asfortranarray(rng.uniform(0.0, 1.0, (5, n)))
    p[2:4] = rng.uniform(-1.0, 1.0, (2, n))
    p[2:4, : int(far * n)] = rng.choice([-60.0, 60.0], (2, int(far * n))) / nx / 0.01
    p[4] = 1.0 / n
    grids = [np.asfortranarray(rng.uniform(-1, 1, (nx, ny))) for _ in range(3)]
    out = []
    for lanes in (True, False):
        ctx = pic.api.Context(pic.TwoDGrid(1.0, nx, 1.0, ny))
        ctx.set_particles(p)
        ctx.set_state(state)
        for g, which in zip(grids, (L.PIC_GRID_EX, L.PIC_GRID_EY, L.PIC_GRID_BZ)):
            ctx.set_grid(which, g)
        if bz:
            ctx.set_bz(L.PIC_BZ_GRID)
        perm = np.arange(n, dtype=np.int32)
        if lanes:
            L.call("pic_sort_lanes", ctx.h, perm.ctypes.data)
        rho = np.zeros((nx, ny), order="F")
        rhos = []
        for mode in (0, 1, 1, 2):
            L.call("pic_step_pass", ctx.h, shape, mode, 0.01, rho.ctypes.data)
            rhos.append(rho.copy())
        q = np.empty_like(p)
        ctx.get_particles(q)
        back = np.empty_like(q)
        back[:, perm] = q
        slow = C.c_uint64()
        L.call("pic_slow_chunks", ctx.h, C.byref(slow))
        out.append((back, rhos[:3], slow.value))
        ctx.close()
    assert out[0][2] >= int(far * n)
    np.testing.assert_array_equal(out[0][0], out[1][0])
    for a, b in zip(out[0][1], out[1][1]):
        assert np.linalg.norm(a - b) <= (1e-12 if state == 0 else 1e-5) * np.linalg.norm(b)

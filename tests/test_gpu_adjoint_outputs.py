"""The adjoint's gradients in whichever output is asked for, and with sorts that
fall between, on and after checkpoints: any sort plan gives the same
gradients."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("state", [0, 1])
@pytest.mark.parametrize("kernel", [0, 1])
def test_outputs_and_sort_plans(gpu, state, kernel):
    """One output alone equals the same one of both; particles come back as
    they were; gradients of other sort plans agree to the rounding of their
    charge sums (1e-10 in FP64; FP32 steps and 2^-30 fixed-point charge over
    7 steps: 1e-3)."""
    pic = gpu
    L = pic._lib
    nx, ny, n, steps = 64, 32, 20_011, 7
    rng = np.random.default_rng(kernel)
    p = np.asfortranarray(rng.uniform(0.0, 1.0, (5, n)))
    p[0] *= 4 * np.pi
    p[1] *= 2 * np.pi
    p[2:4] = rng.standard_normal((2, n))
    p[4] = 8 * np.pi**2 / n
    ctx = pic.api.Context(pic.TwoDGrid(4 * np.pi, nx, 2 * np.pi, ny))
    ref = None
    for ckpt, every in ((7, 0), (3, 2), (2, 1), (1, 0)):
        ctx.set_particles(p)
        ctx.set_state(state)
        got = []
        for want in ((True, True), (True, False), (False, True)):
            out = [np.full((2, n), np.nan, order="F") if w else None for w in want]
            j = C.c_double()
            L.call("pic_adjoint", ctx.h, kernel, 0.05, steps, ckpt, every, C.byref(j),
                   *(o.ctypes.data if o is not None else None for o in out))
            got.append(out)
        tol = 1e-10 if state == 0 else 1e-3
        for a, b in ((got[0][0], got[1][0]), (got[0][1], got[2][1])):
            assert np.linalg.norm(a - b) <= tol * np.linalg.norm(a)
        if ref is None:
            ref = got[0]
        for a, b in zip(got[0], ref):
            assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b)
        q = ctx.get_particles(np.empty_like(p))
        assert np.abs(q - p).max() <= (0.0 if state == 0 else 2e-6)
    ctx.close()

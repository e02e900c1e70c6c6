"""Particles and grids between host and device: the weights' verdict wherever a
weight differs, transfers below and above the size of the kept staging buffer,
and grids of every layout on both sides of the pinned copy's size."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _context(pic, nx, ny):
    return pic.api.Context(pic.TwoDGrid(1.0, nx, 1.0, ny))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 4_097, 1_700_003])
def test_particles_come_back_and_weights_are_judged(gpu, n):
    """Bitwise round trips of one context, uniform and weighted in turn: the
    FP32 state is refused exactly when a weight differs from the first (also
    the last one, or a NaN)."""
    pic = gpu
    ctx = _context(pic, 16, 16)
    rng = np.random.default_rng(n)
    p = np.asfortranarray(rng.uniform(0.01, 0.99, (5, n)))
    for odd in (None, n - 1, None, n // 2, None):
        p[4] = 0.25
        differ = odd is not None and n > 1 and odd > 0
        if odd is not None:
            p[4, odd] = np.nan if odd == n // 2 else 0.5
            differ = differ or n == 1 and bool(np.isnan(p[4, 0]))
        ctx.set_particles(p)
        np.testing.assert_array_equal(ctx.get_particles(np.empty_like(p)), p)
        if differ:
            with pytest.raises(Exception):
                ctx.set_state(1)
        else:
            ctx.set_state(1)
    ctx.close()


@pytest.mark.parametrize("nx,ny", [(4, 4), (33, 20), (512, 256), (400, 350)])
def test_grids_of_every_layout(gpu, nx, ny):
    """Set and read back bitwise: packed, with a ghost line to skip, strided;
    read packed and with the ghost line.  400 x 350 is past the pinned copy."""
    pic = gpu
    L = pic._lib
    ctx = _context(pic, nx, ny)
    rng = np.random.default_rng(nx)
    for which in (L.PIC_GRID_RHO, L.PIC_GRID_EX, L.PIC_GRID_EY, L.PIC_GRID_BZ, L.PIC_GRID_PHI):
        for layout in ("packed", "ghost", "strided"):
            g = rng.standard_normal((nx, ny))
            if layout == "packed":
                ctx.set_grid(which, np.asfortranarray(g))
            elif layout == "ghost":
                a = np.full((nx + 1, ny + 1), np.nan, order="F")
                a[:nx, :ny] = g
                ctx.set_grid(which, a)
            else:
                a = np.full((2, nx, ny), np.nan, order="F")
                a[0] = g
                ctx.set_grid(which, a, stride=2)
            np.testing.assert_array_equal(ctx.get_grid(which), g)
            full = ctx.get_grid(which, ghost=True)
            np.testing.assert_array_equal(full[:nx, :ny], g)
            np.testing.assert_array_equal(full[nx], full[0])
            np.testing.assert_array_equal(full[:, ny], full[:, 0])
    ctx.close()


@pytest.mark.parametrize("nx,ny", [(32, 16), (512, 512)])
@pytest.mark.parametrize("order", ["xy", "yx"])
def test_fields_set_reach_the_fp32_pass(gpu, nx, ny, order):
    """A kick after ex, ey and bz were set (either first) in FP32 agrees with
    the FP64 pass.  Bound: offsets, fields and weights rounded to FP32, a cubic
    of at most 16 weights: under 64 roundings of 6e-8 of the kick (at most 4)."""
    pic = gpu
    L = pic._lib
    rng = np.random.default_rng(nx)
    n = 5_000
    p = np.asfortranarray(rng.uniform(0.01, 0.99, (5, n)))
    p[2:4] *= 1e-3
    p[4] = 1.0 / n
    grids = {w: np.asfortranarray(rng.uniform(-1, 1, (nx, ny)))
             for w in (L.PIC_GRID_EX, L.PIC_GRID_EY, L.PIC_GRID_BZ)}
    seq = [L.PIC_GRID_EX, L.PIC_GRID_EY, L.PIC_GRID_BZ]
    if order == "yx":
        seq.reverse()
    v = []
    for state in (0, 1):
        ctx = _context(pic, nx, ny)
        ctx.set_particles(p)
        ctx.set_state(state)
        for w in seq:
            ctx.set_grid(w, grids[w])
        ctx.set_bz(L.PIC_BZ_GRID)
        L.call("pic_step_pass", ctx.h, 0, 2, 1e-3, None)
        v.append(ctx.get_particles(np.empty_like(p))[2:4])
        ctx.close()
    assert np.abs(v[0] - p[2:4]).max() > 1e-4
    assert np.abs(v[0] - v[1]).max() <= 64 * 2.0**-24 * 4e-3


def _hip():
    """The HIP runtime the library has loaded."""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64.so" in line)
    return C.CDLL(path)


@pytest.mark.parametrize("weighted", [False, True])
def test_device_particles_are_read_on_return(gpu, weighted):
    """pic_set_particles_device has read the caller's array when it returns,
    with one weight and with several: overwritten at once on another stream,
    the particles are still the ones given."""
    pic = gpu
    n = 4_000_000
    rng = np.random.default_rng(1)
    p = np.asfortranarray(rng.uniform(0.05, 0.95, (5, n)))
    if not weighted:
        p[4] = 0.25
    ctx = _context(pic, 16, 16)
    hip = _hip()
    d, s = C.c_void_p(), C.c_void_p()
    assert hip.hipMalloc(C.byref(d), C.c_size_t(p.nbytes)) == 0
    assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0  # non-blocking
    assert hip.hipMemcpy(d, C.c_void_p(p.ctypes.data), C.c_size_t(p.nbytes), 1) == 0
    pic._lib.call("pic_set_particles_device", ctx.h, d, n)
    assert hip.hipMemsetAsync(d, 0, C.c_size_t(p.nbytes), s) == 0
    assert hip.hipStreamSynchronize(s) == 0
    got = ctx.get_particles(np.zeros((5, n), order="F"))
    assert hip.hipFree(d) == 0 and hip.hipStreamDestroy(s) == 0
    np.testing.assert_array_equal(got, p)
    ctx.close()


def test_kept_staging_is_at_most_64_mib(gpu):
    """60 MiB of particles go up through a staging buffer that the context
    keeps: it holds no more than 64 MiB beside their four arrays (multiples of
    the device's 2 MiB pages; a quarter more than the particles were 75)."""
    pic = gpu
    n = 60 * 2**20 // 40
    ctx = _context(pic, 16, 16)
    p = np.asfortranarray(np.random.default_rng(3).uniform(0.05, 0.95, (5, n)))
    p[4] = 0.25
    ctx.set_particles(p[:, :100])  # what a first transfer sets up
    hip = _hip()

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    before = free()
    ctx.set_particles(p)
    assert before - free() <= 4 * 8 * n + 68 * 2**20
    ctx.close()


@pytest.mark.parametrize("state", [0, 1])
def test_fields_of_a_new_context_are_zero(gpu, state):
    """A kick before any field was set or solved leaves the velocities alone, in
    both states, and phi reads as zero: whatever contexts before it left in the
    memory its grids lie in."""
    pic = gpu
    L = pic._lib
    nx = ny = 128
    mesh = pic.TwoDGrid(1.0, nx, 1.0, ny)
    p = np.asfortranarray(np.random.default_rng(9).uniform(0.1, 0.9, (5, 1_000)))
    p[:4] = p[:4].astype(np.float32)
    p[4] = 0.25
    for _ in range(4):
        ctx = _context(pic, nx, ny)
        for which in (L.PIC_GRID_RHO, L.PIC_GRID_EX, L.PIC_GRID_EY, L.PIC_GRID_BZ, L.PIC_GRID_PHI):
            ctx.set_grid(which, np.full((nx, ny), 1e3))
        ctx.close()
    sim = pic.Simulation(mesh, p, pic.M6(), state=state)
    np.testing.assert_array_equal(sim.grid(L.PIC_GRID_PHI), 0.0)
    sim.step_pass(2, 0.1)
    np.testing.assert_array_equal(sim.particles()[2:4], p[2:4])
    sim.close()

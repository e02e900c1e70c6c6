"""The window passes at the edges of their LDS windows, where a particle either
stays on the LDS path or is handed to the global-memory one: bit for bit
against the kernels that take particles in any order."""
import math

import numpy as np
import pytest

from conftest import random_particles

pytestmark = pytest.mark.gpu

SHAPES = ["CloudInCell", "M6", "NearestGridPoint", "TriangularShapeCloud", "M4"]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("nx,ny,n,bz", [(128, 128, 50_001, "none"), (256, 64, 30_003, "grid"),
                                        (512, 16, 9_999, "uniform"), (8, 8, 70, "none")])
def test_f32_pass_without_deposit_at_the_window_edge(gpu, shape, nx, ny, n, bz):
    """Kick and drift without a deposit (the loop's last pass) after the
    particles drifted up to ~40 cells since the sort, past the 32-cell margin
    of its window: every cell, offset and velocity equals that of the kernels
    that take any order, which gather from global memory."""
    pic = gpu
    L = pic._lib
    rng = np.random.default_rng(nx + n)
    mesh = pic.TwoDGrid(4 * math.pi, nx, 4 * math.pi, ny)
    p = random_particles(rng, n, mesh.dimx, mesh.dimy)
    grids = [rng.normal(size=(nx, ny)) for _ in range(3)]
    dt = 0.25
    # fastest particles: ~40 cells along x, and along y, in one step
    p[2] = rng.uniform(-1, 1, n) * 40 * mesh.dx / dt
    p[3] = rng.uniform(-1, 1, n) * 40 * mesh.dy / dt

    def context():
        c = pic.Context(mesh, capacity=n)
        for which, g in zip((L.PIC_GRID_EX, L.PIC_GRID_EY, L.PIC_GRID_BZ), grids):
            c.set_grid(which, g)
        c.set_bz({"none": L.PIC_BZ_NONE, "uniform": L.PIC_BZ_UNIFORM,
                  "grid": L.PIC_BZ_GRID}[bz], 0.7)
        return c

    k = getattr(pic, shape).code
    a = context()
    a.set_particles(p)
    a.set_state(L.PIC_STATE_F32)
    L.call("pic_sort_lanes", a.h, None)
    L.call("pic_step_pass", a.h, k, 1, dt, None)  # the slots stay, the particles drift
    b = context()
    b.set_state_f32(a.get_state_f32(), float(p[4, 0]))
    for c in (a, b):
        L.call("pic_step_pass", c.h, k, 2, dt, None)
    for u, v in zip(a.get_state_f32(), b.get_state_f32()):
        assert np.array_equal(u, v)
    a.close()
    b.close()

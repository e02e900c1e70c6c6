"""The MeshFields M6 charge (compute_rho_m6!, and the UA loop's) against 80-bit
sums at the offsets the reference forms."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIMX, DIMY = 4 * math.pi, 2 * math.pi


def _weights(t):
    s = 1 - t

    def p3(u):
        return ((((10 * u - 20) * u - 20) * u + 20) * u + 50) * u + 26

    def p4(u):
        return ((((-5 * u + 5) * u + 10) * u + 10) * u + 5) * u + 1

    return [w / 120 for w in (s ** 5, p4(s), p3(s), p3(t), p4(t), t ** 5)]


def _charge(x, w, mesh, x0, y0, compat):
    """(rho, raw density) of positions x (2, n) in 80 bits: cell and offset as
    the reference forms them, px = mod(x - x0, dimx) / dx, in FP64."""
    nx, ny = mesh.nx, mesh.ny
    px = np.mod(x[0] - x0, mesh.dimx) / mesh.dx
    py = np.mod(x[1] - y0, mesh.dimy) / mesh.dy
    i, j = px.astype(np.int64), py.astype(np.int64)
    wx = _weights((px - i).astype(np.longdouble))
    wy = _weights((py - j).astype(np.longdouble))
    acc = np.zeros((nx, ny), np.longdouble)

    def node(c, a, n):
        return (c + a - 2 - (1 if compat and a != 2 else 0)) % n

    for a in range(6):
        for b in range(6):
            np.add.at(acc, (node(i, a, nx), node(j, b, ny)), wx[a] * wy[b] * np.longdouble(w))
    raw = acc / (np.longdouble(mesh.dx) * np.longdouble(mesh.dy))
    return raw - acc.sum() / (np.longdouble(mesh.dimx) * np.longdouble(mesh.dimy)), raw


def _bound(n, mesh):
    """Of the error over the raw density's norm: all shares are positive, each
    within eight roundings (the weights' Horner steps and products, the density's
    division and shift), and their sums, of the 36 n / (nx ny) a node receives,
    within the square root of as many; u = 2^-53."""
    return (8 + math.sqrt(36 * n / (mesh.nx * mesh.ny))) * 2.0 ** -53


@pytest.mark.parametrize("nx,ny,n", [(128, 64, 20_000), (200, 144, 30_011)])  # one part, two
@pytest.mark.parametrize("xmin,ymin,compat", [(0.0, 0.0, True), (5.0, -9.0, False)])
def test_charge_keeps_the_offsets_last_bits(gpu, nx, ny, n, xmin, ymin, compat):
    """The offsets come from mod(x - x0, dimx) itself: taken again from the
    position put back into the domain, mod(..) + x0, they lose the bits of x0
    (x0 = xmax with compat), and the charge is 1e-14 off."""
    pic = gpu
    rng = np.random.default_rng(nx + n)
    mesh = pic.TwoDGrid(xmin, xmin + DIMX, nx, ymin, ymin + DIMY, ny)
    p = pic.Particles(n, DIMX * DIMY / n)
    p.x[0], p.x[1] = xmin + rng.uniform(0, DIMX, n), ymin + rng.uniform(0, DIMY, n)
    x0, y0 = (mesh.xmax, mesh.ymax) if compat else (xmin, ymin)
    want, raw = _charge(p.x, p.w, mesh, x0, y0, compat)
    moved = np.stack([np.mod(p.x[0] - x0, mesh.dimx) + x0, np.mod(p.x[1] - y0, mesh.dimy) + y0])
    f = pic.MeshFields2D(mesh)
    pic.compute_rho_m6_(f, p, compat=compat)
    assert np.array_equal(p.x, moved)
    err = np.linalg.norm((f.rho[:nx, :ny] - want).astype(np.float64))
    assert err <= _bound(n, mesh) * np.linalg.norm(raw.astype(np.float64))


def test_ua_charge_at_the_reconstructed_offsets(gpu):
    """update_particles_x! where every tau-sample of a particle is its position
    (and t = 0): the reconstruction is exact, sums of ntau equal values, and the
    offsets are those of mod(x - xmin, dimx)."""
    pic = gpu
    rng = np.random.default_rng(7)
    nx, ny, n, ntau, xmin, ymin = 128, 64, 20_000, 16, 5.0, -9.0
    mesh = pic.TwoDGrid(xmin, xmin + DIMX, nx, ymin, ymin + DIMY, ny)
    p = pic.Particles(n, DIMX * DIMY / n)
    p.x[0], p.x[1] = xmin + rng.uniform(0, DIMX, n), ymin + rng.uniform(0, DIMY, n)
    want, raw = _charge(p.x, p.w, mesh, xmin, ymin, False)
    moved = np.stack([np.mod(p.x[0] - xmin, mesh.dimx) + xmin,
                      np.mod(p.x[1] - ymin, mesh.dimy) + ymin])
    ua = pic.UA(ntau, 0.1, n)
    xt = np.asfortranarray(np.broadcast_to(p.x, (ntau, 2, n)).astype(np.complex128))
    f = pic.MeshFields2D(mesh)
    p.t[...] = 0.0
    pic.update_particles_x_(p, f, ua, xt)
    assert np.array_equal(p.x, moved)
    err = np.linalg.norm((f.rho[:nx, :ny] - want).astype(np.float64))
    assert err <= _bound(n, mesh) * np.linalg.norm(raw.astype(np.float64))


@pytest.mark.parametrize("nx,ny", [(32, 16), (400, 400), (512, 512)])  # one part, eight, past them
def test_one_weight_on_every_grid(gpu, nx, ny):
    """Particles.w is one number: on a context whose particles' weights differ,
    compute_rho_m6!(fields, particles) gives all of them the first one's, on
    grids of either deposit kernel alike: 1e-12 of the charge of particles of
    that weight, the bar of the FP64 charge sums in another order."""
    pic = gpu
    L = pic._lib
    rng = np.random.default_rng(nx)
    n = 3_001
    mesh = pic.TwoDGrid(0.0, DIMX, nx, 0.0, DIMY, ny)
    p = np.zeros((5, n), order="F")
    p[0], p[1] = rng.uniform(0, DIMX, n), rng.uniform(0, DIMY, n)
    p[4] = rng.uniform(0.5, 1.5, n)
    rho = []
    for w in (p[4], p[4, 0]):
        q = p.copy(order="F")
        q[4] = w
        sim = pic.Simulation(mesh, q, pic.M6())
        L.call("pic_compute_rho_m6_fields", sim.ctx.h, 0)
        rho.append(sim.grid(L.PIC_GRID_RHO))
        sim.close()
    assert np.linalg.norm(rho[0] - rho[1]) <= 1e-12 * np.linalg.norm(rho[1])

"""FP64 charge summed in 64-bit fixed point (the segment passes' blocks of 2,048
particles or more of one weight): against 80-bit sums at both sides of that
line, with everything in one cell, with weights of either sign and of any
exponent, and with what cannot be summed that way (weighted particles, offsets
that are no numbers)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LD = np.longdouble


def _ctx(pic, nx, ny):
    return pic.api.Context(pic.TwoDGrid(1.0, nx, 1.0, ny))


def _deposit(pic, ctx, kernel, p, nx, ny):
    L = pic._lib
    ctx.set_particles(p)
    L.call("pic_sort_lanes", ctx.h, None)
    out = np.zeros((nx, ny), order="F")
    L.call("pic_step_pass", ctx.h, kernel, 3, 0.0, out.ctypes.data)
    return out


def _weights(t, m6):
    if not m6:
        return [1 - t, t]
    def p3(t):
        return 26 + t * (50 + t * (20 + t * (-20 + t * (-20 + 10 * t))))
    def p4(t):
        return 1 + t * (5 + t * (10 + t * (10 + t * (5 - 5 * t))))
    u = 1 - t
    return [w / LD(120) for w in (u**5, p4(u), p3(u), p3(t), p4(t), t**5)]


def _reference(p, nx, ny, m6):
    """The sums in 80 bits of the shares at the FP64 cells and offsets."""
    cells, wts = [], []
    for x, n in ((p[0], nx), (p[1], ny)):
        xp = x / (1.0 / n)
        i = np.floor(xp)
        t = ((xp - (i + 1.0)) + 1.0).astype(LD)
        cells.append(i.astype(int))
        wts.append(_weights(t, m6))
    lo = 2 if m6 else 0
    rho = np.zeros(nx * ny, LD)
    for v, wv in enumerate(wts[1]):
        for u, wu in enumerate(wts[0]):
            k = (cells[0] - lo + u) % nx + nx * ((cells[1] - lo + v) % ny)
            order = np.argsort(k, kind="stable")
            ks = k[order]
            at = np.flatnonzero(np.r_[True, ks[1:] != ks[:-1]])
            rho[ks[at]] += np.add.reduceat((wu * wv * p[4])[order], at)
    return rho.reshape(nx, ny, order="F")


@pytest.mark.parametrize("m6", [False, True])
@pytest.mark.parametrize("n,clump,w", [
    (2_047, True, 1.0),          # FP64 sums: one block below the line
    (2_048, True, 1.0 / 3.0),    # the smallest fixed-point block
    (70_001, True, -0.7),        # one cell holds everything
    (600_011, False, 1.1e-150),
    (600_011, False, 3.3e150),
    (600_011, False, 1e-250)])   # FP64 sums: too near the type's limits
def test_fixed_point_charge_against_80_bit_sums(gpu, m6, n, clump, w):
    """1e-15 normwise.  A share is rounded by half a quantum at most, 2^-47 of
    the weight for the largest block here and independent of sign: over a
    cell's N >= 2,000 shares that is under 2^-47 / sqrt(N) = 2e-16 of the
    charge; the offsets' cubic and quintic weights add a few 2^-53."""
    # a block takes a segment of 64 cells whole on 128 x 128, a quarter on 64 x 64
    nx, ny = (128, 128) if clump else (64, 64)
    rng = np.random.default_rng(n)
    p = np.zeros((5, n), order="F")
    side = 1.0 if not clump else 1.0 / nx
    p[0] = rng.uniform(0.0, side, n)
    p[1] = rng.uniform(0.0, side if not clump else 1.0 / ny, n)
    p[4] = w
    ctx = _ctx(gpu, nx, ny)
    rho = _deposit(gpu, ctx, 1 if m6 else 0, p, nx, ny)
    ctx.close()
    ref = _reference(p, nx, ny, m6)
    err = np.sqrt((((rho - ref) / w) ** 2).sum()) / np.sqrt(((ref / w) ** 2).sum())
    assert err <= 1e-15
    assert abs(float(rho.sum() / (w * n)) - 1.0) <= 1e-14


@pytest.mark.parametrize("shape", range(5))
def test_weighted_and_uniform_particles_agree(gpu, shape):
    """The same weights with one particle's a rounding apart take the FP64
    sums; both sums are within 1e-13 of each other."""
    nx, ny, n = 40, 24, 800_003
    rng = np.random.default_rng(shape)
    p = np.asfortranarray(rng.uniform(0.0, 1.0, (5, n)))
    p[4] = 0.3
    q = p.copy(order="F")
    q[4, 5] = np.nextafter(0.3, 1.0)
    ctx = _ctx(gpu, nx, ny)
    a, b = (_deposit(gpu, ctx, shape, s, nx, ny) for s in (p, q))
    ctx.close()
    assert np.linalg.norm(a - b) <= 1e-13 * np.linalg.norm(b)


@pytest.mark.parametrize("m6", [False, True])
def test_a_lost_particle_still_shows(gpu, m6):
    """A velocity that is no number reaches the charge as one, as in FP64 sums,
    and the other nodes keep theirs."""
    L = gpu._lib
    nx, ny, n = 32, 32, 800_000
    rng = np.random.default_rng(3)
    p = np.asfortranarray(rng.uniform(0.0, 1.0, (5, n)))
    p[2:4] = 0.0
    p[4] = 1.0 / n
    p[2, 77] = np.nan
    ctx = _ctx(gpu, nx, ny)
    ctx.set_particles(p)
    L.call("pic_sort_lanes", ctx.h, None)
    out = np.zeros((nx, ny), order="F")
    L.call("pic_step_pass", ctx.h, 1 if m6 else 0, 0, 0.1, out.ctypes.data)
    ctx.close()
    assert np.isnan(out).any()
    keep = np.isfinite(out)
    assert keep.sum() >= nx * ny - 36

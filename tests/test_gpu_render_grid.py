"""Renderings whose cells follow the particles' reach: smoothing lengths below,
at and above the cutoff, lengths that reach nothing, images narrower than a
tile and particles given outside the periods, against a plain sum over every
particle."""
import numpy as np
import pytest

from pyticles_amd import _lib, interpolate

pytestmark = pytest.mark.gpu


def _plain(x, y, r, w, h, Lx, Ly, cutoff):
    # images as the device takes them: one shift where |d| > L / 2
    Z = np.zeros((x.size, y.size))
    mag = np.zeros_like(Z)
    for i in range(x.size):
        dx = r[:, 0] - x[i]
        dx = np.where(dx > Lx / 2, dx - Lx, dx)
        dx = np.where(dx < -Lx / 2, dx + Lx, dx)
        for j in range(y.size):
            dy = y[j] - r[:, 1]
            dy = np.where(dy > Ly / 2, dy - Ly, dy)
            dy = np.where(dy < -Ly / 2, dy + Ly, dy)
            s = np.sqrt(dx * dx + dy * dy)
            k = (s < cutoff) & (s < h)
            q = s[k] / h[k]
            t = w[k] * 5.0 / (np.pi * h[k] ** 2) * (1 + 3 * q) * (1 - q) ** 3
            Z[i, j] = t.sum()
            mag[i, j] = np.abs(t).sum()
    return Z, mag


@pytest.mark.parametrize("Lx,Ly,n,nx,ny,h,cutoff", [
    (40.0, 40.0, 1600, 33, 47, 2.0, 4.0),      # cells finer than the cutoff's
    (40.0, 23.0, 900, 16, 64, (0.5, 2.0), 3.0),  # mixed lengths
    (30.0, 30.0, 700, 17, 15, 3.0, 1.5),       # the cutoff is the reach
    (9.0, 50.0, 400, 1, 70, 2.0, 3.5),         # one pixel wide; two cells across
    (50.0, 9.0, 400, 70, 3, 2.0, 3.5),
    (64.0, 64.0, 37, 20, 20, 0.25, 6.0),       # few particles: the grid is coarsened
    (5.0, 5.0, 60, 9, 9, 2.0, 4.0),            # no stencil: every cell
])
def test_against_every_particle(Lx, Ly, n, nx, ny, h, cutoff):
    rng = np.random.Generator(np.random.PCG64(n))
    r = rng.uniform(0, 1, size=(n, 2)) * (Lx, Ly)
    h = np.full(n, h) if np.isscalar(h) else rng.uniform(*h, size=n)
    h[::17] = (0.0, -1.0, np.nan)[n % 3]
    x = (np.arange(nx) + 0.5) * (Lx / nx)
    y = (np.arange(ny) + 0.5) * (Ly / ny)
    a, m, rho = rng.normal(size=n), rng.uniform(0.8, 1.2, n), rng.uniform(0.9, 1.1, n)
    Z = interpolate.splash_map_2d(x, y, r, m, rho, a, h, (0, Lx, 0, Ly), cutoff)
    want, mag = _plain(x, y, r, a * m / rho, np.where(h > 0, h, 0.0), Lx, Ly, cutoff)
    # every term is a few roundings of FP64 from the plain one
    assert np.all(np.abs(Z - want) <= 64 * np.finfo(float).eps * np.maximum(mag, 1e-300) + 1e-15)

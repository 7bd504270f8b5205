"""Renderings of particles and pixels given outside the periods: a particle is
binned by its wrapped position while its record keeps the given one, whose
images are one shift away at most."""
import numpy as np
import pytest

from pyticles_amd import interpolate
from test_gpu_render_grid import _plain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Lx,Ly,n,nx,ny,h,cutoff", [
    (40.0, 40.0, 1600, 33, 47, 2.0, 4.0),   # cells finer than the cutoff's
    (30.0, 23.0, 700, 17, 15, 3.0, 1.5),    # the cutoff is the reach
    (9.0, 50.0, 400, 12, 70, 2.0, 3.5),     # four cells across
    (5.0, 50.0, 300, 9, 40, 2.0, 3.5),      # no stencil across
])
def test_outside_the_periods(Lx, Ly, n, nx, ny, h, cutoff):
    rng = np.random.Generator(np.random.PCG64(n + 1))
    L = np.array([Lx, Ly])
    r = rng.uniform(0, 1, size=(n, 2)) * L
    r += rng.integers(-1, 2, size=(n, 2)) * L            # a whole period off, on either side
    r[::5] += rng.uniform(-0.6, 0.6, size=(n, 2))[::5] * L  # and across a side by a part of one
    x = (np.arange(nx) + 0.5) * (Lx / nx)
    y = (np.arange(ny) + 0.5) * (Ly / ny)
    x[::4] -= Lx
    x[3::7] += Lx
    y[1::5] += 0.7 * Ly
    y[2] = -0.25 * Ly
    a, m, rho = rng.normal(size=n), rng.uniform(0.8, 1.2, n), rng.uniform(0.9, 1.1, n)
    hh = np.full(n, h)
    Z = interpolate.splash_map_2d(x, y, r, m, rho, a, hh, (0, Lx, 0, Ly), cutoff)
    want, mag = _plain(x, y, r, a * m / rho, hh, Lx, Ly, cutoff)
    assert np.count_nonzero(mag) > 0.3 * mag.size
    # every term is a few roundings of FP64 from the plain one, its separation
    # (of coordinates up to three periods) a few of theirs: |dW / dr| h <= 1.8 W(0)
    sep = 16 * np.finfo(float).eps * 3 * max(Lx, Ly) / h
    lip = (np.abs(a) * m / rho).max() * 5.0 / (np.pi * h * h) * 1.8 * sep * 64
    assert np.all(np.abs(Z - want) <= 64 * np.finfo(float).eps * mag + lip)

"""Renderings around the particle count up to which they skip the launch for the
largest smoothing length and take few cells: against a plain sum over every
particle, with one length far above the others."""
import numpy as np
import pytest

from pyticles_amd import interpolate
from test_gpu_render_grid import _plain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 65, 1023, 1024, 1025])
@pytest.mark.parametrize("big", [0, -1])  # place of the one large length: first and last looked at
def test_against_every_particle(n, big):
    L, cutoff = 40.0, 7.0
    rng = np.random.Generator(np.random.PCG64(n))
    r = rng.uniform(0, L, size=(n, 2))
    h = np.full(n, 1.5)
    h[big] = 6.0
    x, y = (np.arange(21) + 0.5) * (L / 21), (np.arange(19) + 0.5) * (L / 19)
    a, m, rho = rng.normal(size=n), rng.uniform(0.8, 1.2, n), rng.uniform(0.9, 1.1, n)
    Z = interpolate.splash_map_2d(x, y, r, m, rho, a, h, (0, L, 0, L), cutoff)
    want, mag = _plain(x, y, r, a * m / rho, h, L, L, cutoff)
    # every term is a few roundings of FP64 from the plain one
    assert np.all(np.abs(Z - want) <= 64 * np.finfo(float).eps * np.maximum(mag, 1e-300) + 1e-15)

"""Positions outside the box are refused wherever they stand in the array, with
the first one named, and a refused array changes nothing."""
import math

import numpy as np
import pytest

from pyticles_amd import _lib, configs
from pyticles_amd.arena import Arena
from pyticles_amd.device import DeviceBox

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 1000])
def test_first_position_outside(n):
    Lx, Ly = 40.0, 30.0
    rng = np.random.Generator(np.random.PCG64(n))
    r = rng.uniform(0, 1, size=(n, 2)) * (Lx, Ly)
    r[0] = 0.0  # the box holds its lower sides
    v, m = np.zeros((n, 2)), np.ones(n)
    prm = configs.params(Lx, Ly=Ly)
    with DeviceBox(n, prm) as b:
        b.upload(r=r, v=v, m=m, u=np.zeros(n))
        for i in sorted({0, n // 2, n - 1}):
            for c, L in ((0, Lx), (1, Ly)):
                for x in (L, np.nextafter(0.0, -1.0), math.nan, math.inf, -math.inf):
                    bad = r.copy()
                    bad[i, c] = x
                    if i + 1 < n:
                        bad[-1, c] = -1.0  # a later one is not the first
                    with pytest.raises(_lib.SphError, match="particle %d " % i) as e:
                        b.upload(r=bad)
                    assert e.value.code == _lib.SPH_ERR_ARG
                    with Arena(n + 64, precision=_lib.FP64) as ar:
                        with pytest.raises(_lib.SphError):
                            ar.add(configs.System(bad, v, m, 0.9, prm, 1, 0))
        assert np.array_equal(b.download("r"), r)
        r[:, 0] = np.nextafter(Lx, 0.0)
        b.upload(r=r)


@pytest.mark.parametrize("n", [3, 4, 255, 256, 259, 1000])
def test_one_different_mass(n):
    # equal masses drop out of the walks; one other mass anywhere must not:
    # the density of its neighbours grows by (m - 1) W_ij
    L, h = math.sqrt(n) + 8.0, 2.0
    rng = np.random.Generator(np.random.PCG64(n))
    r = configs.lattice(n, L, rng, jitter=0.2)
    prm = configs.params(L, h=h)

    def rho(m):
        with DeviceBox(n, prm) as b:
            b.upload(r=r, v=np.zeros((n, 2)), m=m, u=np.zeros(n))
            b.density()
            return b.download("rho")

    base = rho(np.ones(n))
    for i in sorted({0, 1, n // 2, n - 2, n - 1}):
        m = np.ones(n)
        m[i] = 3.0
        d = r - r[i]
        d -= L * np.rint(d / L)
        q = np.minimum(np.sqrt((d * d).sum(axis=1)) / h, 1.0)
        w = 5.0 / (math.pi * h * h) * (1 + 3 * q) * (1 - q) ** 3
        w[i] = 0.0
        assert np.max(np.abs(rho(m) - base - 2.0 * w)) <= 1e-13 * np.max(base)

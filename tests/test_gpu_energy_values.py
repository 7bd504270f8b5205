"""Energy totals over blocks whose last is part empty: an infinite energy in
the box gives an infinite total, not a NaN, and the slots past the box add
nothing."""
import math

import numpy as np
import pytest

from pyticles_amd import configs
from pyticles_amd.device import DeviceBox

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 1023, 1024, 1025, 1100, 4096, 4097])
@pytest.mark.parametrize("big", [math.inf, -math.inf])
def test_infinite_energy(n, big):
    L = max(8.0, math.sqrt(n))
    rng = np.random.Generator(np.random.PCG64(n))
    v = rng.normal(size=(n, 2))
    with DeviceBox(n, configs.params(L)) as b:
        b.upload(r=configs.lattice(n, L, rng), v=v, m=np.ones(n))
        for i in {0, n // 2, n - 1}:
            u = np.ones(n)
            u[i] = big
            b.upload(u=u)
            ke, ue, tot = b.energy()
            # n terms, any order: each addition rounds by at most eps / 2
            assert abs(ke - 0.5 * (v * v).sum()) <= n * np.finfo(float).eps * ke
            assert ue == big and tot == big

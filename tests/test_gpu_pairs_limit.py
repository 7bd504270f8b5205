"""A pair list past 32-bit counts is refused, and the box works on."""
import math

import numpy as np
import pytest

from pyticles_amd import _lib, configs
from pyticles_amd.device import DeviceBox

pytestmark = pytest.mark.gpu


def test_more_pairs_than_32_bits_count():
    n = 92800
    assert n * (n - 1) // 2 >= 2 ** 32
    L = math.sqrt(n)
    r = configs.lattice(n, L, np.random.Generator(np.random.PCG64(1)))
    with DeviceBox(n, configs.params(L, rc=2.0 * L)) as b:
        b.upload(r=r, v=np.zeros((n, 2)), m=np.ones(n), u=np.zeros(n))
        with pytest.raises(_lib.SphError) as e:
            b.pairs(cap=64)
        assert e.value.code == _lib.SPH_ERR_ARG
        b.set_params(rc=1.5, tol=0.0)
        k = b.pairs()
        d = r[k[:, 0]] - r[k[:, 1]]
        d -= L * np.rint(d / L)
        assert len(k) > 3 * n and np.all((d * d).sum(axis=1) < 2.25 + 1e-9)

"""Pair export around the edges of its rows (56 partners), blocks and waves:
bit-exact against the oracle, in order, with and without room for all."""
import math

import numpy as np
import pytest

from oracle import oracle as O
from pyticles_amd import configs
from pyticles_amd.device import DeviceBox

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,L,rc", [
    (2, 20.0, 4.0), (63, 8.0, 4.0), (65, 9.0, 4.0), (257, 16.0, 4.0), (1023, 33.0, 4.0),
    (57, 30.0, 60.0),    # every pair: particle 0 has 56 partners
    (58, 30.0, 60.0),    # and 57: one past a row
    (900, 30.0, 6.5),    # about 66 partners: the long search
])
def test_against_oracle(n, L, rc):
    rng = np.random.Generator(np.random.PCG64(n))
    r = rng.uniform(0, L, size=(n, 2))
    prm = configs.params(L, rc=rc, tol=1.0)
    want = O.pairs(r, L, L, rc * rc + 1.0)
    with DeviceBox(n, prm) as b:
        b.upload(r=r, v=np.zeros((n, 2)), m=np.ones(n), u=np.zeros(n))
        if len(want):
            b.separations(want[:1])  # before the first export
        assert np.array_equal(b.pairs(), want)
        assert np.array_equal(b.pairs(cap=max(1, len(want) // 3)), want)  # asked again with room for all
        assert math.isfinite(b.separations(want)[2].sum()) if len(want) else True

"""Energy totals at sizes around the block and wave edges of the reduction."""
import math

import numpy as np
import pytest

from pyticles_amd import configs
from pyticles_amd.device import DeviceBox

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 65, 256, 1023, 1024, 1025, 2049, 70001])
def test_totals_at_a_given_state(n):
    rng = np.random.Generator(np.random.PCG64(n))
    L = max(10.0, math.sqrt(n))
    with DeviceBox(n, configs.params(L)) as b:
        r = configs.lattice(n, L, rng)
        v, m, u = rng.normal(size=(n, 2)), rng.uniform(0.5, 2.0, n), rng.normal(size=n)
        b.upload(r=r, v=v, m=m, u=u)
        ke, ue, et = b.energy()
    k = [0.5 * mi * (vx * vx + vy * vy) for mi, (vx, vy) in zip(m, v)]
    e = [mi * ui for mi, ui in zip(m, u)]
    # a sum of n rounded terms in trees of depth <= 4 + 6 + 2 + 8 + 8
    tol = 32 * np.finfo(float).eps
    assert abs(ke - math.fsum(k)) <= tol * math.fsum(k)
    assert abs(ue - math.fsum(e)) <= tol * math.fsum(map(abs, e))
    assert et == ke + ue

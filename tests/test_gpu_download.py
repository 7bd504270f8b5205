"""Many fields downloaded together against each field downloaded alone, at
sizes around the two 65,536-double halves that they travel through, and past 16 MB together."""
import numpy as np
import pytest

from pyticles_amd import configs
from pyticles_amd.device import DeviceBox

pytestmark = pytest.mark.gpu

COLUMNS = 23  # doubles a particle in all thirteen fields
HALF = 65536


@pytest.mark.parametrize("n", [1, HALF // COLUMNS, HALF // COLUMNS + 1, 2 * HALF // COLUMNS,
                               2 * HALF // COLUMNS + 1, 20011, HALF // 4, 100003])
def test_fields_together_and_alone(n):
    rng = np.random.Generator(np.random.PCG64(n))
    L = max(10.0, n ** 0.5)
    with DeviceBox(n, configs.params(L)) as b:
        r, v = configs.lattice(n, L, rng), rng.normal(size=(n, 2))
        b.upload(r=r, v=v, m=np.ones(n), u=rng.normal(size=n))
        b.rates()
        got = b.download(*b.FIELDS)
        assert np.array_equal(got["r"], r) and np.array_equal(got["v"], v)
        for f in b.FIELDS:
            alone = b.download(f)
            assert got[f].shape == alone.shape and np.array_equal(got[f], alone, equal_nan=True), f


def test_pairs_and_separations_past_the_halves():
    n, rng = 20011, np.random.Generator(np.random.PCG64(7))
    L = n ** 0.5
    with DeviceBox(n, configs.params(L)) as b:
        b.upload(r=configs.lattice(n, L, rng), v=rng.normal(size=(n, 2)), m=np.ones(n))
        iap = b.pairs()
        assert 2 * len(iap) > 3 * HALF
        assert np.all(np.diff(iap[:, 0] * n + iap[:, 1]) > 0)
        whole = b.separations(iap)
        step = 10007  # a slice's largest array stays within one half
        for k in range(0, len(iap), step):
            for w, part in zip(whole, b.separations(iap[k:k + step])):
                assert np.array_equal(w[k:k + step], part)

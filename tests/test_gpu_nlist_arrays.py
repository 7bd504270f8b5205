"""A Verlet list's build and separations fill the list's own arrays: with room,
without (the arrays grow), and where a program has put arrays of another kind in
their place."""
import math

import numpy as np
import pytest

from pyticles_amd import _lib, configs, neighbour_list, particles
from pyticles_amd.device import DeviceBox

pytestmark = pytest.mark.gpu

N = 257
L = math.sqrt(N)


def _list():
    rng = np.random.Generator(np.random.PCG64(N))
    p = particles.SmoothParticleSystem(N, d=2, maxn=N, xmax=L, ymax=L, hshort=2.0, hlong=4.0, temperature=0.9)
    p.r[:N], p.v[:N], p.m[:N] = configs.lattice(N, L, rng), rng.normal(size=(N, 2)), 1.0
    return neighbour_list.VerletList(p, cutoff=4.0, tolerance=1.0), p


def _want(p):
    with DeviceBox(N, configs.params(L)) as b:
        b.upload(r=p.r[:N], v=p.v[:N], m=np.ones(N), u=np.zeros(N))
        iap = b.pairs()
        return (iap,) + b.separations(iap)


def _room(nl, cap):
    nl.iap = np.full((cap, 2), -7, dtype=np.int64)
    for name, cols in (("rij", ()), ("rsq", ()), ("wij", ()), ("wij_lr", ()), ("drij", (2,)), ("dv", (2,)),
                       ("dwij", (2,)), ("dwij_lr", (2,))):
        setattr(nl, name, np.full((cap,) + cols, -7.0))


@pytest.mark.parametrize("room", [-1, 0, 1, 500, "few"])
def test_build_fills_or_grows_the_arrays(room):
    nl, p = _list()
    iap, drij, rij, rsq, dv = _want(p)
    k = len(iap)
    cap = 16 if room == "few" else k + room
    _room(nl, cap)
    own = nl.iap
    nl.build()
    assert nl.nip == k and nl.iap.shape[0] >= k
    assert (nl.iap is own) == (cap >= k)
    for got, want in ((nl.iap, iap), (nl.drij, drij), (nl.dv, dv), (nl.rsq, rsq)):
        assert np.array_equal(got[:k], want)
        if cap >= k:
            assert np.all(got[k:] == -7)  # rows past the pairs stay as they were
    assert not np.array_equal(nl.rij[:k], rij)  # build leaves rij to separations
    nl.separations()
    assert np.array_equal(nl.rij[:k], rij) and np.array_equal(nl.drij[:k], drij)


@pytest.mark.parametrize("name,array", [
    ("iap", lambda c: np.zeros((c, 2), dtype=np.int32)),
    ("drij", lambda c: np.zeros((c, 3))),
    ("dv", lambda c: np.zeros((2, c)).T),
    ("rsq", lambda c: np.zeros(c, dtype=np.float32)),
    ("rij", lambda c: np.zeros(2 * c)[::2]),
])
def test_other_arrays_are_copied_to(name, array):
    nl, p = _list()
    iap, drij, rij, rsq, dv = _want(p)
    setattr(nl, name, array(nl.iap.shape[0]))
    nl.build()
    nl.separations()
    k = nl.nip
    assert k == len(iap)
    for got, want in ((nl.iap, iap), (nl.drij[:, :2], drij), (nl.dv, dv), (nl.rsq, rsq), (nl.rij, rij)):
        assert np.array_equal(got[:k], want.astype(got.dtype))


def test_indices_outside_are_refused():
    nl, p = _list()
    with DeviceBox(N, configs.params(L)) as b:
        b.upload(r=p.r[:N], v=p.v[:N], m=np.ones(N), u=np.zeros(N))
        for bad in (-1, N, 2 ** 40, -2 ** 63, 2 ** 63 - 1):
            iap = np.zeros((10, 2), dtype=np.int64)
            iap[7, 1] = bad
            with pytest.raises(_lib.SphError) as e:
                b.separations(iap)
            assert e.value.code == _lib.SPH_ERR_ARG
        assert b.separations(np.array([[0, N - 1]]))[1].shape == (1,)

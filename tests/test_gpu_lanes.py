"""Pair passes that share a particle's list among 1, 2 or 4 lanes give the same
bits: the lane count follows the slots in use (4 up to 32,768, 2 up to 98,304,
then 1), so a box alone and the same box beside fillers that bring the slots
past each line take different walks."""
import numpy as np
import pytest

from pyticles_amd import _lib, configs
from pyticles_amd.arena import Arena

pytestmark = pytest.mark.gpu


def _system(n, seed, precision, masses, terms):
    rng = np.random.Generator(np.random.PCG64(seed))
    L = float(np.sqrt(n))
    prm = configs.params(L, precision=precision, terms=terms)
    m = np.ones(n) if masses == "equal" else rng.uniform(0.8, 1.2, n)
    return configs.System(configs.lattice(n, L, rng, jitter=0.3), configs.velocities(n, 0.8, rng), m, 0.8, prm, 12, seed)


def _result(s, fill, precision):
    """The box's result with filler boxes up to `fill` slots in the arena."""
    filler = [_system(fill - s.n, 7, precision, "equal", _lib.ALL_TERMS)] if fill > s.n else []
    with Arena(s.n + sum(f.n for f in filler), precision=precision) as ar:
        b = ar.add(s)
        for f in filler:
            ar.add(f, nsteps=13)
        for _ in range(60):
            ar.step(1)
            st, _, hl = ar.poll_all()
            assert hl[b] == 0
            if st[b] == _lib.BOX_DONE:
                return ar.result(b)
    raise AssertionError("the box did not finish")


@pytest.mark.parametrize("precision", [_lib.FP64, _lib.FP32C])
@pytest.mark.parametrize("n,masses,terms", [
    (257, "equal", _lib.ALL_TERMS),       # three cells a side; a wave and a lane of the next
    (1031, "equal", _lib.ALL_TERMS),
    (4099, "unequal", _lib.ALL_TERMS),
    (2048, "unequal", _lib.PRESSURE | _lib.COHESION),
    (1500, "equal", _lib.PRESSURE | _lib.CONDUCTION),
])
def test_shared_lists_give_the_same_bits(precision, n, masses, terms):
    s = _system(n, 3 + n, precision, masses, terms)
    ref = _result(s, 0, precision)                   # 4 lanes
    for fill in (32768, 32769, 98304, 98305):        # 4, 2, 2, 1 lanes
        got = _result(s, fill, precision)
        for k in ("r", "v", "u", "rho"):
            assert np.array_equal(got[k], ref[k]), (fill, k)
        assert (got["E0"], got["E1"]) == (ref["E0"], ref["E1"])

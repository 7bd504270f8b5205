"""Rates asked for in the middle of an open run: the run closes with the box's
own terms first, so its velocities, energies and the rates themselves are those
of a run closed before the call, whatever terms the call asks for."""
import numpy as np
import pytest

from pyticles_amd import _lib, configs
from pyticles_amd.device import from_system

pytestmark = pytest.mark.gpu

INVISCID = _lib.PRESSURE | _lib.COHESION
FIELDS = ("r", "v", "u", "rho", "acc", "udot")


@pytest.mark.parametrize("precision", [_lib.FP64, _lib.FP32C])
@pytest.mark.parametrize("own,asked", [(INVISCID, _lib.ALL_TERMS), (_lib.ALL_TERMS, _lib.PRESSURE),
                                       (INVISCID, INVISCID)])
@pytest.mark.parametrize("steps", [0, 1, 4, 9])  # 0: up to a step before a build, which the closing step makes
def test_rates_close_the_run_first(precision, own, asked, steps):
    visc = dict(eta=1.0, kcond=5.0) if own == _lib.ALL_TERMS else dict(eta=0.0, kcond=0.0)
    s = configs.square_system(20, 0.9, 11, 1, terms=own, precision=precision, **visc)

    def run(close):
        with from_system(s) as b:
            if steps:
                b.advance(steps)
            else:
                # the build counter shows where a step built; stop right before the third build
                k, builds = 0, []
                with from_system(s) as probe:
                    while len(builds) < 4:
                        probe.advance(1)
                        k += 1
                        builds += [k] * (probe.run_stats()["builds"] - len(builds))
                b.advance(builds[2] - 1)
            if close:
                b.sync()
            b.rates(asked)
            return b.download(*FIELDS)

    got, want = run(False), run(True)
    for k in FIELDS:
        assert np.array_equal(got[k], want[k]), k

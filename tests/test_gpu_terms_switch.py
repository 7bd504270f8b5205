"""Switching a box's terms over the line between steps with and without a
gradient pass: the step graphs of both kinds are kept, so a switch costs what
any parameter change costs, and the steps after it are those of a box that had
these terms all along."""
import time

import numpy as np
import pytest

from pyticles_amd import _lib, configs
from pyticles_amd.device import from_system

pytestmark = pytest.mark.gpu

INVISCID = dict(terms=_lib.PRESSURE | _lib.COHESION)
FULL = dict(terms=_lib.ALL_TERMS)
FIELDS = ("r", "v", "u", "rho", "acc", "udot")


def _least(f, reps=20):
    best = float("inf")
    for _ in range(reps):
        t = time.perf_counter()
        f()
        best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.parametrize("first", [FULL, INVISCID])
def test_switch_costs_a_parameter_change(first):
    other = INVISCID if first is FULL else FULL
    s = configs.square_system(32, 0.9, 12, 1, **first)
    with from_system(s) as b:
        b.step(20)
        same = _least(lambda: b.set_params(**first))

        def there_and_back():
            b.set_params(**other)
            b.set_params(**first)
        # capturing ten graphs again is hundreds of times a parameter change
        assert _least(there_and_back) < 20 * same + 200e-6


@pytest.mark.parametrize("precision", [_lib.FP64, _lib.FP32C])
@pytest.mark.parametrize("first", [FULL, INVISCID])
def test_steps_after_a_switch(precision, first):
    other = INVISCID if first is FULL else FULL
    with from_system(configs.square_system(24, 0.9, 13, 1, precision=precision, **first)) as b:
        for terms in (other, first, other):
            for nsteps in (9, 24):  # odd and even: graphs of both parities, and chunks
                state = b.download("r", "v", "u")
                b.set_params(**terms)
                b.upload(**state)
                b.step(nsteps)
                got = b.download(*FIELDS)
                with from_system(configs.square_system(24, 0.9, 13, 1, precision=precision, **terms)) as c:
                    c.upload(**state)
                    c.step(nsteps)
                    want = c.download(*FIELDS)
                # the lists hold the same pairs in another order (slots were
                # sorted from another order): rounding of the sums, grown by
                # the few steps
                tol = 1e-11 if precision == _lib.FP64 else 1e-5
                for k in FIELDS:
                    assert np.max(np.abs(got[k] - want[k])) <= tol * np.max(np.abs(want[k])), (terms, nsteps, k)

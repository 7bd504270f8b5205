"""Boxes and arenas of one context driven by several threads at once: they share
its stream, its pinned memory and its graph captures (terms that switch make a
box capture while others launch), and each gets what it gets alone."""
import threading

import numpy as np
import pytest

from pyticles_amd import _lib, configs
from pyticles_amd.arena import Arena
from pyticles_amd.device import from_system

pytestmark = pytest.mark.gpu

INVISCID = _lib.PRESSURE | _lib.COHESION
FIELDS = ("r", "v", "u", "rho", "acc", "udot")


def _box(k):
    s = configs.square_system(20 + 3 * k, 0.9, 30 + k, 1)
    return from_system(s), s


def _drive_box(b, s):
    out = []
    for terms in (_lib.ALL_TERMS, INVISCID, _lib.ALL_TERMS, INVISCID):
        b.set_params(terms=terms)
        b.step(11)
        for _ in range(4):
            b.advance(3)
            out.append(b.download(*FIELDS))
        out.append(dict(e=np.array(b.energy())))
        p = b.pairs()
        out.append(dict(zip(("drij", "rij", "rsq", "dv"), b.separations(p)), p=p))
        b.upload(r=s.r, v=s.v)
    return out


def _drive_arena(ar, systems):
    out = []
    for _ in range(3):
        ids = [ar.add(s, nsteps=9) for s in systems]
        ar.step(11)
        for i in ids:
            assert ar.done(i)[0]
            out.append(ar.result(i))
            ar.remove(i)
    return out


def test_threads_get_what_they_get_alone():
    systems = [configs.square_system(12 + k, 0.7, 60 + k, 1) for k in range(6)]
    want = []
    for k in range(3):
        b, s = _box(k)
        want.append(_drive_box(b, s))
        b.close()
    with Arena(4000, precision=_lib.FP64) as ar:
        want.append(_drive_arena(ar, systems))
    boxes = [_box(k) for k in range(3)]
    got = [None] * 4
    with Arena(4000, precision=_lib.FP64) as ar:
        work = [lambda k=k: _drive_box(*boxes[k]) for k in range(3)] + [lambda: _drive_arena(ar, systems)]

        def run(k):
            got[k] = work[k]()
        threads = [threading.Thread(target=run, args=(k,)) for k in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    for k in range(4):
        assert got[k] is not None and len(got[k]) == len(want[k])
        for g, w in zip(got[k], want[k]):
            for f in w:
                assert np.array_equal(g[f], w[f]), (k, f)
    for b, _ in boxes:
        b.close()

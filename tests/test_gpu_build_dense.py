"""Shared list builds of cells of more than 64 slots (single-cell boxes, wide
supports, clustered particles): the entries and order of the one-lane build,
the same verdict on lists that overflow, and no slower chain of candidates."""
import numpy as np
import pytest

from pyticles_amd import _lib, configs
from pyticles_amd.arena import Arena
from pyticles_amd.device import from_system

pytestmark = pytest.mark.gpu

FILL = 8 * 49152 + 8  # slots past which a box of this size takes one lane a slot
LISTCAP = 8


def _system(n, Lx, Ly, seed, precision, **kw):
    rng = np.random.Generator(np.random.PCG64(seed))
    cols = int(np.ceil(np.sqrt(n * Lx / Ly)))
    rows = -(-n // cols)
    k = np.arange(n)
    j = rng.uniform(0.4, 0.6, size=(n, 2))
    r = np.stack([(k % cols + j[:, 0]) * (Lx / cols), (k // cols + j[:, 1]) * (Ly / rows)], axis=1)
    prm = configs.params(Lx, Ly=Ly, precision=precision, **kw)
    return configs.System(np.ascontiguousarray(r), configs.velocities(n, 0.8, rng), np.ones(n), 0.8, prm, 8, seed)


def _run(systems, fill, precision, bits):
    n = sum(s.n for s in systems)
    filler = [_system(fill - n, 700.0, (fill - n) / 700.0, 5, precision)] if fill else []
    with Arena(n + sum(f.n for f in filler), precision=precision) as ar:
        ar.set_list_bits(bits)
        ids = [ar.add(s) for s in systems]
        for f in filler:
            ar.add(f, nsteps=1)
        health = np.zeros(len(ids), dtype=int)
        for _ in range(20):
            ar.step(1)
            st, _, hl = ar.poll_all()
            health |= hl[ids]
            if np.all(st[ids] == _lib.BOX_DONE):
                break
        return health, [ar.result(i) for i in ids]


@pytest.mark.parametrize("precision,bits", [(_lib.FP64, 32), (_lib.FP64, 16), (_lib.FP32C, 16)])
def test_same_lists_as_one_lane(precision, bits):
    systems = [
        _system(64, 8.0, 8.0, 1, precision),               # one cell, at the line
        _system(65, 8.0, 8.1, 2, precision),               # and past it
        _system(129, 11.4, 11.4, 3, precision),
        _system(169, 13.0, 13.0, 4, precision),
        _system(700, 13.0, 54.0, 6, precision),            # one cell across
        _system(640, 32.0, 20.0, 7, precision, rc=8.0, hl=5.0),
        _system(900, 36.0, 36.0, 8, precision, rc=9.5),    # cells of ~144 slots
    ]
    h0, ref = _run(systems, 0, precision, bits)
    h1, got = _run(systems, FILL, precision, bits)
    assert not h0.any() and not h1.any()
    for a, b in zip(ref, got):
        for k in ("r", "v", "u", "rho"):
            assert np.array_equal(a[k], b[k]), k


def test_overflowing_lists_are_flagged_alike():
    s = _system(400, 30.0, 30.0, 9, _lib.FP64)
    s.r = np.ascontiguousarray(15.0 + (s.r - 15.0) * 0.2)  # all in one cell's reach: lists of 399
    h0, _ = _run([s], 0, _lib.FP64, 16)
    h1, _ = _run([s], FILL, _lib.FP64, 16)
    assert h0[0] & LISTCAP and h1[0] & LISTCAP


def test_build_time_of_one_cell():
    def build_us(n, L):
        with from_system(_system(n, L, L, 10, _lib.FP64)) as b:
            b.step(2)
            return min(b.time_pass(b.BUILD, 40) for _ in range(5))
    # 169 slots are 11 rounds of 16 candidates a lane against 4 of 49's; a
    # slot's first lane alone, one candidate at a time, took 3.3 times as long
    assert build_us(169, 13.0) < 2.0 * build_us(49, 7.0)

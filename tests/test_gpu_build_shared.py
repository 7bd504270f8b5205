"""Lists built by four lanes of a slot (single boxes of up to 49,152 slots,
arenas of up to eight times as many) and by one lane hold the same entries in
the same order: a box alone and beside a filler that brings its arena past the
line gives the same bits, for boxes without a stencil along an axis, with
cells of more than 64 slots and with both entry widths."""
import numpy as np
import pytest

from pyticles_amd import _lib, configs
from pyticles_amd.arena import Arena

pytestmark = pytest.mark.gpu

FILL = 8 * 49152 + 8


def _system(n, Lx, Ly, seed, precision, **kw):
    rng = np.random.Generator(np.random.PCG64(seed))
    r = rng.uniform(0, 1, size=(n, 2)) * 0.2
    cols = int(np.ceil(np.sqrt(n * Lx / Ly)))
    rows = -(-n // cols)
    k = np.arange(n)
    r = np.stack([(k % cols + 0.4 + r[:, 0]) * (Lx / cols), (k // cols + 0.4 + r[:, 1]) * (Ly / rows)], axis=1)
    prm = configs.params(Lx, Ly=Ly, precision=precision, **kw)
    return configs.System(np.ascontiguousarray(r), configs.velocities(n, 0.8, rng), np.ones(n), 0.8, prm, 15, seed)


def _run(systems, fill, precision, bits):
    n = sum(s.n for s in systems)
    filler = [_system(fill - n, 700.0, (fill - n) / 700.0, 5, precision)] if fill else []
    with Arena(n + sum(f.n for f in filler), precision=precision) as ar:
        ar.set_list_bits(bits)
        ids = [ar.add(s) for s in systems]
        for f in filler:
            ar.add(f, nsteps=1)
        for _ in range(60):
            ar.step(1)
            st, _, hl = ar.poll_all()
            assert not hl[ids].any()
            if np.all(st[ids] == _lib.BOX_DONE):
                return [ar.result(i) for i in ids]
    raise AssertionError("the boxes did not finish")


@pytest.mark.parametrize("precision,bits", [(_lib.FP64, 16), (_lib.FP32C, 32)])
def test_same_lists_as_one_lane(precision, bits):
    systems = [
        _system(37, 6.0, 6.2, 1, precision),             # one cell
        _system(700, 9.0, 78.0, 2, precision),           # one cell across
        _system(700, 78.0, 9.0, 3, precision),
        _system(1500, 40.0, 40.0, 4, precision, rc=8.0),  # cells of ~94 slots
        _system(2900, 50.0, 58.0, 6, precision),
    ]
    ref = _run(systems, 0, precision, bits)
    got = _run(systems, FILL, precision, bits)
    for a, b in zip(ref, got):
        for k in ("r", "v", "u", "rho"):
            assert np.array_equal(a[k], b[k]), k

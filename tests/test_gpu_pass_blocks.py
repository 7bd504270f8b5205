"""The pair passes' block size where one lane walks a slot's list, which is
where it applies: depths that do not share lists, and boxes past the sharing
line.  It changes which work-items share a block, never a slot's walk."""
import numpy as np
import pytest

from pyticles_amd import _lib, configs
from pyticles_amd.device import from_system

pytestmark = pytest.mark.gpu


def _run(s, **schedule):
    with from_system(s) as b:
        b.set_schedule(**schedule)
        b.step(s.steps)
        return b.download("r", "v", "u", "rho", "acc", "udot")


@pytest.mark.parametrize("precision", [_lib.FP64, _lib.FP32C])
@pytest.mark.parametrize("nside,steps,unroll", [
    (24, 25, 1),   # no sharing at depth 1
    (314, 4, 0),   # 98,596 slots at the default depth
    (314, 4, 4),
    (24, 25, 0),   # shared lists: blocks of 256 whatever is asked
])
def test_block_sizes_agree(precision, nside, steps, unroll):
    s = configs.square_system(nside, 0.9, 7, steps, precision=precision)
    base = _run(s, unroll=unroll)
    for block in (128, 512):
        got = _run(s, unroll=unroll, block=block)
        for k in base:
            assert np.array_equal(got[k], base[k]), (block, k)

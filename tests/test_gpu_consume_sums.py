"""The CG run-ahead on grids whose passes form alpha and beta from the block
sums of the pass before them (up to 2048 blocks of 512 cells) and on the
first size past that, where a finisher forms them: bit for bit the iteration
without the run-ahead, every pass but the first taken over, at the edges of the
tree's groups of 512 blocks."""

import pytest

from tests.test_gpu_cg_hold_u import _check
from tests.test_gpu_run_ahead import H, _cg, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x,y", [(20, 12),       # one block
                                 (512, 512),     # 512 blocks, one group
                                 (514, 512),     # 514: a second group
                                 (1024, 1024),   # 2048: the last consuming grid
                                 (1026, 1024)])  # 2052: finishers
def test_consuming_passes_match_the_plain_iteration(x, y):
    assert x > 2 * H and y > 2 * H
    s0, f0, r0 = _cg(x, y, 11, False, 12)
    s1, f1, r1 = _cg(x, y, 11, True, 12)
    assert r0 == 0 and r1 >= 2 * 10
    assert _same(s0, s1)
    for n in f0:
        assert _same(f0[n], f1[n]), n
    _check(x, y, H, 12)

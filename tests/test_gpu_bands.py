"""The pair- and quad-per-thread passes' order of blocks (segments dealt to the
XCDs in bands, or launch order where rows are a multiple of eight blocks and up
to an eighth of a block long)
and their plain or streaming loads and stores: every solver's steps, scalars
and fields are bit for bit those of the one-cell kernels (TEA_HIP_PAIRS=0)."""

import pytest

from tests.test_gpu_odd_widths import _same, _steps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("x,y", [
    # rows of one block: the number of blocks is y; segments of 1024 blocks
    (512, 8), (512, 9), (512, 1023), (512, 1024), (512, 1025), (512, 1031), (512, 2049),
    (1500, 701),                              # rows of 2.93 blocks, two segments
    (4096, 130), (4144, 129), (4146, 129),
    (4160, 129), (4161, 129), (4162, 129),    # launch order up to 4096 + 64
    (1600, 2000), (1600, 2001),               # streaming from 3.2 M cells on (FP64 CG)
    (3100, 2000), (3101, 2000),               # and from 6.2 M (FP32)
])
def test_blocks_in_bands(x, y):
    s0, f0 = _steps(x, y, 2, False)
    s1, f1 = _steps(x, y, 2, True)
    assert _same(s0, s1)
    assert len(f0) == len(f1)
    for a, b in zip(f0, f1):
        assert _same(a, b)

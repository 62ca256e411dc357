"""The pair-per-lane kernels on odd row lengths, where every other row's pairs
are shifted by a cell, a pair may straddle two rows, and the last pair of an
odd number of cells has one cell: every solver's steps, scalars and fields bit
for bit against the one-cell kernels (TEA_HIP_PAIRS=0)."""

import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _chunk(x, y, h, pairs):
    from exploringsycl_amd.chunk import DeviceChunk
    old = os.environ.get("TEA_HIP_PAIRS")
    os.environ["TEA_HIP_PAIRS"] = "1" if pairs else "0"
    try:
        return DeviceChunk(x, y, h)
    finally:
        if old is None:
            del os.environ["TEA_HIP_PAIRS"]
        else:
            os.environ["TEA_HIP_PAIRS"] = old


def _steps(x, y, h, pairs):
    rng = np.random.default_rng(17)
    density, energy = rng.uniform(0.1, 100.0, x * y), rng.uniform(0.1, 25.0, x * y)
    out, scalars = [], []

    def read(c, *names):
        out.extend(c.read(n) for n in names)

    with _chunk(x, y, h, pairs) as c:
        c.write("density", density)
        c.write("energy", energy)
        # CG
        rro = c.cg_init(2, 0.8, 1.3)
        c.local_halos(1, ["u", "p"])
        c.copy_u()
        for _ in range(5):
            pw = c.cg_calc_w()
            rrn = c.cg_calc_ur(rro / pw)
            c.cg_calc_p(rrn / rro)
            c.local_halos(1, ["u", "p"])
            scalars += [pw, rrn]
            rro = rrn
        scalars.append(c.calculate_2norm("r"))
        read(c, "u", "p", "r", "w")
        # Chebyshev (an odd number of steps: pairs and a lone one), then PPCG
        c.cheby_init(3.0)
        c.local_halos(1, ["u"])
        for _ in range(3):
            c.cheby_iterate(0.3, 0.4)
            c.local_halos(1, ["u"])
        read(c, "u", "p", "r", "w")
        c.ppcg_init(3.0)
        for _ in range(3):
            c.local_halos(1, ["sd"])
            c.ppcg_inner_iteration(0.3, 0.4)
        read(c, "u", "r", "sd")
        # Jacobi
        c.jacobi_init(1, 0.8, 1.3)
        c.copy_u()
        c.local_halos(1, ["u"])
        for _ in range(3):
            scalars.append(c.jacobi_iterate())
            c.local_halos(1, ["u"])
        read(c, "u", "r")
        # Mixed precision and Jacobi-preconditioned flexible CG
        scalars += c.mpcg_init(2, 0.8, 1.3)
        alpha = beta = 0.0
        for it in range(4):
            pw, pr = c.mpcg_calc_w(alpha, it > 0, beta, it > 0)
            alpha = pr / pw
            rr, rw = c.mpcg_calc_r(alpha)
            beta = -rw / pw
            scalars += [pw, pr, rr, rw]
        scalars += c.mpcg_refresh(alpha, 1)
        out.extend(c.read_mp(n) for n in ("p", "r", "w"))
        read(c, "u")
        c.fcg_attach()
        scalars += c.fcg_init(2, 0.8, 1.3)
        scalars.append(c.fcg_precondition(0))
        scalars += c.fcg_calc_w(0.0, 0, 0.0)
        scalars += c.fcg_calc_r_precondition(0.05, 0)
        out.append(c.read_z())
    return np.array(scalars), out


def _same(a, b):
    """Bit for bit, any NaN equal to any other (with a halo of 1 the reference
    leaves the domain edge's face coefficients 0 / 0)."""
    nan = np.isnan(a) & np.isnan(b)
    return np.array_equal(np.where(nan, 0, a).view(np.uint8), np.where(nan, 0, b).view(np.uint8))


@pytest.mark.parametrize("x,y,h", [(9, 9, 1),      # 81 cells: an odd number
                                   (9, 9, 2), (13, 10, 2),  # rows shorter than a wave
                                   (1025, 33, 2),
                                   (127, 64, 2), (129, 31, 3),
                                   (515, 77, 2),   # rows longer than a block
                                   (1025, 33, 1)])
def test_odd_widths_match_the_one_cell_kernels(x, y, h):
    s0, f0 = _steps(x, y, h, False)
    s1, f1 = _steps(x, y, h, True)
    assert _same(s0, s1)
    if h > 1:
        assert np.isfinite(s0).all()
    for a, b in zip(f0, f1):
        assert _same(a, b)

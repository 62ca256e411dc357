"""The run-ahead of mixed-precision CG and FCG: calc_w queues the r-step (with
FCG also z = M(r)) and calc_r the next w-step, into spare buffers, with alpha
and beta formed on the device.  The drivers' call sequences with it and without
(TEA_HIP_RUN_AHEAD=0) give the same scalars and fields bit for bit, also when
the host strays from them."""

import os

import numpy as np
import pytest

from exploringsycl_amd import learned

pytestmark = pytest.mark.gpu
H = 2


def _chunk(x, y, ahead):
    from exploringsycl_amd.chunk import DeviceChunk
    old = os.environ.get("TEA_HIP_RUN_AHEAD")
    os.environ["TEA_HIP_RUN_AHEAD"] = "1" if ahead else "0"
    try:
        return DeviceChunk(x, y, H)
    finally:
        if old is None:
            del os.environ["TEA_HIP_RUN_AHEAD"]
        else:
            os.environ["TEA_HIP_RUN_AHEAD"] = old


def _attach(c, coarse):
    if coarse == "sweeps":
        from exploringsycl_amd.native import check
        check(c.lib.tea_hip_fcg_attach_sweeps(c.handle, 6, 8, 2), "attach")
    elif coarse == "net":
        params, norm, coarsen = learned.read_weights()
        c.fcg_attach(params, norm, coarsen=coarsen, levels=2)
    else:
        c.fcg_attach()


def _solve(cells, coarse, ahead, iters, refresh, stray=None):
    """coarse None: mixed-precision CG; else FCG with that preconditioner."""
    x, y = cells[0] + 2 * H, cells[1] + 2 * H
    rng = np.random.default_rng(x + y)
    scalars = []
    with _chunk(x, y, ahead) as c:
        c.write("density", rng.uniform(0.1, 100.0, x * y))
        c.write("energy", rng.uniform(0.1, 25.0, x * y))
        fcg = coarse is not None
        use = int(coarse in ("sweeps", "net"))
        if fcg:
            _attach(c, coarse)
            scalars += c.fcg_init(2, 0.8, 1.3)
            scalars.append(c.fcg_precondition(use))
        else:
            scalars += c.mpcg_init(2, 0.8, 1.3)
        alpha = beta = 0.0
        pu = pp = False
        for it in range(iters):
            if fcg:
                pw, pr = c.fcg_calc_w(alpha, pu, beta)
            else:
                pw, pr = c.mpcg_calc_w(alpha, pu, beta, pp)
            alpha = pr / pw
            if stray:
                stray.beta = beta
                alpha, use = stray(c, it, alpha, use)
            if fcg:
                rr, rx = c.fcg_calc_r_precondition(alpha, use)
            else:
                rr, rx = c.mpcg_calc_r(alpha)
            scalars += [pw, pr, rr, rx]
            pu = pp = True
            if (it + 1) % refresh == 0:
                scalars += c.mpcg_refresh(alpha, True)
                rx = scalars[-1]
                if fcg:
                    rx = c.fcg_precondition(use)
                    scalars.append(rx)
                pu = False
            beta = -rx / pw
        fields = [c.read_mp(n) for n in ("p", "r", "w")]
        if fcg:
            fields.append(c.read_z())
        fields.append(c.read("u"))
        taken = c.ahead_taken()[1]
    return np.array(scalars), fields, taken


def _same(a, b):
    return np.array_equal(np.asarray(a).view(np.uint8), np.asarray(b).view(np.uint8))


def _check(cells, coarse, least, **kw):
    """`least`: passes that the run-ahead has to have been taken over for."""
    s0, f0, n0 = _solve(cells, coarse, False, **kw)
    s1, f1, n1 = _solve(cells, coarse, True, **kw)
    assert n0 == 0 and n1 >= least, (n0, n1)
    assert np.isfinite(s0).all()
    assert _same(s0, s1)
    for a, b in zip(f0, f1):
        assert _same(a, b)


# Four cells per lane, two (x = 254; and odd), one coarse level and two; 2064
# blocks: a finisher in one block; 8640: a block per group.
@pytest.mark.parametrize("cells,coarse", [
    ((124, 60), None), ((250, 40), None), ((121, 50), None), ((1024, 1024), None),
    ((2100, 2100), None), ((124, 60), "jacobi"), ((121, 50), "jacobi"), ((72, 40), "sweeps"),
    ((128, 64), "sweeps"), ((1024, 1024), "sweeps"), ((256, 64), "net"), ((1024, 96), "net")])
def test_run_ahead_is_the_plain_iteration(cells, coarse):
    """22 iterations, a refresh after every 7: the second refresh falls where
    the first taught the library not to queue a w-step.  Every step but the
    first w-step and those after a refresh is taken over."""
    _check(cells, coarse, 2 * 22 - 4, iters=22, refresh=7)


@pytest.mark.parametrize("coarse", [None, "sweeps"])
def test_run_ahead_is_dropped_when_the_host_strays(coarse):
    """Another alpha than the device's (iteration 3), reads of u and r (5), a
    U halo update (7), a 2-norm (9), another preconditioner (11, FCG) and
    CG steps on the same chunk (13) between calc_w and calc_r."""
    def stray(c, it, alpha, use):
        if it == 3:
            alpha *= 1.0 + 2.0 ** -40
        if it == 5:
            c.read("u")
            c.read_mp("r")
        if it == 7:
            c.local_halos(1, ["u"])
        if it == 9:
            c.calculate_2norm("u")
        if it == 11 and coarse:
            use = 0
        if it == 13:
            c.cg_calc_w()
            c.cg_calc_ur(1e-3)
        return alpha, use

    _check((128, 64), coarse, 18, iters=18, refresh=50, stray=stray)


@pytest.mark.parametrize("cells,coarse", [((128, 64), None), ((121, 50), None),
                                          ((1100, 1000), None), ((128, 64), "sweeps")])
def test_a_pass_in_flight_is_taken_over_only_in_its_turn(cells, coarse):
    """The r-step (4) and the w-step (6) asked for twice in a row, with the
    scalars that the passes in flight behind them were made with."""
    def stray(c, it, alpha, use):
        if it == 4:
            (c.fcg_calc_r_precondition(alpha, use) if coarse else c.mpcg_calc_r(alpha))
        if it == 6:
            beta = stray.beta
            pw, pr = (c.fcg_calc_w(alpha, True, beta) if coarse
                      else c.mpcg_calc_w(alpha, True, beta, True))
            alpha = pr / pw
        return alpha, use

    _check(cells, coarse, 9, iters=9, refresh=50, stray=stray)


def test_init_of_a_second_solve_drops_a_pass_in_flight():
    """Two solves on one chunk; the first ends with passes queued."""
    for ahead in (False, True):
        with _chunk(132, 68, ahead) as c:
            rng = np.random.default_rng(4)
            c.write("density", rng.uniform(0.1, 100.0, 132 * 68))
            c.write("energy", rng.uniform(0.1, 25.0, 132 * 68))
            out = []
            for _ in range(2):
                out += c.mpcg_init(2, 0.8, 1.3)
                alpha = beta = 0.0
                for it in range(5):
                    pw, pr = c.mpcg_calc_w(alpha, it > 0, beta, it > 0)
                    alpha = pr / pw
                    rr, rw = c.mpcg_calc_r(alpha)
                    beta = -rw / pw
                    out += [pw, pr, rr, rw]
            half = len(out) // 2
            assert out[:half] == out[half:]
            if ahead:
                assert out == want
            want = out

"""FP64 CG with u's updates left to every third w-step (and the passes queued
two ahead) against each update made in its own w-step (TEA_HIP_HOLD_U=0,
TEA_HIP_RUN_AHEAD=0): the same scalars and fields bit for bit, also where other
calls come between the steps."""

import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FIELDS = ("u", "p", "r", "w", "sd", "u0", "energy")


def _chunk(x, y, h, on):
    from exploringsycl_amd.chunk import DeviceChunk
    names = ("TEA_HIP_HOLD_U", "TEA_HIP_RUN_AHEAD")
    old = {n: os.environ.get(n) for n in names}
    for n in names:
        os.environ[n] = "1" if on else "0"
    try:
        return DeviceChunk(x, y, h)
    finally:
        for n in names:
            if old[n] is None:
                del os.environ[n]
            else:
                os.environ[n] = old[n]


def _between(c, what, seen):
    """Calls that read or write u or p, or that other solvers make."""
    if what == "read":
        seen.append(c.read("u"))
    elif what == "norm":
        seen.append(np.array([c.calculate_2norm("u")]))
    elif what == "halos2":
        c.local_halos(2, ["u", "p"])
    elif what == "u_halo":
        c.local_halos(1, ["u"])
    elif what == "cheby":
        c.cheby_init(3.0)
        c.local_halos(1, ["u"])
        for _ in range(3):
            c.cheby_iterate(0.3, 0.4)
            c.local_halos(1, ["u"])
    elif what == "ppcg":
        c.ppcg_init(3.0)
        for _ in range(2):
            c.local_halos(1, ["sd"])
            c.ppcg_inner_iteration(0.3, 0.4)
    elif what == "residual":
        c.calculate_residual()
    elif what == "finalise":
        c.finalise()
        c.local_halos(1, ["energy1"])
    elif what == "summary":
        seen.append(np.array(c.field_summary()))
    elif what == "mixed":
        seen.append(np.array(c.mpcg_refresh(1e-3, 1)))
    elif what == "mixed_w":
        seen.append(np.array(c.mpcg_calc_w(1e-3, 1, 0.5, 1)))
    elif what == "fcg_w":
        seen.append(np.array(c.fcg_calc_w(1e-3, 1, 0.5)))


def _run(x, y, h, on, iters, between=(), where="end"):
    rng = np.random.default_rng(x * y)
    seen = []
    with _chunk(x, y, h, on) as c:
        c.set_chunk_data(0.0, 0.0, 0.1, 0.1)
        c.write("density", rng.uniform(0.1, 100.0, x * y))
        c.write("energy", rng.uniform(0.1, 25.0, x * y))
        if set(between) & {"mixed", "mixed_w", "fcg_w"}:
            c.fcg_attach()
            c.fcg_init(2, 0.8, 1.3)
            c.fcg_precondition(0)
        rro = c.cg_init(2, 0.8, 1.3)
        c.local_halos(1, ["u", "p"])
        c.copy_u()
        scalars = [rro]
        for it in range(iters):
            # One interruption after every fourth iteration: with 0, 1 and 2
            # updates held in turn.
            what = between[it // 4] if it % 4 == 3 and it // 4 < len(between) else None
            pw = c.cg_calc_w()
            if what and where == "after_w":
                _between(c, what, seen)
            rrn = c.cg_calc_ur(rro / pw)
            if what and where == "after_ur":
                _between(c, what, seen)
            c.cg_calc_p(rrn / rro)
            if what != "no_halo":
                c.local_halos(1, ["u", "p"])
            if what and where == "end":
                _between(c, what, seen)
            scalars += [pw, rrn]
            rro = rrn
        fields = [c.read(n) for n in FIELDS]
        taken = c.ahead_taken()[0]
    return np.array(scalars), seen + fields, taken


def _check(x, y, h, iters, **kw):
    s0, f0, n0 = _run(x, y, h, False, iters, **kw)
    s1, f1, n1 = _run(x, y, h, True, iters, **kw)
    # Every step but the first and, with three interruptions, those they drop;
    # none at odd x.
    assert n0 == 0
    assert n1 == 0 if x % 2 else n1 >= (2 * iters - 1 if not kw else iters)
    assert np.isfinite(s0).all()
    assert np.array_equal(s0.view(np.uint64), s1.view(np.uint64))
    assert len(f0) == len(f1)
    for a, b in zip(f0, f1):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


# An odd width (held, not queued ahead), one block, halo depth 3, passes with
# consumed sums and with finishers (2052 blocks); 11 to 14 iterations leave 0,
# 1 and 2 updates held at the end.
@pytest.mark.parametrize("x,y,h,iters", [
    (125, 54, 2, 11), (20, 12, 2, 12), (128, 64, 2, 13), (130, 70, 3, 14), (1026, 1024, 2, 12)])
def test_held_updates_are_the_steps_one_by_one(x, y, h, iters):
    _check(x, y, h, iters)


@pytest.mark.parametrize("where", ["after_w", "after_ur", "end"])
@pytest.mark.parametrize("between", [
    ("read", "norm", "summary"), ("halos2", "u_halo", "halos2"), ("no_halo", "no_halo", "read"),
    ("cheby", "ppcg", "ppcg"), ("residual", "finalise", "residual"), ("ppcg", "cheby", "u_halo"),
    ("mixed", "mixed", "mixed")])
def test_held_updates_are_made_before_other_calls(between, where):
    _check(128, 64, 2, 14, between=between, where=where)


@pytest.mark.parametrize("where", ["after_w", "after_ur", "end"])
@pytest.mark.parametrize("x", [128, 127])
@pytest.mark.parametrize("between", [("mixed_w",) * 3, ("fcg_w",) * 3])
def test_held_updates_are_made_before_a_mixed_precision_one(between, x, where):
    _check(x, 64, 2, 14, between=between, where=where)

"""Solves where the spare buffers do not fit (TEA_HIP_EXTRA_BYTES limits what a
chunk may take beyond its fields): every solver runs in the memory it cannot do
without, after any other on the same chunk, with the scalars and fields of the
unlimited one bit for bit."""

import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
SMALL = 1 << 16   # scalars and, at these sizes, the coarse levels


def _chunk(x, y, limit):
    from exploringsycl_amd.chunk import DeviceChunk
    if limit is not None:
        os.environ["TEA_HIP_EXTRA_BYTES"] = str(int(limit))
    try:
        return DeviceChunk(x, y, 2)
    finally:
        os.environ.pop("TEA_HIP_EXTRA_BYTES", None)


def _field(x, y):
    return 8 * (x * y + x * y % 2)


def _cg(c, iters=11):
    rro = c.cg_init(2, 0.8, 1.3)
    c.local_halos(1, ["u", "p"])
    c.copy_u()
    out = [rro]
    for _ in range(iters):
        pw = c.cg_calc_w()
        rrn = c.cg_calc_ur(rro / pw)
        c.cg_calc_p(rrn / rro)
        c.local_halos(1, ["u", "p"])
        out += [pw, rrn]
        rro = rrn
    return out + [c.read(n) for n in ("u", "p", "r", "w")]


def _jacobi(c, sweeps=7):
    c.jacobi_init(1, 0.8, 1.3)
    c.copy_u()
    c.local_halos(1, ["u"])
    out = []
    for _ in range(sweeps):
        out.append(c.jacobi_iterate())
        c.local_halos(1, ["u"])
    return out + [c.read(n) for n in ("u", "r")]


def _cheby(c):
    out = _cg(c, 4)
    c.cheby_init(3.0)
    c.local_halos(1, ["u"])
    for _ in range(5):
        c.cheby_iterate(0.3, 0.4)
        c.local_halos(1, ["u"])
    return out + [c.read(n) for n in ("u", "p", "r", "w")]


def _ppcg(c):
    out = _cg(c, 4)
    c.ppcg_init(3.0)
    for _ in range(5):
        c.local_halos(1, ["sd"])
        c.ppcg_inner_iteration(0.3, 0.4)
    return out + [c.read(n) for n in ("u", "r", "sd")]


def _flexible(c, fcg):
    if fcg:
        from exploringsycl_amd.native import check
        check(c.lib.tea_hip_fcg_attach_sweeps(c.handle, 6, 8, 2), "attach")
        out = list(c.fcg_init(2, 0.8, 1.3))
        out.append(c.fcg_precondition(1))
    else:
        out = list(c.mpcg_init(2, 0.8, 1.3))
    alpha = beta = 0.0
    for it in range(11):
        if fcg:
            pw, pr = c.fcg_calc_w(alpha, it > 0, beta)
        else:
            pw, pr = c.mpcg_calc_w(alpha, it > 0, beta, it > 0)
        alpha = pr / pw
        rr, rx = (c.fcg_calc_r_precondition(alpha, 1) if fcg else c.mpcg_calc_r(alpha))
        beta = -rx / pw
        out += [pw, pr, rr, rx]
    return out + [c.read_mp(n) for n in ("p", "r", "w")] + [c.read("u")]


# Solver and the field buffers that it cannot do without.
SOLVERS = {"cg": (_cg, 0), "jacobi": (_jacobi, 0), "cheby": (_cheby, 2), "ppcg": (_ppcg, 2),
           "mixed": (lambda c: _flexible(c, False), 3.5),
           "fcg": (lambda c: _flexible(c, True), 4)}


def _run(x, y, solvers, limit):
    rng = np.random.default_rng(x)
    density, energy = rng.uniform(0.1, 100.0, x * y), rng.uniform(0.1, 25.0, x * y)
    out = []
    with _chunk(x, y, limit) as c:
        for name in solvers:
            c.write("density", density)
            c.write("energy", energy)
            out += SOLVERS[name][0](c)
    return out


def _check(x, y, solvers, limit):
    want, got = _run(x, y, solvers, None), _run(x, y, solvers, limit)
    assert len(want) == len(got)
    for a, b in zip(want, got):
        a, b = np.atleast_1d(a), np.atleast_1d(b)
        assert a.dtype == b.dtype and np.array_equal(a.view(np.uint8), b.view(np.uint8))


# Rows of four cells, of two and odd; up to 2048 blocks and more.
SIZES = [(132, 68), (134, 68), (1028, 1028)]


@pytest.mark.parametrize("x,y", SIZES + [(133, 69)])
@pytest.mark.parametrize("name", [n for n in SOLVERS if n != "fcg"])
def test_solves_in_what_it_cannot_do_without(name, x, y):
    """From the least memory, in steps of half a field (one FP32 buffer), until
    every spare buffer fits: each buffer in turn is the first refused."""
    need = SOLVERS[name][1]
    for halves in range(15):
        _check(x, y, [name], (need + halves / 2) * _field(x, y) + SMALL // 2)


@pytest.mark.parametrize("x,y", [(132, 68), (1028, 1028)])
def test_fcg_solves_in_what_it_cannot_do_without(x, y):
    for halves in range(12):
        _check(x, y, ["fcg"], (4 + halves / 2) * _field(x, y) + (x * y) // 2 + SMALL)


@pytest.mark.parametrize("order", [
    ("cg", "mixed", "fcg", "cheby", "cg"), ("jacobi", "fcg", "ppcg", "mixed"),
    ("mixed", "cg", "jacobi", "fcg"), ("fcg", "jacobi", "cheby", "mixed", "jacobi")])
@pytest.mark.parametrize("x,y", [(132, 68), (1028, 1028)])
def test_spare_buffers_of_one_solver_make_room_for_another(x, y, order):
    need = 4 + (2 if "cheby" in order or "ppcg" in order else 0)
    for halves in (0, 1, 3, 6, 9):
        _check(x, y, order, (need + halves / 2) * _field(x, y) + (x * y) // 2 + SMALL)


def test_what_does_not_fit_is_refused_and_the_chunk_goes_on():
    from exploringsycl_amd.native import TeaHipError
    x, y = 132, 68
    want = _run(x, y, ["cg"], None)
    rng = np.random.default_rng(x)
    density, energy = rng.uniform(0.1, 100.0, x * y), rng.uniform(0.1, 25.0, x * y)
    with _chunk(x, y, 3 * _field(x, y)) as c:
        c.write("density", density)
        c.write("energy", energy)
        with pytest.raises(TeaHipError, match=r"\(-3\)"):
            c.mpcg_init(2, 0.8, 1.3)
        got = _cg(c)
    for a, b in zip(want, got):
        assert np.array_equal(np.atleast_1d(a).view(np.uint8), np.atleast_1d(b).view(np.uint8))


@pytest.mark.parametrize("room", [0.1, 0.6, 0.97])
@pytest.mark.parametrize("net", [False, True])
def test_an_attach_that_fails_half_way_leaves_no_level(net, room):
    """The coarse levels take less than a field: with `room` of what they need
    some of their buffers are there (with 0.97 the first level's) and the attach
    fails; the Jacobi preconditioner goes on."""
    from exploringsycl_amd import learned
    from exploringsycl_amd.native import TeaHipError, check
    x, y = 1028, 516   # two levels, of 128 x 64 and 32 x 16 cells
    coarse = 4 * (128 * 64 + 32 * 16) * (8 if net else 4)
    rng = np.random.default_rng(x)
    with _chunk(x, y, 4 * _field(x, y) + 64 + room * coarse) as c:
        c.write("density", rng.uniform(0.1, 100.0, x * y))
        c.write("energy", rng.uniform(0.1, 25.0, x * y))
        c.mpcg_init(2, 0.8, 1.3)
        with pytest.raises(TeaHipError, match=r"\(-3\)"):
            if net:
                params, norm, coarsen = learned.read_weights()
                c.fcg_attach(params, norm, coarsen=coarsen, levels=2)
            else:
                check(c.lib.tea_hip_fcg_attach_sweeps(c.handle, 6, 8, 2), "attach")
        assert c.fcg_levels() == 0
        c.fcg_init(2, 0.8, 1.3)
        with pytest.raises(TeaHipError, match="no coarse correction"):
            c.fcg_precondition(1)
        assert np.isfinite(c.fcg_precondition(0))

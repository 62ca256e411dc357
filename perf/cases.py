"""What this framework is used for, as cases that can be timed.

A solve case is one TeaLeaf timestep on one GPU, called as the host program
calls it (exploringsycl_amd/host/diffuse.cpp and the drivers beside it): the
C ABI of include/tea_hip.h, one call per step of the solver, the scalars of
every iteration formed on the host.  `prepare` makes the chunk, the mesh and
the states (and loads the network where the solver has one), which a program
does once per run; `run` is the timestep: energy reset, depth-2 halos, the
solver, energy = u / density and the field summary.  The outputs are the
temperature field u and the energy on the interior, in device memory, the
four sums of the field summary, and for the FP64 solvers, whose stop test is
on a number that is part of the interface, the iteration count.

The other two kinds are the network of the learned preconditioner: one epoch
of training on a resident set (forward, backward and Adam), and inference
from and to host memory.

Sizes come from the decks of the repository's tests and benchmark: 64 to
4096 cells a side with the tea.in states, seeded rectangles of density
uniform in [0.1, 100] or log10 density uniform in [-1, 2] or [-2, 2], K =
density or 1 / density, and the 256^2 training windows (32^2 on the coarse grid) in
batches of 64.
"""

import ctypes
import math

import numpy as np
import torch
import torch.nn.functional as F

from exploringsycl_amd import learned, native
from exploringsycl_amd.chunk import DeviceChunk
from exploringsycl_amd.deck import TEA_IN_STATES, seeded_rectangles
from exploringsycl_amd.native import FIELD_ID, HALO_SLOTS, check
from exploringsycl_amd.nn import LAYER_SHAPES, Net

HALO = 2
DT = 0.004
REFRESH = 50        # FP64 true-residual refresh of the mixed-precision solvers
PRESTEPS = 30       # CG steps before Chebyshev or PPCG (the host's default)
INNER = 10          # PPCG inner steps
REL = 1e-10
# Laws of the rectangles' density: the benchmark's, the mixed-precision
# workload's and the time-to-solution field's.
DENSITY = {"uniform": ("uniform", 0.1, 100.0), "log10": ("log10", -1.0, 2.0),
           "stiff": ("log10", -2.0, 2.0)}


def _solve(name, solver, nx, ny, iters, rects=0, density="uniform", coef="inverse",
           extent=10.0, eps=0.0, coarse="", work_iters=0):
    """iters caps the iterations (sweeps, Chebyshev steps, PPCG outer steps);
    eps > 0 is the solver's own stop test, absolute for cg, relative for the
    flexible solvers; work_iters is about what it takes to get there."""
    c = dict(kind="solve", solver=solver, nx=nx, ny=ny, iters=iters, rects=rects,
             density=density, coef=coef, extent=extent, eps=eps, coarse=coarse,
             work_iters=work_iters or iters)
    if name:
        c["name"] = name
    return c


def _net(name, kind, batch, height, width, samples):
    c = dict(kind=kind, batch=batch, height=height, width=width, samples=samples)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest deck in use (tea.problems 64^2): every call is latency.
        _solve("cg_64", "cg", 64, 64, 1000, coef="density", eps=1e-15, work_iters=67),
        # A timestep of the CPU-sized deck, tea.in states, solved to its end.
        _solve("cg_512", "cg", 512, 512, 2000, coef="density", eps=1e-15, work_iters=580),
        # A grid with odd sides, as a user's mesh has them.
        _solve("cg_1001x777", "cg", 1001, 777, 100, rects=16),
        # The benchmark field: 4096^2, 16 rectangles, K = 1 / density.
        _solve("cg_4096", "cg", 4096, 4096, 100, rects=16),
        # Mixed precision to 1e-10 on its own workload's field, a middling size.
        _solve("mpcg_1024", "mpcg", 1024, 1024, 6000, rects=32, density="log10", eps=REL,
               work_iters=2300),
        # Time to solution with the learned preconditioner: the headline.
        _solve("fcg_net_4096", "fcg", 4096, 4096, 3000, rects=64, density="stiff",
               eps=REL, coarse="net", work_iters=1115),
        # The two-level preconditioner with Jacobi sweeps, not square.
        _solve("fcg_sweeps_2048x1536", "fcg", 2048, 1536, 3000, rects=64, density="stiff",
               extent=5.0, eps=REL, coarse="sweeps", work_iters=680),
        # The other solvers of the reference's boundary.
        _solve("cheby_2048", "cheby", 2048, 2048, 200, coef="density"),
        _solve("ppcg_1100x900", "ppcg", 1100, 900, 20, coef="density"),
        _solve("jacobi_1000", "jacobi", 1000, 1000, 200, coef="density"),
        # Training as the shipped network was trained, and its inference.
        _net("train_64x32x32", "train", 64, 32, 32, 1024),
        _net("infer_64x32x32", "infer", 64, 32, 32, 64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cg", "cg", "cg", "mpcg", "jpcg", "sweeps", "net", "cheby", "ppcg",
                       "jacobi", "train", "infer"])
    if kind == "train":
        return _net(None, "train", rng.choice([16, 32, 64]), 32, 32, 64 * rng.randint(2, 24))
    if kind == "infer":
        b = rng.randint(1, 64)
        return _net(None, "infer", b, rng.choice([16, 32, 48, 64]), 32 * rng.randint(1, 4), b)
    if kind in ("sweeps", "net"):
        # One coarse level, or two where 32 divides both sides; the network
        # needs a coarse width that is a multiple of 32.
        nx = 256 * rng.randint(1, 6) if kind == "net" else 8 * _log_int(rng, 16, 256)
        ny = 8 * _log_int(rng, 16, 192)
        extent = 10.0 * max(nx, ny) / 4096
        return _solve(None, "fcg", nx, ny, 4000, rects=64, density="stiff", extent=extent,
                      eps=REL, coarse=kind, work_iters=1000)
    nx, ny = _log_int(rng, 10, 3000), _log_int(rng, 10, 3000)
    coef = rng.choice(["density", "inverse"])
    if kind in ("mpcg", "jpcg"):
        # No more than the stiff 1024^2 solve costs, to 1e-10.
        nx, ny = _log_int(rng, 32, 1024), _log_int(rng, 32, 1024)
        return _solve(None, "mpcg" if kind == "mpcg" else "fcg", nx, ny, 6000, rects=32,
                      density="log10", eps=REL, work_iters=max(nx, ny))
    iters = int(min(300, max(20, 3e9 / (nx * ny) / 5)))
    if kind == "ppcg":
        iters = max(2, iters // 10)
    return _solve(None, kind, nx, ny, iters, rects=rng.randint(0, 32), coef=coef)


# ---- the problem -----------------------------------------------------------

def _states(case, seed):
    """tea.in's states and the case's rectangles, scaled to its extent, as the
    parser leaves them (rectangles shrunk by a hundredth of a cell).  The
    tea.in energies are scaled by a seeded factor per state."""
    f = case["extent"] / 10.0
    scale = np.random.default_rng(seed).uniform(0.5, 1.5, len(TEA_IN_STATES))
    states = []
    for s, k in zip(TEA_IN_STATES, scale):
        states.append({**s, "energy": s["energy"] * float(k),
                       **{q: s[q] * f for q in ("xmin", "xmax", "ymin", "ymax") if q in s}})
    if case["rects"]:
        law, lo, hi = DENSITY[case["density"]]
        states += seeded_rectangles(case["rects"], 1000003 * (seed + 1), density=law,
                                    density_range=(lo, hi), domain=(0.0, case["extent"]))
    dx, dy = _steps(case)[:2]
    return [dict(density=s["density"], energy=s["energy"],
                 x_min=s.get("xmin", 0.0) + dx / 100.0, x_max=s.get("xmax", 0.0) - dx / 100.0,
                 y_min=s.get("ymin", 0.0) + dy / 100.0, y_max=s.get("ymax", 0.0) - dy / 100.0)
            for s in states]


def _steps(case):
    dx, dy = case["extent"] / case["nx"], case["extent"] / case["ny"]
    return dx, dy, DT / (dx * dx), DT / (dy * dy)


class _DeviceArray:
    """A field's device memory, for torch to look at."""

    def __init__(self, chunk, name):
        ptr, _ = chunk.field_info(name)
        self.owner = chunk
        self.__cuda_array_interface__ = dict(shape=(chunk.y, chunk.x), typestr="<f8",
                                             data=(ptr, False), version=2)


class _Gpu:
    """The steps of the solvers on a chunk, through the C ABI."""

    def __init__(self, case, seed):
        dx, dy, self.rx, self.ry = _steps(case)
        self.coef = native.CONDUCTIVITY if case["coef"] == "density" else \
            native.RECIP_CONDUCTIVITY
        self.chunk = c = DeviceChunk(case["nx"] + 2 * HALO, case["ny"] + 2 * HALO, HALO)
        c.set_chunk_data(0.0, 0.0, dx, dy)
        c.set_chunk_state(_states(case, seed))
        c.local_halos(2, ["density", "energy0", "energy1"])
        c.store_energy()
        self.use_coarse = case["coarse"] != ""
        if case["solver"] == "fcg":
            if case["coarse"] == "net":
                params, norm, coarsen = learned.read_weights()
                c.fcg_attach(params, norm, coarsen=coarsen, levels=2)
            elif case["coarse"] == "sweeps":
                check(c.lib.tea_hip_fcg_attach_sweeps(c.handle, 6, 8, 2), "attach_sweeps")
            else:
                c.fcg_attach()
        self.lib, self.h = c.lib, c.handle
        self.v = [ctypes.c_double() for _ in range(4)]
        self.p = [ctypes.byref(v) for v in self.v]
        self.r = ctypes.c_void_p()
        self.faces = (ctypes.c_int * 4)(-1, -1, -1, -1)
        self.masks = {}

    def halos(self, depth, *fields):
        m = self.masks.get(fields)
        if m is None:
            m = self.masks[fields] = (ctypes.c_int * 6)(*[int(s in fields) for s in HALO_SLOTS])
        check(self.lib.tea_hip_local_halos(self.h, depth, self.faces, m))

    def start(self):
        check(self.lib.tea_hip_store_energy(self.h))
        self.halos(2, "density", "energy1")

    def finish(self):
        check(self.lib.tea_hip_finalise(self.h))
        self.halos(1, "energy1")
        check(self.lib.tea_hip_field_summary(self.h, *self.p))
        check(self.lib.tea_hip_flush(self.h))
        inner = (slice(HALO, -HALO), slice(HALO, -HALO))
        fields = [torch.as_tensor(_DeviceArray(self.chunk, n), device="cuda")[inner]
                  for n in ("u", "energy")]
        return fields, [v.value for v in self.v]

    def _out(self, status, n):
        check(status)
        v = self.v
        return v[0].value if n == 1 else tuple(a.value for a in v[:n])

    def cg_init(self):
        return self._out(self.lib.tea_hip_cg_init(self.h, self.coef, self.rx, self.ry,
                                                  self.p[0]), 1)

    def cg_calc_w(self):
        return self._out(self.lib.tea_hip_cg_calc_w(self.h, self.p[0]), 1)

    def cg_calc_ur(self, alpha):
        return self._out(self.lib.tea_hip_cg_calc_ur(self.h, alpha, self.p[0]), 1)

    def cg_calc_p(self, beta):
        check(self.lib.tea_hip_cg_calc_p(self.h, beta))

    def copy_u(self):
        check(self.lib.tea_hip_copy_u(self.h))

    def residual(self):
        check(self.lib.tea_hip_calculate_residual(self.h))

    def norm_r(self):
        check(self.lib.tea_hip_field(self.h, FIELD_ID["r"], ctypes.byref(self.r), None))
        return self._out(self.lib.tea_hip_calculate_2norm(self.h, self.r, self.p[0]), 1)

    def jacobi_init(self):
        check(self.lib.tea_hip_jacobi_init(self.h, self.coef, self.rx, self.ry))

    def jacobi_iterate(self):
        return self._out(self.lib.tea_hip_jacobi_iterate(self.h, self.p[0]), 1)

    def cheby_init(self, theta):
        check(self.lib.tea_hip_cheby_init(self.h, theta))

    def cheby_iterate(self, a, b):
        check(self.lib.tea_hip_cheby_iterate(self.h, a, b))

    def ppcg_init(self, theta):
        check(self.lib.tea_hip_ppcg_init(self.h, theta))

    def ppcg_inner(self, a, b):
        check(self.lib.tea_hip_ppcg_inner_iteration(self.h, a, b))

    def mpcg_init(self):
        return self._out(self.lib.tea_hip_mpcg_init(self.h, self.coef, self.rx, self.ry,
                                                    self.p[0], self.p[1]), 2)

    def mpcg_calc_w(self, alpha, apply_u, beta, apply_p):
        return self._out(self.lib.tea_hip_mpcg_calc_w(self.h, alpha, apply_u, beta, apply_p,
                                                      self.p[0], self.p[1]), 2)

    def mpcg_calc_r(self, alpha):
        return self._out(self.lib.tea_hip_mpcg_calc_r(self.h, alpha, self.p[0], self.p[1]), 2)

    def mpcg_refresh(self, alpha):
        return self._out(self.lib.tea_hip_mpcg_refresh(self.h, alpha, 1, *self.p[:3]), 3)

    def fcg_init(self):
        return self._out(self.lib.tea_hip_fcg_init(self.h, self.coef, self.rx, self.ry,
                                                   self.p[0], self.p[1]), 2)

    def fcg_precondition(self):
        return self._out(self.lib.tea_hip_fcg_precondition(self.h, self.use_coarse,
                                                           self.p[0]), 1)

    def fcg_calc_r_precondition(self, alpha):
        return self._out(self.lib.tea_hip_fcg_calc_r_precondition(
            self.h, alpha, self.use_coarse, self.p[0], self.p[1]), 2)

    def fcg_calc_w(self, alpha, apply_u, beta):
        return self._out(self.lib.tea_hip_fcg_calc_w(self.h, alpha, apply_u, beta, self.p[0],
                                                     self.p[1]), 2)


class _Plain:
    """The same steps of the FP64 solvers in plain torch, 64 bits."""

    def __init__(self, case, seed):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        nx, ny = case["nx"], case["ny"]
        self.dx, self.dy, rx, ry = _steps(case)
        xv = self.dx * torch.arange(nx + 1, dtype=torch.float64, device=self.dev)[None, :]
        yv = self.dy * torch.arange(ny + 1, dtype=torch.float64, device=self.dev)[:, None]
        self.rho = self.energy0 = None
        for s in _states(case, seed):
            if self.rho is None:
                self.rho = torch.full((ny, nx), s["density"], dtype=torch.float64,
                                      device=self.dev)
                self.energy0 = torch.full_like(self.rho, s["energy"])
                continue
            inside = ((xv[:, 1:] >= s["x_min"]) & (xv[:, :-1] < s["x_max"]) &
                      (yv[1:] >= s["y_min"]) & (yv[:-1] < s["y_max"]))
            self.rho[inside] = s["density"]
            self.energy0[inside] = s["energy"]
        self.k = k = self.rho if case["coef"] == "density" else 1.0 / self.rho
        self.rx, self.ry = rx, ry
        self.kx = torch.zeros((ny, nx + 1), dtype=torch.float64, device=self.dev)
        self.ky = torch.zeros((ny + 1, nx), dtype=torch.float64, device=self.dev)
        self.kx[:, 1:-1] = rx * (k[:, :-1] + k[:, 1:]) / (2.0 * k[:, :-1] * k[:, 1:])
        self.ky[1:-1, :] = ry * (k[:-1] + k[1:]) / (2.0 * k[:-1] * k[1:])

    def start(self):
        pass

    def halos(self, depth, *fields):
        pass

    def finish(self):
        v = self.dx * self.dy
        sums = [float(v * self.rho.numel()), float((v * self.rho).sum()),
                float((v * self.rho * self.energy0).sum()), float((v * self.rho * self.u).sum())]
        return [self.u, self.u / self.rho], sums

    def _a(self, u):
        # Zero flux through the domain's faces.
        fx, fy = torch.zeros_like(self.kx), torch.zeros_like(self.ky)
        fx[:, 1:-1] = self.kx[:, 1:-1] * (u[:, 1:] - u[:, :-1])
        fy[1:-1] = self.ky[1:-1] * (u[1:] - u[:-1])
        return u - (fx[:, 1:] - fx[:, :-1]) - (fy[1:] - fy[:-1])

    def cg_init(self):
        self.u = self.energy0 * self.rho
        self.u0 = self.u.clone()
        self.r = self.u - self._a(self.u)
        self.p = self.r.clone()
        return float((self.r * self.r).sum())

    def cg_calc_w(self):
        self.w = self._a(self.p)
        return float((self.p * self.w).sum())

    def cg_calc_ur(self, alpha):
        self.u = self.u + alpha * self.p
        self.r = self.r - alpha * self.w
        return float((self.r * self.r).sum())

    def cg_calc_p(self, beta):
        self.p = beta * self.p + self.r

    def copy_u(self):
        self.u0 = self.u.clone()

    def residual(self):
        self.r = self.u0 - self._a(self.u)

    def norm_r(self):
        return float((self.r * self.r).sum())

    def jacobi_init(self):
        self.u = self.energy0 * self.rho
        # The diagonal with the domain's faces, whose mirrored neighbours
        # stand for themselves in the sweep: r (k + k) / (2 k k) there.
        k, d = self.k, 1.0 + self.kx[:, 1:] + self.kx[:, :-1] + self.ky[1:] + self.ky[:-1]
        d[:, 0] += self.rx / k[:, 0]
        d[:, -1] += self.rx / k[:, -1]
        d[0] += self.ry / k[0]
        d[-1] += self.ry / k[-1]
        self.diag = d

    def jacobi_iterate(self):
        old = self.u
        self.u = old + (self.u0 - self._a(old)) / self.diag
        return float((self.u - old).abs().sum())

    def cheby_init(self, theta):
        self.r = self.u0 - self._a(self.u)
        self.p = self.r / theta

    def cheby_iterate(self, a, b):
        self.r = self.u0 - self._a(self.u)
        self.p = a * self.p + b * self.r
        self.u = self.u + self.p

    def ppcg_init(self, theta):
        self.sd = self.r / theta

    def ppcg_inner(self, a, b):
        self.r = self.r - self._a(self.sd)
        self.u = self.u + self.sd
        self.sd = a * self.sd + b * self.r


# ---- the drivers' control flow ---------------------------------------------

def _cg_start(e):
    rro = e.cg_init()
    e.halos(1, "u", "p")
    e.copy_u()
    return rro


def _cg_step(e, rro, halo):
    pw = e.cg_calc_w()
    alpha = rro / pw
    rrn = e.cg_calc_ur(alpha)
    beta = rrn / rro
    e.cg_calc_p(beta)
    e.halos(1, *halo)
    return rrn, alpha, beta


def _run_cg(e, case):
    rro = _cg_start(e)
    for it in range(case["iters"]):
        rro = _cg_step(e, rro, ("u", "p"))[0]
        if math.sqrt(abs(rro)) < case["eps"]:
            break
    return it + 1


def _chebyshev(e, count):
    """PRESTEPS CG steps, then theta and the coefficients of the Chebyshev
    iteration on the Lanczos matrix's extreme eigenvalues, widened by 5%."""
    rro = _cg_start(e)
    al, be = [], []
    for _ in range(PRESTEPS):
        rro, a, b = _cg_step(e, rro, ("u", "p"))
        al.append(a)
        be.append(b)
    t = np.zeros((PRESTEPS, PRESTEPS))
    for k in range(PRESTEPS):
        t[k, k] = 1.0 / al[k] + (be[k - 1] / al[k - 1] if k else 0.0)
        if k + 1 < PRESTEPS:
            t[k, k + 1] = t[k + 1, k] = math.sqrt(be[k]) / al[k]
    eig = np.linalg.eigvalsh(t)
    lo, hi = 0.95 * float(eig[0]), 1.05 * float(eig[-1])
    theta, delta = (hi + lo) / 2.0, (hi - lo) / 2.0
    sigma = theta / delta
    prev, coef = 1.0 / sigma, []
    for _ in range(count):
        rho = 1.0 / (2.0 * sigma - prev)
        coef.append((rho * prev, 2.0 * rho / delta))
        prev = rho
    return rro, theta, coef


def _run_cheby(e, case):
    _, theta, coef = _chebyshev(e, case["iters"])
    e.cheby_init(theta)
    e.halos(1, "u")
    for k in range(1, case["iters"]):
        e.cheby_iterate(*coef[k])
        if k % 50 == 0:
            e.norm_r()
        e.halos(1, "u")
    return case["iters"]


def _run_ppcg(e, case):
    rro, theta, coef = _chebyshev(e, INNER)
    e.residual()
    e.halos(1, "p")
    for _ in range(case["iters"]):
        alpha = rro / e.cg_calc_w()
        e.cg_calc_ur(alpha)
        e.ppcg_init(theta)
        for a, b in coef:
            e.halos(1, "sd")
            e.ppcg_inner(a, b)
        rrn = e.norm_r()
        e.cg_calc_p(rrn / rro)
        e.halos(1, "p")
        rro = rrn
    return case["iters"]


def _run_jacobi(e, case):
    e.jacobi_init()
    e.copy_u()
    e.halos(1, "u")
    for it in range(case["iters"]):
        e.jacobi_iterate()
        if it % 50 == 0:
            e.halos(1, "u")
            e.residual()
            e.norm_r()
        e.halos(1, "u")
    return case["iters"]


def _run_mpcg(e, case):
    _, bb = e.mpcg_init()
    tol2 = case["eps"] ** 2 * bb
    alpha = beta = 0.0
    apply_u = apply_p = False
    since = 0
    for _ in range(case["iters"]):
        pw, pr = e.mpcg_calc_w(alpha, apply_u, beta, apply_p)
        alpha = pr / pw
        rr, rw = e.mpcg_calc_r(alpha)
        apply_u = True
        since += 1
        if since >= REFRESH or rr < tol2:
            rr, rr_true, rw = e.mpcg_refresh(alpha)
            apply_u, since = False, 0
            if rr_true < tol2:
                break
        beta = -rw / pw
        apply_p = True
    if apply_u:
        e.mpcg_refresh(alpha)


def _run_fcg(e, case):
    _, bb = e.fcg_init()
    tol2 = case["eps"] ** 2 * bb
    zw = e.fcg_precondition()
    alpha = beta = 0.0
    apply_u = False
    since = 0
    for _ in range(case["iters"]):
        pw, pr = e.fcg_calc_w(alpha, apply_u, beta)
        alpha = pr / pw
        rr, zw = e.fcg_calc_r_precondition(alpha)
        apply_u = True
        since += 1
        if since >= REFRESH or rr < tol2:
            rr, rr_true, _ = e.mpcg_refresh(alpha)
            apply_u, since = False, 0
            if rr_true < tol2:
                break
            zw = e.fcg_precondition()
        beta = -zw / pw
    if apply_u:
        e.mpcg_refresh(alpha)


_RUN = dict(cg=_run_cg, cheby=_run_cheby, ppcg=_run_ppcg, jacobi=_run_jacobi, mpcg=_run_mpcg,
            fcg=_run_fcg)


# ---- the network -----------------------------------------------------------

def _samples(case, seed):
    """Inputs and targets of the training set's kind: a scaled residual of
    unit RMS, smooth and rough, two normalised features that are constant on
    rectangles, and a target of the residual's size."""
    n, h, w = case["samples"], case["height"], case["width"]
    rng = np.random.default_rng(seed)
    rough = rng.standard_normal((n, h, w), dtype=np.float32)
    smooth = rough.copy()
    for _ in range(2):
        smooth = 0.2 * (smooth + np.roll(smooth, 1, 1) + np.roll(smooth, -1, 1) +
                        np.roll(smooth, 1, 2) + np.roll(smooth, -1, 2))
    mix = rng.uniform(0.0, 1.0, (n, 1, 1)).astype(np.float32)
    res = mix * rough + (1.0 - mix) * 3.0 * smooth
    res /= np.sqrt(np.mean(res * res, axis=(1, 2), keepdims=True)) + 1e-6
    feat = np.zeros((n, h, w, 2), dtype=np.float32)
    for _ in range(4):
        a, b = np.sort(rng.integers(0, h + 1, 2)), np.sort(rng.integers(0, w + 1, 2))
        feat[:, a[0]:a[1], b[0]:b[1]] = rng.standard_normal((n, 1, 1, 2), dtype=np.float32)
    x = np.concatenate([res[..., None], feat], axis=3).astype(np.float32)
    t = (res + 2.0 * smooth).astype(np.float32)
    return x, t


def _forward64(x, params):
    """The network in 64 bits; params a list of (weight, bias)."""
    a = x.permute(0, 3, 1, 2)
    for i, (wt, b) in enumerate(params):
        cols = F.unfold(a, 3, padding=1)
        a = (torch.matmul(wt.reshape(wt.shape[0], -1), cols) + b[:, None]).reshape(
            a.shape[0], wt.shape[0], a.shape[2], a.shape[3])
        if i + 1 < len(params):
            a = torch.relu(a)
    return a[:, 0]


def _split(flat, dev):
    out, at = [], 0
    for o, i in LAYER_SHAPES:
        n = o * i * 9
        wt = torch.tensor(flat[at:at + n].reshape(o, i, 3, 3), dtype=torch.float64, device=dev)
        b = torch.tensor(flat[at + n:at + n + o], dtype=torch.float64, device=dev)
        out.append((wt, b))
        at += n + o
    return out


def _train64(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x, t = _samples(case, seed)
    x, t = (torch.tensor(v, dtype=torch.float64, device=dev) for v in (x, t))
    params = _split(learned.initial_params(seed), dev)
    flat = [v.requires_grad_(True) for pair in params for v in pair]
    opt = torch.optim.Adam(flat, lr=1e-3, betas=(0.9, 0.999), eps=1e-8)
    order, losses = _order(case, seed), []
    for s in range(0, len(order), case["batch"]):
        ids = torch.tensor(order[s:s + case["batch"]], dtype=torch.long, device=dev)
        opt.zero_grad()
        loss = ((_forward64(x[ids], params) - t[ids]) ** 2).mean()
        loss.backward()
        opt.step()
        losses.append(float(loss.detach()))
    return [torch.cat([v.detach().reshape(-1) for v in flat]), float(np.mean(losses))]


def _order(case, seed):
    order = np.random.default_rng(seed + 1).permutation(case["samples"]).astype(np.int32)
    return order[:len(order) // case["batch"] * case["batch"]]


# ---- the cases' functions --------------------------------------------------

def prepare(case, seed):
    if case["kind"] == "solve":
        return dict(case=case, engine=_Gpu(case, seed))
    net = Net(case["batch"], case["height"], case["width"])
    x, t = _samples(case, seed)
    if case["kind"] == "train":
        net.load_dataset(x, t)
        return dict(case=case, net=net, params=learned.initial_params(seed),
                    order=_order(case, seed))
    net.set_params(learned.read_weights()[0])
    return dict(case=case, net=net, x=x)


def run(state):
    case = state["case"]
    if case["kind"] == "train":
        net = state["net"]
        net.set_params(state["params"])
        loss = net.train_epoch(state["order"], case["batch"], 1e-3)
        return [net.get_params(), loss]
    if case["kind"] == "infer":
        return [state["net"].forward(state["x"])]
    e = state["engine"]
    e.start()
    iters = _RUN[case["solver"]](e, case)
    fields, sums = e.finish()
    # The flexible solvers' counts follow the rounding of the preconditioner.
    return [*fields, *sums] + ([iters] if iters is not None else [])


def exact(case, seed):
    if case["kind"] == "train":
        return _train64(case, seed)
    if case["kind"] == "infer":
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        x = torch.tensor(_samples(case, seed)[0], dtype=torch.float64, device=dev)
        return [_forward64(x, _split(learned.read_weights()[0], dev))]
    if case["solver"] in ("mpcg", "fcg"):
        # The solution itself, by CG to well below their stop test.
        if case["nx"] * case["ny"] > 4 << 20:
            return None
        e = _Plain(case, seed)
        rro = _cg_start(e)
        bb = float((e.u0 * e.u0).sum())
        for _ in range(20000):
            rro = _cg_step(e, rro, ())[0]
            if rro < 1e-26 * bb:
                break
        fields, sums = e.finish()
        return [*fields, *sums]
    e = _Plain(case, seed)
    _RUN[case["solver"]](e, case)
    fields, sums = e.finish()
    return [*fields, *sums, None]


def work(case):
    if case["kind"] != "solve":
        px = case["samples"] * case["height"] * case["width"]
        macs = sum(9 * o * i for o, i in LAYER_SHAPES)
        nparam = sum(o * i * 9 + o for o, i in LAYER_SHAPES)
        if case["kind"] == "train":
            # Inputs, targets and parameters in; parameters out.
            return {"bytes": px * 16 + 8 * nparam, "flops": 6 * macs * px}
        return {"bytes": px * 16, "flops": 2 * macs * px}
    cells, n = case["nx"] * case["ny"], case["work_iters"]
    # Per iteration each array of the recursion once in and, where it
    # changes, once out: cg reads u, p, r, kx, ky and writes u, p, r (FP64);
    # the mixed-precision ones keep all but u in FP32; a Chebyshev or PPCG
    # inner step and a Jacobi sweep likewise.
    words = dict(cg=(64, 22), mpcg=(40, 26), fcg=(40, 34), cheby=(64, 20), ppcg=(56, 20),
                 jacobi=(40, 14))[case["solver"]]
    if case["solver"] == "ppcg":
        n *= INNER + 1
    flops = words[1] * cells * n
    if case["coarse"] == "net":
        flops += 2 * sum(9 * o * i for o, i in LAYER_SHAPES) * cells // 64 * n
    return {"bytes": words[0] * cells * n + 48 * cells, "flops": flops}

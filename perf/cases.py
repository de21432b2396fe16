"""Performance cases: what a user of the framework has it do, from one cell to a full grid.

A case is a dict of plain values.  `kind` names the entry points it goes through:

  cell      one cell through the drop-in kernel calls of the generated solver glue
  grid      a device-resident ADER-DG grid: set-up, time steps, the solution back
  limiter   the same with the a-posteriori subcell limiter (a blast)
  fv        the stand-alone finite-volumes grid
  patches   many uneven independent patches with a time step of their own
  amr       every cell of a level refined, and the fine level restricted back

The time-stepping kinds run whole jobs (initial condition on the device, K steps,
the solution into the caller's page-locked buffer), because that is the shortest
thing a program calls that hands results back.  `exact` restates the same jobs in
plain float64 torch.
"""
import ctypes
import math

import numpy as np
import torch

from exahype_amd import capi

PNPM = (1.0, 0.33, 0.17, 0.1, 0.069, 0.045, 0.038, 0.03, 0.02, 0.015)
GOLDEN = 0x9E3779B97F4A7C15
MASK = (1 << 64) - 1


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def grid_case(name, pde, order, n, steps, bits, periodic=True, linear=False, fused=False, plot=False):
    case = dict(kind="grid", pde=pde, order=order, nx=n[0], ny=n[1], nz=n[2], steps=steps, bits=bits,
                periodic=periodic, linear=linear, fused=fused, plot=plot)
    return dict(name=name, **case) if name else case


def listed():
    return [
        # A solver generated by the toolkit that calls the kernels cell by cell
        # (the drop-in boundary): twelve host calls for one cell's step.
        dict(name="cell_n3", kind="cell", order=3),
        # A small simulation of the smallest patch side (9^3): every launch counts.
        grid_case("euler_n3_9", "euler", 3, (9, 9, 9), 50, 64),
        # Double precision at the headline order on an uneven grid.
        grid_case("euler_n5_47x45x41_fp64", "euler", 5, (47, 45, 41), 8, 64),
        # The headline workload: 81^3 cells, order 5, FP32-bulk form.
        grid_case("euler_n5_81_fp32", "euler", 5, (81, 81, 81), 24, 32),
        # High order with open boundaries and fused time stepping, an odd grid,
        # and the vertex output of a plot at its end (order 6 is the plotter's highest).
        grid_case("euler_n6_27x19x13_fused_plot", "euler", 6, (27, 19, 13), 20, 32, periodic=False, fused=True,
                  plot=True),
        # Seismic workloads: linear elasticity, nonlinear kernels (both precisions
        # are in use) and the linear solver's kernels.
        grid_case("elastic_n4_41_fp64", "elastic", 4, (41, 41, 41), 8, 64),
        grid_case("elastic_n4_linear_45x37x41", "elastic", 4, (45, 37, 41), 8, 64, periodic=False, linear=True),
        # Shocks: the limiting solver on a small grid and on a large one.
        dict(name="limiter_n2_15", kind="limiter", order=2, nx=15, ny=15, nz=15, steps=25, fused=False, godunov=False),
        dict(name="limiter_n3_63x60x55", kind="limiter", order=3, nx=63, ny=60, nz=55, steps=16, fused=False,
             godunov=False),
        # The finite-volumes demonstrator's patch size, 27^3 cells of 10^3 subcells.
        dict(name="fv_godunov_27_L10", kind="fv", L=10, nx=27, ny=27, nz=27, steps=80, muscl=False, periodic=True),
        # A set of uneven patches with their own time steps.
        dict(name="patches_fp32", kind="patches", count=8, sides="9,15,27,27,9,15,9,15", orders="7,6,5,4,5,3,2,7",
             steps=30, bits=32, elastic=False),
        # Refinement of a whole level and its restriction back, order 5.
        dict(name="amr_n5_21", kind="amr", order=5, nx=21, ny=19, nz=17, delta=1),
    ]


def draw(rng):
    """One more case: the kinds of listed() over the sizes the framework is used at."""
    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def box(order, most):
        """Three sides of 5 to 60, scaled down to `most` nodes in all."""
        n = [side(5, 60) for _ in range(3)]
        while n[0] * n[1] * n[2] * (order + 1) ** 3 > most:
            n = [max(3, int(0.85 * v)) for v in n]
        return tuple(n)

    kind = rng.choice(("cell", "euler", "euler", "euler", "elastic", "elastic", "limiter", "limiter", "fv", "fv",
                       "patches", "amr"))
    if kind == "cell":
        return dict(kind="cell", order=rng.randint(2, 7))
    if kind == "euler":
        order, fused = rng.randint(2, 7), rng.random() < 0.3
        return grid_case(None, "euler", order, box(order, 15e6), rng.randint(4, 30), rng.choice((32, 64)),
                         periodic=rng.random() < 0.6, fused=fused, plot=order <= 6 and rng.random() < 0.2)
    if kind == "elastic":
        order, linear = rng.randint(2, 5), rng.random() < 0.5
        return grid_case(None, "elastic", order, box(order, 8e6), rng.randint(4, 20),
                         64 if linear else rng.choice((32, 64)), periodic=rng.random() < 0.5, linear=linear)
    if kind == "limiter":
        order = rng.randint(2, 3)
        n = box(order, 9e6)
        return dict(kind="limiter", order=order, nx=n[0], ny=n[1], nz=n[2], steps=rng.randint(6, 30),
                    fused=rng.random() < 0.3, godunov=rng.random() < 0.3)
    if kind == "fv":
        muscl = rng.random() < 0.4
        L = rng.choice((5, 7)) if muscl else rng.randint(4, 12)
        n = box(L - 1, 9e6 if muscl else 18e6)
        return dict(kind="fv", L=L, nx=n[0], ny=n[1], nz=n[2], steps=rng.randint(10, 80), muscl=muscl,
                    periodic=rng.random() < 0.6)
    if kind == "patches":
        count, elastic = rng.randint(3, 8), rng.random() < 0.3
        sides = [rng.choice((5, 9, 11, 15, 21, 27)) for _ in range(count)]
        orders = [rng.randint(2, 5 if elastic else 7) for _ in range(count)]
        return dict(kind="patches", count=count, sides=",".join(map(str, sides)), orders=",".join(map(str, orders)),
                    steps=rng.randint(10, 40), bits=rng.choice((32, 64)), elastic=elastic)
    order, delta = rng.randint(1, 5), 2 if rng.random() < 0.2 else 1
    n = tuple(side(4, 24) if delta == 1 else side(3, 8) for _ in range(3))
    return dict(kind="amr", order=order, nx=n[0], ny=n[1], nz=n[2], delta=delta)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def splitmix64(state):
    state = (state + GOLDEN) & MASK
    z = state
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & MASK
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & MASK
    return state, z ^ (z >> 31)


def euler_ic(seed):
    """A smooth moving density wave with eight small Fourier modes."""
    r = np.random.default_rng(seed)
    return dict(rho0=1.0, amp=float(r.uniform(0.1, 0.3)), k=tuple(int(v) for v in r.integers(1, 3, 3)),
                vel=tuple(float(v) for v in r.uniform(0.5, 1.0, 3)), p=float(r.uniform(0.9, 1.1)), nmodes=8,
                mode_amp=0.01, seed=int(r.integers(1, 1 << 40)))


def elastic_ic(seed):
    """The seeded two-layer material with a Gaussian velocity pulse."""
    r = np.random.default_rng(seed)
    return dict(seed=int(r.integers(1, 1 << 40)), width=float(r.uniform(0.08, 0.15)), amp=1.0)


def blast_ic(seed):
    r = np.random.default_rng(seed)
    return dict(seed=int(r.integers(1, 1 << 40)), radius=float(r.uniform(0.19, 0.22)), p_in=10.0, p_out=0.1,
                noise=0.01)


def dims(case):
    return case["nx"], case["ny"], case["nz"]


def solver(case):
    prec = capi.PRECISION_FP32_BULK if case.get("bits") == 32 else capi.PRECISION_FP64
    make = capi.elastic_solver if case.get("pde") == "elastic" else capi.euler_solver
    return make(case["order"], precision=prec, linear=case.get("linear", False))


def locked(n, dtype=torch.float64):
    """A page-locked host buffer, as a program that reads results back keeps one."""
    return torch.empty(n, dtype=dtype, pin_memory=torch.cuda.is_available())


def dptr(t):
    return ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_double))


def patch_specs(case, seed):
    r = np.random.default_rng(seed)
    out = []
    for n, order in zip(map(int, case["sides"].split(",")), map(int, case["orders"].split(","))):
        k, amp = tuple(int(v) for v in r.integers(1, 4, 3)), float(r.uniform(0.05, 0.3))
        if case["elastic"]:
            out.append(capi.elastic_patch(n, order, seed=int(r.integers(1, 1 << 40)), width=float(r.uniform(0.08, 0.15))))
        else:
            out.append((n, order, k, amp))
    return out


def amr_items(n, r):
    """Rows (fine block, coarse block, sx, sy, sz), coarse-major, of a level refined r times per direction."""
    nx, ny, nz = n
    c = np.arange(nx * ny * nz)
    s = np.arange(r ** 3)
    sx, sy, sz = s % r, (s // r) % r, s // (r * r)
    fi = (c % nx)[:, None] * r + sx
    fj = ((c // nx) % ny)[:, None] * r + sy
    fk = (c // (nx * ny))[:, None] * r + sz
    rows = [fi + nx * r * (fj + ny * r * fk), np.repeat(c[:, None], r ** 3, 1)] + [
        np.broadcast_to(v, fi.shape) for v in (sx, sy, sz)]
    return np.stack(rows, -1).reshape(-1, 5).astype(np.int32)


def cell_state(case, seed):
    """One cell's nodal values of a smooth flow, its size and a time step below the stable one."""
    B = case["order"] + 1
    r = np.random.default_rng(seed)
    x = gauss(B)[0]
    X = np.stack(np.meshgrid(x, x, x, indexing="ij"), -1)
    a = r.uniform(-1, 1, (5, 3))
    f = [0.05 * np.sin(X @ a[i] + i) for i in range(5)]
    rho, u = 1.0 + f[0], [0.5 + f[1], 0.3 + f[2], -0.4 + f[3]]
    p = 1.0 + f[4]
    Q = np.stack([rho, rho * u[0], rho * u[1], rho * u[2], p / 0.4 + 0.5 * rho * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)], -1)
    dx = 0.05 * (1.0 + 0.2 * r.uniform(0, 1, 3))
    return Q.ravel().copy(), dx, 0.8 * 0.9 * PNPM[case["order"]] * float(dx.min()) / 6.0


def prepare(case, seed):
    """What the program holds before the call: the grid, plan or arrays, the initial condition's
    parameters, and the buffers that results go to."""
    kind = case["kind"]
    st = dict(case=case)
    if kind == "cell":
        st["s"] = solver(case)
        st["luh"], st["dx"], st["dt"] = cell_state(case, seed)
    elif kind == "grid":
        s = solver(case)
        g = capi.Grid(s, dims(case), boundary=capi.BC_PERIODIC if case["periodic"] else capi.BC_TRANSMISSIVE)
        if case["fused"]:
            g.set_fused_time_stepping(True, 0.9)
        st.update(g=g, ic=elastic_ic(seed) if case["pde"] == "elastic" else euler_ic(seed),
                  luh=locked(g.ncells * s.B ** 3 * s.D))
        if case["plot"]:
            st["vertices"] = locked(g.ncells * s.B ** 3 * s.D)
    elif kind == "limiter":
        s = solver(case)
        g = capi.LimitingGrid(s, dims(case), fv_scheme=capi.FV_GODUNOV if case["godunov"] else capi.FV_MUSCLHANCOCK)
        st.update(g=g, ic=blast_ic(seed), luh=locked(g.ncells * s.B ** 3 * 5), status=locked(g.ncells, torch.int32))
    elif kind == "fv":
        g = capi.FVGrid(capi.euler_solver(3), case["L"], dims(case),
                        boundary=capi.BC_PERIODIC if case["periodic"] else capi.BC_TRANSMISSIVE,
                        scheme=capi.FV_MUSCLHANCOCK if case["muscl"] else capi.FV_GODUNOV)
        st.update(g=g, ic=euler_ic(seed), u=locked(g.size))
    elif kind == "patches":
        specs = patch_specs(case, seed)
        st["b"] = capi.PatchSet(specs, precision=capi.PRECISION_FP32_BULK if case["bits"] == 32 else capi.PRECISION_FP64,
                                keep_max_cells=10 ** 6)
    else:
        st.update(amr_arrays(case, seed, "cuda"))
        st["s"] = capi.euler_solver(case["order"])
        for k in ("fine", "acc"):
            st[k] = torch.empty_like(st["coarse"] if k == "acc" else st["values"])
        del st["values"]
    return st


def amr_arrays(case, seed, device):
    n, r, size = dims(case), 3 ** case["delta"], 5 * (case["order"] + 1) ** 3
    items = amr_items(n, r)
    gen = torch.Generator().manual_seed(int(seed))
    coarse = torch.randn(n[0] * n[1] * n[2], size, generator=gen, dtype=torch.float64)
    return dict(coarse=coarse.to(device), values=torch.empty(len(items), size, dtype=torch.float64, device=device),
                items=torch.from_numpy(items).to(device),
                back=torch.from_numpy(np.ascontiguousarray(items[:, [1, 0, 2, 3, 4]])).to(device),
                ptr=torch.arange(0, len(items) + 1, r ** 3, dtype=torch.int32, device=device))


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(st):
    case = st["case"]
    kind, L = case["kind"], capi.lib()
    if kind == "cell":
        return run_cell(st)
    if kind == "grid":
        g = st["g"]
        (g.init_elastic if case["pde"] == "elastic" else g.init_euler)(**st["ic"])
        g.step(case["steps"])
        out = [st["luh"]]
        capi.check(L.exa_grid_download_solution(g._h, dptr(st["luh"])), "download")
        if case["plot"]:
            capi.check(L.exa_grid_plot_vertices(g._h, dptr(st["vertices"]), None), "plot")
            out.append(st["vertices"])
        return out
    if kind == "limiter":
        g = st["g"]
        g.init_blast(**st["ic"])
        g.set_fused_time_stepping(case["fused"])
        g.step(case["steps"])
        capi.check(L.exa_lgrid_download(g._h, dptr(st["luh"])), "download")
        status = ctypes.cast(st["status"].data_ptr(), ctypes.POINTER(ctypes.c_int))
        capi.check(L.exa_lgrid_status(g._h, status, None), "status")
        return [st["luh"], st["status"]]
    if kind == "fv":
        g = st["g"]
        g.init_euler(**st["ic"])
        g.step(case["steps"])
        capi.check(L.exa_fvgrid_download(g._h, dptr(st["u"])), "download")
        return [st["u"]]
    if kind == "patches":
        b = st["b"]
        b.run(case["steps"])
        return [b.solution(j) for j in range(case["count"])]
    s, n = st["s"], len(st["items"])
    coarse, fine, acc = st["coarse"], st["fine"], st["acc"]
    capi.check(L.exa_volume_unknowns_prolongation_batch(
        ctypes.byref(s), fine.data_ptr(), n, coarse.data_ptr(), len(coarse), st["items"].data_ptr(), n, case["delta"],
        None), "prolongation")
    acc.zero_()
    capi.check(L.exa_volume_unknowns_restriction_batch(
        ctypes.byref(s), acc.data_ptr(), len(acc), fine.data_ptr(), n, st["ptr"].data_ptr(), len(acc),
        st["back"].data_ptr(), n, case["delta"], None), "restriction")
    return [fine, acc]


def run_cell(st):
    """One time step of a cell that neighbours itself, call by call."""
    s, luh, dx, dt = st["s"], st["luh"], st["dx"], st["dt"]
    B, V = s.B, s.num_variables
    p = capi.space_time_predictor_nonlinear(s, luh, dx, dt, temps=True)
    lduh = capi.volume_integral_nonlinear(s, p["lFhi"], dx)
    Q, F = p["lQhbnd"].reshape(6, -1), p["lFhbnd"].reshape(6, -1).copy()
    for d in range(3):
        F[2 * d + 1], F[2 * d] = capi.riemann_solver_nonlinear(s, F[2 * d + 1], F[2 * d], Q[2 * d + 1], Q[2 * d], dt, d)
    lduh = capi.surface_integral_nonlinear(s, lduh, F.ravel(), dx)
    new = capi.solution_update(s, luh, lduh, dt)
    return [p["lQhbnd"], p["lFhbnd"], lduh, new, np.array([capi.stable_time_step_size(s, new, dx)])]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def picard_iterations(case):
    return 1 if case.get("pde") == "elastic" else (2 if case.get("bits") == 32 else 3)


def step_work(order, V, D, iterations, ncp):
    """Bytes and operations of one cell's time step: the solution read and written once (the global
    time step lies between two steps); Picard iterations after the first, which needs the terms of
    one time slice only, the time averages, the face and volume operators."""
    B = order + 1
    slice_ = (6 * V * B + (42 + 3 * V if ncp else 40 + 4 * V)) * B ** 3
    flops = slice_ * (1 + B * (iterations - 1)) + 2 * V * B ** 5 * iterations
    flops += 2 * (3 * V + D) * B ** 4 + 12 * (D + V) * B ** 3 + 6 * V * B ** 4 + 12 * V * B ** 3
    return 8 * (D + V) * B ** 3, flops


def work(case):
    kind = case["kind"]
    if kind == "cell":
        by, fl = step_work(case["order"], 5, 5, 3, False)
        return dict(bytes=by, flops=fl)
    if kind in ("grid", "limiter"):
        B, V, D = case["order"] + 1, *((9, 12) if case.get("pde") == "elastic" else (5, 5))
        cells = case["nx"] * case["ny"] * case["nz"]
        if case.get("linear"):  # Cauchy-Kowalevski: B derivatives of 3 V gradients per node
            by, fl = 8 * (D + V) * B ** 3, B * (6 * V * B + 60) * B ** 3 + 12 * (D + V) * B ** 3 + 12 * V * B ** 3
        else:
            its = 2 if kind == "limiter" else picard_iterations(case)
            by, fl = step_work(case["order"], V, D, its, case.get("pde") == "elastic")
        out = 8 * cells * D * B ** 3 * (2 if case.get("plot") else 1)
        return dict(bytes=cells * by * case["steps"] + out, flops=cells * fl * case["steps"])
    if kind == "fv":
        n = case["nx"] * case["ny"] * case["nz"] * case["L"] ** 3
        return dict(bytes=n * 80 * case["steps"] + 40 * n, flops=n * (300 if case["muscl"] else 150) * case["steps"])
    if kind == "patches":
        by = fl = 0
        V, D = (9, 12) if case["elastic"] else (5, 5)
        for n, order in zip(map(int, case["sides"].split(",")), map(int, case["orders"].split(","))):
            b, f = step_work(order, V, D, 1 if case["elastic"] else (2 if case["bits"] == 32 else 3), case["elastic"])
            by += n ** 3 * (b * case["steps"] + 8 * D * (order + 1) ** 3)
            fl += n ** 3 * f * case["steps"]
        return dict(bytes=by, flops=fl)
    B, coarse = case["order"] + 1, case["nx"] * case["ny"] * case["nz"]
    fine = coarse * 27 ** case["delta"]
    block = 5 * B ** 3
    return dict(bytes=8 * block * (2 * fine + 3 * coarse) + 40 * fine, flops=2 * fine * 6 * B * block * case["delta"])


def tolerance(case):
    """Four times what the jobs were measured to be off `exact` (or more, where few were measured).
    float64: the order of the sums, 8e-12 at most (one cell's update, a difference of large terms).
    FP32-bulk: float rounding in the predictor and its stopping rule, 1e-7 to 6e-7, and single
    values near open boundaries, where inflow amplifies it, up to 6e-4.  Limiter: no `exact`;
    rounding must not change a cell's status."""
    if case["kind"] == "limiter":
        return dict(rel=1e-10, max=1e-7, differ=0.0)
    if case.get("bits") == 32:
        open_ = not case.get("periodic", True)
        return dict(rel=4e-6 if open_ else 2.4e-6, max=2.4e-3 if open_ else 1e-5)
    return dict(rel=4e-11, max=4e-10)


# ---------------------------------------------------------------------------
# The same in float64 torch
# ---------------------------------------------------------------------------
def gauss(B):
    x, w = np.polynomial.legendre.leggauss(B)
    return 0.5 * (x + 1.0), 0.5 * w


def lagrange(nodes, x):
    """phi_l(x) and phi_l'(x), rows l."""
    B = len(nodes)
    c = np.linalg.inv(np.vander(nodes, B, increasing=True))  # columns: coefficients of phi_l
    p = np.vander(np.atleast_1d(x), B, increasing=True)
    dp = np.zeros_like(p)
    dp[:, 1:] = p[:, :-1] * np.arange(1, B)
    return (p @ c).T, (dp @ c).T


class Tables:
    def __init__(self, order, device):
        B = order + 1
        x, w = gauss(B)
        phi1, d = lagrange(x, 1.0)[0][:, 0], lagrange(x, x)[1]  # d[l, n] = phi_l'(x_n)
        phi0 = lagrange(x, 0.0)[0][:, 0]
        kxi = d * w  # Kxi[l][n] = w_n phi_l'(x_n)
        t = lambda a: torch.tensor(np.asarray(a), dtype=torch.float64, device=device)  # noqa: E731
        self.B, self.x, self.w, self.FL, self.FR, self.kxi, self.D = B, t(x), t(w), t(phi0), t(phi1), t(kxi), t(d.T)
        self.iK1 = t(np.linalg.inv(np.outer(phi1, phi1) - kxi))
        self.w2 = self.w[:, None] * self.w
        self.w3 = self.w[:, None, None] * self.w2


def along(M, q, d):
    """out[.., l, ..] = sum_n M[l, n] q[.., n, ..] along direction d (0 = x) of [..., z, y, x, var]."""
    ax = q.dim() - 2 - d
    return torch.movedim(torch.tensordot(q, M, dims=([ax], [1])), -1, ax)


def face_values(c, q, d):
    """The values at a face normal to d: sum_l c[l] q(l)."""
    return torch.tensordot(q, c, dims=([q.dim() - 2 - d], [0]))


class Euler:
    V = D = 5

    @staticmethod
    def pressure(Q):
        return 0.4 * (Q[..., 4] - 0.5 * (Q[..., 1:4] ** 2).sum(-1) / Q[..., 0])

    @classmethod
    def flux(cls, Q, d):
        p = cls.pressure(Q)
        u = Q[..., 1 + d] / Q[..., 0]
        F = Q * u[..., None]
        F[..., 0] = Q[..., 1 + d]
        F[..., 1 + d] += p
        F[..., 4] += p * u
        return F

    @classmethod
    def speed(cls, Q, d):
        return (Q[..., 1 + d] / Q[..., 0]).abs() + torch.sqrt(1.4 * cls.pressure(Q) / Q[..., 0])


class Elastic:
    V, D = 9, 12
    #: per direction: (variable, variable of its gradient, coefficient)
    TERMS = (((0, 6, "l2m"), (1, 6, "lam"), (2, 6, "lam"), (3, 7, "mu"), (5, 8, "mu"), (6, 0, "irho"), (7, 3, "irho"),
              (8, 5, "irho")),
             ((0, 7, "lam"), (1, 7, "l2m"), (2, 7, "lam"), (3, 6, "mu"), (4, 8, "mu"), (6, 3, "irho"), (7, 1, "irho"),
              (8, 4, "irho")),
             ((0, 8, "lam"), (1, 8, "lam"), (2, 8, "l2m"), (4, 7, "mu"), (5, 6, "mu"), (6, 5, "irho"), (7, 4, "irho"),
              (8, 2, "irho")))

    @classmethod
    def product(cls, Q, g, d):
        """B_d(Q) g."""
        lam, mu, rho = Q[..., 9], Q[..., 10], Q[..., 11]
        c = dict(lam=lam, mu=mu, l2m=lam + 2 * mu, irho=1 / rho)
        out = torch.zeros_like(g)
        for m, n, k in cls.TERMS[d]:
            out[..., m] -= c[k] * g[..., n]
        return out

    @staticmethod
    def speed(Q, d):
        return torch.sqrt((Q[..., 9] + 2 * Q[..., 10]) / Q[..., 11])


def predict(T, pde, q, dx, dt):
    """Space-time predictor of [cells, z, y, x, var]: time-averaged state and fluxes (or source)."""
    B, V = T.B, pde.V
    par = q[..., V:]
    ncp = pde is Elastic
    qt = q[:, None, ..., :V].expand(-1, B, -1, -1, -1, -1).contiguous()
    live = torch.arange(len(q), device=q.device)
    qh = torch.empty_like(q)
    Fh = [torch.zeros_like(q[..., :V]) for _ in range(1 if ncp else 3)]
    for it in range(2 * B):
        full = torch.cat([qt, par[live][:, None].expand(-1, B, -1, -1, -1, -1)], -1) if ncp else qt
        if ncp:
            terms = [-sum(pde.product(full, along(T.D, qt, d) / dx[d], d) for d in range(3))]
            s = terms[0]
        else:
            terms = [pde.flux(full, d) for d in range(3)]
            s = -sum(along(T.D, terms[d], d) / dx[d] for d in range(3))
        rhs = T.FL.view(-1, 1, 1, 1, 1) * q[live][:, None, ..., :V] + dt * T.w.view(-1, 1, 1, 1, 1) * s
        new = torch.movedim(torch.tensordot(rhs, T.iK1, dims=([1], [1])), -1, 1)
        res = ((new - qt) ** 2).flatten(1).sum(1)
        done = (res < 1e-14) if it + 1 < 2 * B else torch.ones_like(res, dtype=torch.bool)
        at = live[done]
        qh[at] = torch.cat([torch.tensordot(new[done], T.w, dims=([1], [0])), par[at]], -1)
        for f, t in zip(Fh, terms):
            f[at] = torch.tensordot(t[done], T.w, dims=([1], [0]))
        live, qt = live[~done], new[~done]
        if not len(live):
            break
    return qh, Fh


def predict_linear(T, q, dx, dt):
    V, par = Elastic.V, q[..., Elastic.V:]
    qi, c = q[..., :V], 1.0
    qh, Fh = torch.zeros_like(qi), [torch.zeros_like(qi) for _ in range(3)]
    for i in range(T.B):
        P = [Elastic.product(q, along(T.D, qi, d) / dx[d], d) for d in range(3)]
        qh += c * qi
        for d in range(3):
            Fh[d] += c * P[d]
        qi = -(P[0] + P[1] + P[2])
        c *= dt / (i + 2)
    return torch.cat([qh, par], -1), Fh


def volume(T, Fh, dx, source, linear):
    if linear:
        return -T.w3[..., None] * (Fh[0] + Fh[1] + Fh[2])
    if source:
        return T.w3[..., None] * Fh[0]
    du = 0
    for d in range(3):
        k = [T.w[:, None, None], T.w[None, :, None], T.w[None, None, :]]
        k[2 - d] = torch.ones(1, 1, 1, dtype=torch.float64, device=T.w.device)
        du = du + along(T.kxi, Fh[d], d) * (k[0] * k[1] * k[2])[..., None] / dx[d]
    return du


def face_term(T, pde, QL, QR, FL, FR, d, linear):
    """What the face gives to its left and its right cell."""
    V = pde.V
    aL, aR = (torch.tensordot(Q, T.w2, dims=([-3, -2], [0, 1])) for Q in (QL, QR))
    smax = torch.maximum(pde.speed(aL, d), pde.speed(aR, d))[..., None, None, None]
    jump = (QR - QL)[..., :V]
    if linear:
        f = Elastic.product((0.5 * (aL + aR))[..., None, None, :].expand_as(QL), 0.5 * jump, d)
        return f - 0.5 * smax * jump, f + 0.5 * smax * jump
    F = -0.5 * smax * jump + (0.5 * (FL + FR) if FL is not None else 0)
    if pde is Elastic:
        n = Elastic.product(0.5 * (QL + QR), jump, d)
        return F + 0.5 * n, F - 0.5 * n
    return F, F


def correct(T, pde, n, q, du, qh, Fh, dx, dt, periodic, linear):
    nx, ny, nz = n
    V = pde.V
    du = du.clone()
    for d in range(3):
        ax = 2 - d  # grid axis of direction d in [nz, ny, nx, ...]
        sides = []
        for c in (T.FL, T.FR):
            Q = face_values(c, qh, d)
            F = face_values(c, Fh[d], d) if pde is Euler else None
            sides.append((Q.view(nz, ny, nx, *Q.shape[1:]), F.view(nz, ny, nx, *F.shape[1:]) if F is not None else None))
        (Q0, F0), (Q1, F1) = sides
        nxt = lambda a: torch.roll(a, -1, ax) if a is not None else None  # noqa: E731
        left, right = face_term(T, pde, Q1, nxt(Q0), F1, nxt(F0), d, linear)
        hi, lo = left, torch.roll(right, 1, ax)
        if not periodic:  # the outside state is the inside one: the inner flux, no fluctuation
            at = [slice(None)] * 3
            at[ax] = -1
            hi[tuple(at)] = F1[tuple(at)] if F1 is not None else 0.0
            at[ax] = 0
            lo = lo.clone()
            lo[tuple(at)] = F0[tuple(at)] if F0 is not None else 0.0
        shape = [1, 1, 1, 1, 1]
        shape[1 + ax] = -1
        hi, lo = (v.reshape(-1, *v.shape[3:]).unsqueeze(1 + ax) for v in (hi, lo))
        k = [T.w[:, None, None], T.w[None, :, None], T.w[None, None, :]]
        k[ax] = torch.ones(1, 1, 1, dtype=torch.float64, device=T.w.device)
        us = (k[0] * k[1] * k[2])[..., None] / dx[d]
        du -= (hi * T.FR.view(shape) + (lo if linear else -lo) * T.FL.view(shape)) * us
    q = q.clone()
    q[..., :V] += dt * du / T.w3[..., None]
    return q, du


def stable_dt(pde, order, q, dx):
    lam = sum(pde.speed(q, d) / dx[d] for d in range(3))
    return 0.9 * PNPM[order] / float(lam.max())


def aderdg(order, pde, n, q, steps, periodic=True, linear=False, fused=False):
    T = Tables(order, q.device)
    dx = [1.0 / v for v in n]

    def both(q, dt):
        if linear:
            qh, Fh = predict_linear(T, q, dx, dt)
        else:
            qh, Fh = predict(T, pde, q, dx, dt)
        return qh, Fh, volume(T, Fh, dx, pde is Elastic, linear)

    dt = dtp = stable_dt(pde, order, q, dx)
    qh, Fh, du = both(q, dt)
    for _ in range(steps):
        q, _ = correct(T, pde, n, q, du, qh, Fh, dx, dt, periodic, linear)
        s = stable_dt(pde, order, q, dx)
        if fused:
            again = dtp > s
            nxt = 0.9 * s if again else 0.5 * (dtp + 0.9 * s)
            dt = nxt if again else dtp
            qh, Fh, du = both(q, dt)
            dtp = nxt
        else:
            dt = s
            qh, Fh, du = both(q, dt)
    return q


def node_coordinates(order, n, device):
    x = torch.tensor(gauss(order + 1)[0], dtype=torch.float64, device=device)
    c = [(torch.arange(v, dtype=torch.float64, device=device)[:, None] + x) / v for v in n]  # [cell, node]
    X = c[0].view(1, 1, n[0], 1, 1, -1)
    Y = c[1].view(1, n[1], 1, 1, -1, 1)
    Z = c[2].view(n[2], 1, 1, -1, 1, 1)
    return torch.broadcast_tensors(X, Y, Z)


def euler_field(X, rho0, amp, k, vel, p, nmodes, mode_amp, seed):
    tp = 2 * math.pi
    rho = rho0 + amp * torch.sin(tp * (k[0] * X[0] + k[1] * X[1] + k[2] * X[2]))
    u = [torch.full_like(rho, v) for v in vel]
    state = seed
    for _ in range(nmodes):
        while True:
            kk = []
            for _ in range(3):
                state, z = splitmix64(state)
                kk.append(z % 7 - 3)
            if any(kk):
                break
        arg = tp * (kk[0] * X[0] + kk[1] * X[1] + kk[2] * X[2])
        ph = []
        for _ in range(4):
            state, z = splitmix64(state)
            ph.append(tp * (z >> 11) * 2.0 ** -53)
        rho = rho + mode_amp * torch.sin(arg + ph[0])
        for i in range(3):
            u[i] = u[i] + mode_amp * torch.sin(arg + ph[i + 1])
    E = p / 0.4 + 0.5 * rho * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    return torch.stack([rho, rho * u[0], rho * u[1], rho * u[2], E], -1)


def elastic_field(X, seed, width, amp):
    x, y, z = X
    r = [(splitmix64((seed + c * GOLDEN) & MASK)[1] >> 11) * 2.0 ** -53 for c in range(6)]
    tp = 2 * math.pi
    upper = z > 0.5 + 0.1 * torch.sin(tp * x + tp * r[0]) * torch.sin(tp * y + tp * r[1])
    pick = lambda a, b: torch.where(upper, torch.full_like(x, a), torch.full_like(x, b))  # noqa: E731
    rho = pick(2.05 + 0.9 * r[2], 2.05 + 0.9 * r[3]) + 0.05 * torch.sin(tp * (x + y + z))
    cp = pick(4.1 + 1.8 * r[4], 4.1 + 1.8 * r[5]) + 0.1 * torch.sin(tp * (x - y + z))
    mu = rho * cp * cp / 3.0
    g = amp * torch.exp(-((x - 0.5) ** 2 + (y - 0.5) ** 2 + (z - 0.5) ** 2) / (2 * width * width))
    o = torch.zeros_like(x)
    return torch.stack([o] * 6 + [g, g, g, rho * cp * cp - 2 * mu, mu, rho], -1)


def cells_first(q):
    return q.reshape(-1, *q.shape[3:])


def exact(case, seed):
    kind = case["kind"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "cell":
        return exact_cell(case, seed, dev)
    if kind == "grid":
        nodes = case["nx"] * case["ny"] * case["nz"] * (case["order"] + 1) ** 4 * case["steps"]
        if nodes > 2.5e9:  # would take over 20 seconds and much of the card
            return None
        X = node_coordinates(case["order"], dims(case), dev)
        elastic = case["pde"] == "elastic"
        q = cells_first(elastic_field(X, **elastic_ic(seed)) if elastic else euler_field(X, **euler_ic(seed)))
        q = aderdg(case["order"], Elastic if elastic else Euler, dims(case), q, case["steps"], case["periodic"],
                   case["linear"], case["fused"])
        out = [q.reshape(-1)]
        if case["plot"]:
            B = case["order"] + 1
            M = torch.tensor(lagrange(gauss(B)[0], np.linspace(0, 1, B))[0].T.copy(), dtype=torch.float64, device=dev)
            v = q
            for d in range(3):
                v = along(M, v, d)
            out.append(v.reshape(-1))
        return out
    if kind == "fv" and not case["muscl"]:
        return [exact_godunov(case, seed, dev)]
    if kind == "patches":
        out = []
        for spec in patch_specs(case, seed):
            if case["elastic"]:
                n, order = spec["n"], spec["order"]
                q = elastic_field(node_coordinates(order, (n,) * 3, dev), spec["seed"], spec["width"], spec["amp"])
            else:
                n, order = spec[0], spec[1]
                q = euler_field(node_coordinates(order, (n,) * 3, dev), 1.0, spec[3], spec[2], (1.0,) * 3, 1.0, 0, 0, 0)
            if n ** 3 * (order + 1) ** 4 * case["steps"] > 1.5e9:
                out.append(None)
                continue
            q = aderdg(order, Elastic if case["elastic"] else Euler, (n,) * 3, cells_first(q), case["steps"])
            out.append(q.reshape(-1))
        return out
    if kind == "amr":
        return exact_amr(case, seed, dev)
    # The limiting solver and the MUSCL-Hancock patches are state machines over
    # per-cell patches with never-filled edge ghosts: no plain restatement here.
    return None


def exact_cell(case, seed, dev):
    order = case["order"]
    luh, dx, dt = cell_state(case, seed)
    T = Tables(order, dev)
    B = order + 1
    q = torch.tensor(luh, dtype=torch.float64, device=dev).view(1, B, B, B, 5)
    qh, Fh = predict(T, Euler, q, dx, dt)
    faces = lambda f: torch.stack([face_values(c, f(d), d)[0] for d in range(3) for c in (T.FL, T.FR)])  # noqa: E731
    new, du = correct(T, Euler, (1, 1, 1), q, volume(T, Fh, dx, False, False), qh, Fh, dx, dt, True, False)
    return [faces(lambda d: qh).reshape(-1), faces(lambda d: Fh[d]).reshape(-1), du.reshape(-1), new.reshape(-1),
            np.array([stable_dt(Euler, order, new, dx)])]


def exact_godunov(case, seed, dev):
    n, L = dims(case), case["L"]
    N = [v * L for v in n]
    c = [(torch.arange(v, dtype=torch.float64, device=dev) + 0.5) / v for v in N]
    X = torch.broadcast_tensors(c[0].view(1, 1, -1), c[1].view(1, -1, 1), c[2].view(-1, 1, 1))
    u = euler_field(X, **euler_ic(seed))
    h = [1.0 / v for v in N]
    dt = None
    for _ in range(case["steps"]):
        if dt is None:
            dt = min(0.9 / 3 * h[d] / float(Euler.speed(u, d).max()) for d in range(3))
        new = u.clone()
        for d in range(3):
            ax = 2 - d
            r = torch.roll(u, -1, ax)
            if not case["periodic"]:
                at = [slice(None)] * 3
                at[ax] = -1
                r[tuple(at)] = u[tuple(at)]
            s = torch.maximum(Euler.speed(u, d), Euler.speed(r, d))[..., None]
            F = 0.5 * s * (u - r) + 0.5 * (Euler.flux(u, d) + Euler.flux(r, d))
            G = torch.roll(F, 1, ax)
            if not case["periodic"]:
                at[ax] = 0
                G[tuple(at)] = Euler.flux(u[tuple(at)], d)
            new -= dt / h[d] * (F - G)
        u = new
        dt = min(0.9 / 3 * h[d] / float(Euler.speed(u, d).max()) for d in range(3))
    u = u.view(n[2], L, n[1], L, n[0], L, 5).permute(0, 2, 4, 1, 3, 5, 6)
    return u.reshape(-1)


def exact_amr(case, seed, dev):
    a = amr_arrays(case, seed, dev)
    B = case["order"] + 1
    x, w = gauss(B)
    P = torch.tensor(np.stack([lagrange(x, (x + j) / 3.0)[0].T for j in range(3)]), dtype=torch.float64, device=dev)
    w = torch.tensor(w, dtype=torch.float64, device=dev)
    R = P.transpose(1, 2) * w / w[:, None] / 3.0  # R[j][m][n] = w_n P_j[n][m] / (3 w_m)
    coarse = a["coarse"].view(-1, B, B, B, 5)
    sub = a["items"][:, 2:].long()
    levels = range(case["delta"])
    up, down = [], []
    for d in range(3):
        u = v = torch.eye(B, dtype=torch.float64, device=dev).expand(len(sub), B, B)
        for l in levels:
            u = P[(sub[:, d] // 3 ** (case["delta"] - 1 - l)) % 3] @ u
            v = R[(sub[:, d] // 3 ** l) % 3] @ v
        up.append(u)
        down.append(v)

    def apply(M, q):
        for d in range(3):
            ax = 3 - d
            t = q.movedim(ax, 1)
            q = torch.matmul(M[d], t.reshape(len(t), B, -1)).view(t.shape).movedim(1, ax)
        return q

    fine = torch.empty(len(sub), B, B, B, 5, dtype=torch.float64, device=dev)
    rows = apply(up, coarse[a["items"][:, 1].long()])
    fine[a["items"][:, 0].long()] = rows
    acc = torch.zeros_like(coarse)
    acc.index_add_(0, a["items"][:, 1].long(), apply(down, rows))
    return [fine.reshape(len(sub), -1), acc.reshape(len(acc), -1)]

"""A user PDE compiled into the device kernels (include/exahype_amd/user_solver.hpp,
the example in exahype_amd/examples/user_euler.hip) and driven through
exa_grid_create_user: the reference's user-solver route (the generated
AbstractMySolver calling the generic kernels with the user's flux,
eigenvalues, boundaryValues and adjustPointSolution,
UserSolverInterface.h:64-171).

Bars: the user Euler against the built-in Euler on the same grid, <= 1e-12
relative per DOF after 5 steps (the same formulas in another instantiation);
reflecting walls (boundaryValues, boundaryConditions.cpph:24-85) and the
per-step adjustPointSolution (solutionAdjustment.cpph:17-47 after the update
at t + dt) against the oracle's grid with the same hooks, <= 1e-12 of each
variable's scale, the dt sequence to 1e-13; FP32-bulk against FP64 on the
user grid, relative L2 < 1e-6.
"""
import ctypes

import numpy as np
import pytest

from refutil import elastic_cells, rel_per_dof

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _table(exa, order):
    return getattr(exa.user_example(), f"exa_user_euler_order{order}")


def _user_grid(exa, order, n, boundary=0, precision=0):
    return exa.Grid.from_user_solver(_table(exa, order), n, precision=precision, boundary=boundary)


def _scaled_err(a, b):
    """max over variables of max|a-b| / max|b| (momenta cross zero at walls)."""
    a, b = a.reshape(-1, 5), b.reshape(-1, 5)
    return float((np.abs(a - b).max(axis=0) / np.abs(b).max(axis=0)).max())


def test_user_solver_table(exa):
    g = _user_grid(exa, 5, 2)
    assert (g.user.order, g.user.num_variables, g.user.num_parameters) == (5, 5, 0)
    assert g.user.has_boundary_values == 1 and g.user.has_adjust == 1
    assert g.user.cfl == 0.9
    g.close()


@pytest.mark.parametrize("order,n", [(3, 5), (5, 4)])
def test_user_euler_matches_builtin_periodic(exa, order, n):
    print(f"case: user Euler vs built-in, N={order} {n}^3 periodic", flush=True)
    u = _user_grid(exa, order, n)
    u.adjust_solution()  # adjustPointSolution at t = 0: the entropy wave
    b = exa.Grid(exa.euler_solver(order), n)
    b.init_euler()  # the same entropy wave from the built-in initialiser
    ic_err = rel_per_dof(u.solution(), b.solution())
    print(f"  IC rel per DOF {ic_err:.2e}", flush=True)
    assert ic_err < 1e-14
    b.init_euler(nmodes=8, mode_amp=0.05, seed=order)
    u.upload(b.solution())
    u.step(5)
    b.step(5)
    err = rel_per_dof(u.solution(), b.solution())
    du, db = u.dt_history(6), b.dt_history(6)
    print(f"  rel per DOF {err:.2e}", flush=True)
    assert err < TOL
    assert np.abs(du - db).max() <= 1e-13 * db.max()
    u.close()
    b.close()


def test_user_euler_matches_builtin_transmissive(exa):
    order, n = 5, 4  # the example compiles orders 3 and 5
    print(f"case: user Euler vs built-in, N={order} {n}^3 transmissive", flush=True)
    b = exa.Grid(exa.euler_solver(order), n, boundary=exa.BC_TRANSMISSIVE)
    b.init_euler(nmodes=8, mode_amp=0.05, seed=2)
    u = _user_grid(exa, order, n, boundary=exa.BC_TRANSMISSIVE)
    u.upload(b.solution())
    u.step(5)
    b.step(5)
    err = _scaled_err(u.solution(), b.solution())
    print(f"  scaled err {err:.2e}", flush=True)
    assert err < TOL
    u.close()
    b.close()


def _vs_oracle(exa, oracle, order, n, steps, wall, adjust):
    boundary = exa.BC_USER if wall else exa.BC_PERIODIC
    g = _user_grid(exa, order, n, boundary=boundary)
    g.adjust_solution()
    if adjust:
        g.set_adjust_solution(True)
    luh0 = g.solution()
    g.step(steps)
    gpu = g.solution()
    dts = g.dt_history(steps + 1)
    o = oracle.Grid(oracle.make_solver(order, 5, 0), n, transmissive=wall)
    o.set_user(wall, adjust)
    o.set_solution(luh0)
    odts, _ = o.step(steps)
    g.close()
    return gpu, o.solution(), dts[:steps], odts


@pytest.mark.parametrize("order,n,steps", [(3, 5, 6), (5, 4, 4)])
def test_reflecting_walls_vs_oracle(exa, oracle, order, n, steps):
    print(f"case: user boundaryValues (reflecting walls) N={order} {n}^3 {steps} steps", flush=True)
    gpu, cpu, dts, odts = _vs_oracle(exa, oracle, order, n, steps, wall=True, adjust=False)
    err = _scaled_err(gpu, cpu)
    print(f"  scaled err {err:.2e}", flush=True)
    assert err < TOL
    assert np.abs(dts - odts).max() <= 1e-13 * odts.max()


@pytest.mark.parametrize("order,n,steps", [(3, 5, 6), (5, 3, 4)])
def test_adjust_every_step_vs_oracle(exa, oracle, order, n, steps):
    print(f"case: user adjustPointSolution every step N={order} {n}^3 {steps} steps", flush=True)
    gpu, cpu, dts, odts = _vs_oracle(exa, oracle, order, n, steps, wall=False, adjust=True)
    err = _scaled_err(gpu, cpu)
    print(f"  scaled err {err:.2e}", flush=True)
    assert err < TOL
    assert np.abs(dts - odts).max() <= 1e-13 * odts.max()


def test_walls_and_adjust_vs_oracle(exa, oracle):
    order, n, steps = 3, 4, 5
    print(f"case: user walls + adjust N={order} {n}^3 {steps} steps", flush=True)
    gpu, cpu, dts, odts = _vs_oracle(exa, oracle, order, n, steps, wall=True, adjust=True)
    err = _scaled_err(gpu, cpu)
    print(f"  scaled err {err:.2e}", flush=True)
    assert err < TOL
    assert np.abs(dts - odts).max() <= 1e-13 * odts.max()


def test_fp32_bulk_user_grid(exa):
    order, n, steps = 5, 4, 4
    print(f"case: user grid FP32-bulk vs FP64 N={order} {n}^3 walls", flush=True)
    out = []
    for precision in (exa.PRECISION_FP64, exa.PRECISION_FP32_BULK):
        g = _user_grid(exa, order, n, boundary=exa.BC_USER, precision=precision)
        g.adjust_solution()
        g.step(steps)
        out.append(g.solution())
        g.close()
    l2 = np.linalg.norm(out[1] - out[0]) / np.linalg.norm(out[0])
    print(f"  L2 {l2:.2e}", flush=True)
    assert l2 < 1e-6


@pytest.mark.parametrize("name,order,n,steps,npar", [("order1_many", 1, 5, 6, 10), ("order2", 2, 4, 6, 3),
                                                     ("order4", 4, 3, 4, 3)])
def test_flux_free_user_pde_vs_oracle(exa, oracle, name, order, n, steps, npar):
    """Elasticity as a user's PDE (a non-conservative product and no flux):
    gradients from the iterate in place, or from a staged slice where the
    parameters outnumber the iterate's rows.  Bars of the library's elastic grid."""
    print(f"case: flux-free user PDE {name} {n}^3", flush=True)
    nodes = np.array([oracle.table(oracle.T_NODES, order, i) for i in range(order + 1)])
    luh = elastic_cells(order, n, seed=5, nodes=nodes, width=0.15).reshape(-1, 12)
    extra = np.random.default_rng(order).uniform(-1, 1, (len(luh), npar - 3))
    o = oracle.Grid(oracle.elastic_solver(order), n)
    o.set_solution(luh.ravel())
    odts, _ = o.step(steps)
    want = np.concatenate([o.solution().reshape(-1, 12), extra], 1)
    for precision, tol in ((exa.PRECISION_FP64, 1e-12), (exa.PRECISION_FP32_BULK, None)):
        g = exa.Grid.from_user_solver(getattr(exa.user_example(), f"exa_user_elastic_{name}"), n, precision=precision)
        g.upload(np.concatenate([luh, extra], 1).ravel())
        g.step(steps)
        got = g.solution().reshape(-1, 9 + npar)
        assert np.array_equal(got[:, 9:], want[:, 9:])
        if tol:
            assert np.abs(g.dt_history(steps) - odts).max() <= 1e-13 * odts.max()
            assert np.array_equal(g.picard_iterations(), o.picard_iterations())
            assert (np.abs(got - want).max(axis=0) <= tol * np.abs(want).max(axis=0)).all()
        else:
            assert np.linalg.norm(got[:, :9] - want[:, :9]) <= 1e-5 * np.linalg.norm(want[:, :9])
        g.close()


@pytest.mark.parametrize("order,other", [(3, "split_order3"), (4, "split_order4"), (5, "split_order5"),
                                         (4, "source_order4")])
@pytest.mark.parametrize("precision", [0, 1])
def test_user_flux_with_product_or_source(exa, order, other, precision):
    """Constant coefficients: half of a linear PDE as a flux and half as a
    non-conservative product, or the flux beside a zero source, compute what the
    flux alone does, but for rounding and the Picard iteration's end: face
    fluxes are of the iterate before the last, states of the last, and in double
    these differ by up to 1e-7 in the stopping norm.  States of size 1e6 put that
    at 1e-13 of their scale a step, beside which 5 steps stay below 1e-12;
    FP32-bulk, which stops at 1e-6 of the state's norm: 1e-6 relative L2.  These
    forms run their time slices in rolled loops of their own."""
    # (bound for iterations that end by the residual, as all do at the PDE's CFL
    # number of 0.05; at 0.9 the limit of 2 (N + 1) iterations left 2e-11 of the scale)
    print(f"case: user PDE waves {other} precision {precision}", flush=True)
    n, D = (4, 3, 5), 5
    cells = n[0] * n[1] * n[2]
    luh = 1e6 * np.random.default_rng(order).uniform(-1, 1, (cells, (order + 1) ** 3, D))
    out, its = [], []
    for name in (f"order{order}", other):
        g = exa.Grid.from_user_solver(getattr(exa.user_example(), f"exa_user_waves_{name}"), n, precision=precision)
        g.upload(luh.ravel())
        g.step(5)
        out.append(g.solution().reshape(-1, D))
        its.append(g.picard_iterations())
        g.close()
    assert max(its[0].max(), its[1].max()) < 2 * (order + 1)
    a, b = out
    if precision == 0:
        assert np.array_equal(*its)
        assert (np.abs(b - a).max(axis=0) <= TOL * np.abs(a).max(axis=0)).all()
    else:
        assert np.linalg.norm(b - a) <= 1e-6 * np.linalg.norm(a)


def test_user_route_refusals(exa):
    L = exa.lib()
    b = exa.Grid(exa.euler_solver(3), 2)
    # the library's Euler has no boundaryValues / adjustPointSolution
    assert L.exa_grid_set_adjust_solution(b._h, 1) == exa.EXA_E_UNSUPPORTED
    assert L.exa_grid_adjust_solution(b._h) == exa.EXA_E_UNSUPPORTED
    b.close()
    h = ctypes.c_void_p()
    lo = (ctypes.c_double * 3)(0, 0, 0)
    hi = (ctypes.c_double * 3)(1, 1, 1)
    assert L.exa_grid_create(ctypes.byref(exa.euler_solver(3)), 2, 2, 2, lo, hi, exa.BC_USER,
                             ctypes.byref(h)) == exa.EXA_E_UNSUPPORTED
    u = _user_grid(exa, 3, 2, boundary=exa.BC_USER)
    # user grids run the one-kernel corrector only
    assert L.exa_grid_set_fused_corrector(u._h, 0) == exa.EXA_E_UNSUPPORTED
    assert L.exa_grid_set_adjust_solution(u._h, 1) == exa.EXA_OK
    u.close()

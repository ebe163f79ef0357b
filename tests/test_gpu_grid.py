"""The kernels whose workgroups exchange data without leaving the kernel (fvm_grid.hpp),
at the sizes where their layout changes: one workgroup, whole and ragged last
workgroups, rows wider than the unrolled widths.

fvm_trbdf2_affine against the host integrator on the same problem, both with Newton
stopped at 1e-7 and GMRES at 1e-9 of their scales: the two then take the same steps and
differ by the Newton tolerance times the error norm's scale (abstol + reltol |u|, 1e-3
|u| here) per solve, two solves a step: at most 2e-10 |u| per step, 1e-8 |u| over the
fifty steps allowed here, and 1e-7 with the step controller's own amplification."""
import contextlib
import ctypes

import numpy as np
import pytest

import finitevolumemethod as FVM
from test_gpu_templates import wheel_triangulation

pytestmark = pytest.mark.gpu


def _problem(tri, steps=0.05):
    mesh = FVM.FVMGeometry(tri)
    segs = tri.num_boundary_segments()
    fns = tuple((lambda x, y, t, u, p, k=k: 0.3 * k + 0.0 * u) for k in range(segs))
    types = tuple(FVM.Dirichlet if k % 2 else FVM.Neumann for k in range(segs))
    u0 = 1.0 + np.sin(2 * tri.x) * np.cos(3 * tri.y)
    return FVM.FVMProblem(mesh, FVM.BoundaryConditions(mesh, fns, types),
                          diffusion_function=lambda x, y, t, u, p: 0.2 + 0.1 * x * y,
                          source_function=lambda x, y, t, u, p: x - 0.5 * u, initial_condition=u0, final_time=steps)


@pytest.mark.parametrize("shape", [(3, 3), (16, 16), (257, 1), (23, 41), (128, 128), (131, 127), "wheel"], ids=str)
def test_affine_trbdf2_matches_the_host_integrator(gpu, shape):
    if shape == "wheel":
        tri = wheel_triangulation()
    elif shape[1] == 1:  # 257 nodes: one row in the second workgroup
        g = FVM.triangulate_rectangle(0.0, 1.0, 0.0, 1.0, 16, 16, single_boundary=True)
        tri = FVM.triangulate(np.append(g.x, 1.5), np.append(g.y, 0.4))
    else:
        tri = FVM.triangulate_rectangle(0.0, 1.0, 0.0, 1.0, *shape, single_boundary=False)
    prob = _problem(tri)
    opts = dict(newton_kappa=1e-7, krylov_rtol=1e-9)
    a = FVM.solve(prob, FVM.TRBDF2(**opts), saveat=[0.02, 0.05])
    b = FVM.solve(prob, FVM.TRBDF2(device_loop=False, **opts), saveat=[0.02, 0.05])
    assert a.stats.get("device_loop") and a.retcode == b.retcode == "Success"
    assert a.stats["naccept"] == b.stats["naccept"] <= 50, (a.stats, b.stats)
    for x, y in zip(a.u, b.u):
        assert np.max(np.abs(x - y)) <= 1e-7 * np.max(np.abs(y))
    again = FVM.solve(prob, FVM.TRBDF2(**opts), saveat=[0.02, 0.05])
    assert all(np.array_equal(x, y) for x, y in zip(a.u, again.u))  # sums in a fixed order


@pytest.mark.parametrize("shape", [(5, 4), (16, 16), (61, 47), (131, 127), "wheel"], ids=str)
def test_nonlinear_trbdf2_with_a_frozen_jacobian_matches_the_matrix_free_loop(gpu, shape, monkeypatch):
    """The same loop with each linear system solved in one launch on the extracted J
    (fvm_jacobian_ell, fvm_gmres_ell) or matrix-free: a hub's wide rows keep the latter.
    Tolerances as above."""
    from finitevolumemethod import implicit

    wheel = shape == "wheel"
    tri = wheel_triangulation() if wheel else FVM.jittered_rectangle(0.0, 1.0, 0.0, 1.0, *shape, jitter=0.2, seed=3)
    mesh = FVM.FVMGeometry(tri)
    u0 = 0.5 + 0.4 * np.sin(5 * tri.x) * np.cos(4 * tri.y)
    prob = FVM.FVMProblem(mesh, FVM.BoundaryConditions(mesh, lambda x, y, t, u, p: 0.2 * t + 0.0 * u, FVM.Neumann),
                          diffusion_function=lambda x, y, t, u, p: 0.1 + u ** 2,
                          source_function=lambda x, y, t, u, p: u * (1 - u), initial_condition=u0, final_time=0.02)
    assert (implicit.FrozenJacobian.of(prob) is None) == wheel
    opts = dict(newton_kappa=1e-7, krylov_rtol=1e-9)
    colours, take = [], implicit.FrozenJacobian.take
    monkeypatch.setattr(implicit.FrozenJacobian, "take", lambda J, u, t: (colours.append(J.n_colours), take(J, u, t)))
    a = FVM.solve(prob, FVM.TRBDF2(**opts), saveat=[0.01, 0.02])
    if not wheel:  # the products made: those that J is extracted from, once per step's start
        assert a.stats["njvp"] == sum(colours) > 0 and len(colours) == a.stats["naccept"], (a.stats, colours)
    b = FVM.solve(prob, FVM.TRBDF2(device_loop=False, **opts), saveat=[0.01, 0.02])
    assert a.retcode == b.retcode == "Success"
    assert a.stats["naccept"] == b.stats["naccept"] <= 50 and a.stats["nnewton"] > 0, (a.stats, b.stats)
    for x, y in zip(a.u, b.u):
        assert np.max(np.abs(x - y)) <= 1e-7 * np.max(np.abs(y))


@pytest.mark.parametrize("case", ["outside", "callback", "dirichlet"])
def test_frozen_jacobian_over_free_points_and_callbacks(gpu, case):
    """Points that are no vertices (rows of the diagonal alone), a user callback that changes u
    after every step, Dirichlet values that depend on t: J is taken where the step starts."""
    from finitevolumemethod import implicit

    base = FVM.jittered_rectangle(0.0, 1.0, 0.0, 1.0, 23, 19, jitter=0.2, seed=3, single_boundary=False)
    x, y, tri = base.x, base.y, base
    if case == "outside":
        new = np.random.default_rng(8).permutation(len(x) + 3)
        x, y = np.full(len(new), 0.5), np.full(len(new), 0.5)
        x[new[:-3]], y[new[:-3]] = base.x, base.y
        tri = FVM.Triangulation(x, y, new[base.triangles], new[base.boundary_edges], base.boundary_segments)
    mesh = FVM.FVMGeometry(tri)
    hold = FVM.Dirichlet if case == "dirichlet" else FVM.Neumann
    prob = FVM.FVMProblem(mesh, FVM.BoundaryConditions(mesh, (lambda x, y, t, u, p: 0.5 + 0.3 * t + 0.0 * u,) * 4,
                                                       (hold, FVM.Neumann) * 2),
                          diffusion_function=lambda x, y, t, u, p: 0.1 + u ** 2,
                          source_function=lambda x, y, t, u, p: u * (1 - u),
                          initial_condition=0.5 + 0.4 * np.sin(5 * x) * np.cos(4 * y), final_time=0.02)
    J = implicit.FrozenJacobian.of(prob)
    assert J is not None and (J.op.width > 0)
    calls = []

    def callback(u, t):
        calls.append(t)
        u.upload(0.97 * u.to_host())

    kw = dict(saveat=[0.01, 0.02], callback=callback if case == "callback" else None)
    opts = dict(newton_kappa=1e-7, krylov_rtol=1e-9)
    a = FVM.solve(prob, FVM.TRBDF2(**opts), **kw)
    seen, calls[:] = list(calls), []
    b = FVM.solve(prob, FVM.TRBDF2(device_loop=False, **opts), **kw)
    assert a.retcode == b.retcode == "Success" and a.stats["naccept"] == b.stats["naccept"] <= 50
    # times of steps agree to the controller's amplification of the states' differences
    assert len(seen) == len(calls) == (a.stats["naccept"] if case == "callback" else 0)
    np.testing.assert_allclose(seen, calls, rtol=1e-5)
    for p, q in zip(a.u, b.u):
        assert np.max(np.abs(p - q)) <= 1e-7 * np.max(np.abs(q))


def _frozen(nx, ny):
    from finitevolumemethod import implicit

    tri = FVM.jittered_rectangle(0.0, 1.0, 0.0, 1.0, nx, ny, jitter=0.2, seed=3)
    mesh = FVM.FVMGeometry(tri)
    u0 = 0.5 + 0.4 * np.sin(5 * tri.x) * np.cos(4 * tri.y)
    prob = FVM.FVMProblem(mesh, FVM.BoundaryConditions(mesh, lambda x, y, t, u, p: 0.0 * u, FVM.Neumann),
                          diffusion_function=lambda x, y, t, u, p: 0.1 + u ** 2, initial_condition=u0, final_time=0.01)
    return prob, implicit.FrozenJacobian.of(prob)


@pytest.mark.parametrize("shape", [(5, 4), (61, 47)], ids=str)  # one workgroup, several
def test_a_failed_gmres_leaves_no_stale_solution(gpu, shape):
    """The work memory's fault word, set here by the host, as a timed-out exchange leaves it:
    the solves on that memory give NaN, not what x held, and the count of iterations raises."""
    from finitevolumemethod import _lib

    prob, J = _frozen(*shape)
    n = J.n
    u = FVM.DeviceArray.from_host(prob.initial_condition)
    J.take(u, 0.0)
    b, x = FVM.DeviceArray.from_host(np.random.default_rng(0).random(n)), FVM.DeviceArray.from_host(np.full(n, 3.0))
    J.solve(1.0, -1e-4, b, x, 1e-3, 20, 400, True)
    assert np.all(np.isfinite(x.to_host())) and J.iterations() > 0
    w = J.work.to_host()
    w.view(np.uint64)[2] = 1  # kGridFault
    J.work.upload(w)
    for _ in range(2):
        x.upload(np.full(n, 3.0))
        J.solve(1.0, -1e-4, b, x, 1e-3, 20, 400, True)
        assert np.all(np.isnan(x.to_host()))
    with pytest.raises(_lib.FVMError, match="timed out"):
        J.iterations()


@pytest.mark.parametrize("sides", ["neumann", "dirichlet"])
@pytest.mark.parametrize("shape", [(3, 3), (16, 16), (32, 32), (64, 40), (13, 197), (45, 46, 0.25), (64, 32, 0.25),
                                   (90, 80, 0.25), (256, 256), (200, 190, "permuted"), "wheel", ("hub", 11, 3),
                                   ("hub", 18, 40), ("hub", 19, 140), ("hub", 300, 2), ("hub", 300, 12)], ids=str)
def test_one_launch_tsit5_is_the_host_loop_bit_for_bit(gpu, shape, sides):
    """A small ODE template's whole Tsit5 loop in one launch: one workgroup up to the rows
    its registers hold (2,560 with up to 6 off-diagonals a row, 2,048 with more), a resident
    grid up to 65,536, 16- and 32-bit columns, a hub's row of 11 to 300 (one, eight, nine and
    many entries beyond the ten slots) in either: every saved state, time and counter equals
    the multi-kernel arithmetic of the host loop.  Dirichlet rows have no flux but keep their
    neighbours as entries of zero: the grid form needs a symmetric pattern, or waves of such
    rows alone (a side of a large rectangle) could run ahead of the others' reads."""
    from finitevolumemethod.solve import integrate
    from test_gpu_amg import _hub
    from test_gpu_templates import _permuted

    if shape == "wheel":
        tri = wheel_triangulation()
    elif shape[0] == "hub":
        tri = _hub(*shape[1:])
    elif len(shape) == 2:
        tri = FVM.triangulate_rectangle(0.0, 1.0, 0.0, 1.0, *shape, single_boundary=True)
    else:
        tri = FVM.jittered_rectangle(0.0, 1.0, 0.0, 1.0, *shape[:2], jitter=0.25, seed=5)
        if shape[2] == "permuted":
            tri = _permuted(tri, 2)
    mesh = FVM.FVMGeometry(tri)
    n = tri.num_points()
    u0 = np.random.default_rng(n).random(n)
    bc = FVM.Neumann if sides == "neumann" else FVM.Dirichlet
    prob = FVM.DiffusionEquation(mesh, FVM.BoundaryConditions(mesh, lambda x, y, t, u, p: 1.5, bc),
                                 diffusion_function=lambda x, y, p: 0.5 + x, initial_condition=u0,
                                 final_time=25.0 / n)
    if sides == "dirichlet":  # the property itself, of the assembled operator
        A = prob.A.copy()
        A.data[:] = 1.0
        assert np.all(np.diff(A.indptr) > 1) and (A != A.T).nnz == 0
    ts = [0.0, 7.0 / n, 25.0 / n]
    a = FVM.solve(prob, FVM.Tsit5(), saveat=ts)
    p = prob.problem
    if shape[-1] == "permuted":
        assert p.ell_info(index_bytes=True)[2] == 4
    b = integrate(lambda u, du, t: p.apply(u, du), prob._u0[:n], 0.0, 25.0 / n, FVM.Tsit5(), saveat=ts, fsal=True)
    assert a.retcode == b.retcode == "Success" and a.stats == b.stats and a.stats["naccept"] > 3, (a.stats, b.stats)
    for x, y in zip(a.u, b.u):
        assert np.array_equal(x[:-1], y)


@contextlib.contextmanager
def _resident(wgs):
    from finitevolumemethod import _lib

    f = _lib.hip_lib().fvm_test_resident_limit
    f.argtypes, f.restype = [ctypes.c_int64], None
    f(wgs)
    try:
        yield
    finally:
        f(0)


def test_a_device_that_does_not_hold_the_grid_keeps_the_other_loops(gpu):
    """Fewer resident workgroups than a launch needs (as where fewer CUs are visible; a limit
    of the library's own here): Tsit5 runs the multi-kernel loop to the same bits, TR-BDF2 the
    host integrator, and the C entry points return FVM_ERR_STATE with nothing done."""
    from finitevolumemethod import _lib, implicit

    prob, J = _frozen(61, 47)  # 12 workgroups
    n = J.n
    u = FVM.DeviceArray.from_host(prob.initial_condition)
    J.take(u, 0.0)
    b, x = FVM.DeviceArray.from_host(np.ones(n)), FVM.DeviceArray.from_host(np.full(n, 3.0))
    tri = FVM.triangulate_rectangle(0.0, 1.0, 0.0, 1.0, 67, 61, single_boundary=True)
    mesh = FVM.FVMGeometry(tri)
    u0 = np.random.default_rng(2).random(tri.num_points())
    ode = FVM.DiffusionEquation(mesh, FVM.BoundaryConditions(mesh, lambda x, y, t, u, p: 0.0 * x, FVM.Neumann),
                                diffusion_function=lambda x, y, p: 0.5 + x, initial_condition=u0, final_time=0.005)
    affine = _problem(FVM.triangulate_rectangle(0.0, 1.0, 0.0, 1.0, 61, 47, single_boundary=False))
    opts, ts = dict(newton_kappa=1e-7, krylov_rtol=1e-9), [0.005, 0.01]
    cases = [lambda: FVM.solve(ode, FVM.Tsit5(), saveat=[0.0025, 0.005]), lambda: FVM.solve(prob, FVM.Tsit5(), saveat=ts, dt=1e-6),
             lambda: FVM.solve(prob, FVM.TRBDF2(**opts), saveat=ts), lambda: FVM.solve(affine, FVM.TRBDF2(**opts), saveat=ts)]
    whole = [c() for c in cases]
    assert whole[3].stats.get("device_loop") and implicit.resident(n)
    A, o, st = implicit.affine_operator(affine).op(), implicit.TrbOpts(), implicit.TrbStats()
    o.tf, o.dt, o.abstol, o.reltol, o.maxiters = 0.05, 1e-3, 1e-6, 1e-3, 1000
    o.newton_kappa, o.max_newton, o.krylov_restart, o.krylov_rtol = 1e-2, 10, 20, 1e-3
    L = _lib.hip_lib()
    with _resident(11):
        assert not implicit.resident(n) and implicit.resident(11 * 256) and implicit.FrozenJacobian.of(prob) is None
        with pytest.raises(_lib.FVMError, match="at once"):
            J.solve(1.0, -1e-4, b, x, 1e-3, 20, 400, True)
        assert L.fvm_trbdf2_affine(ctypes.byref(A), ctypes.byref(o), x.ptr, ctypes.byref(st), None) == -4
        assert np.all(x.to_host() == 3.0)
        part = [c() for c in cases]
    assert "device_loop" not in part[3].stats
    for k, (w, p) in enumerate(zip(whole, part)):
        assert w.retcode == p.retcode == "Success" and w.stats["naccept"] == p.stats["naccept"]
        assert k < 2 or w.stats["naccept"] <= 50
        for a, b in zip(w.u, p.u):
            assert np.array_equal(a, b) if k < 2 else np.max(np.abs(a - b)) <= 1e-7 * np.max(np.abs(b)), k

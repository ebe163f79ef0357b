"""TR-BDF2 for small problems whose right-hand side is affine in u, in one launch.

When the traced closures make fvm_eqs! affine in u and constant in t (a diffusion
coefficient that does not depend on u, a source s(x, y) + s1 u, conditions with
values constant in t and Dirichlet values independent of u), f(u) = J u + c with a
constant J.  The reference hands such problems to TRBDF2 with a KLU factorisation of
J on its jacobian_sparsity pattern (solve.jl:50-77, 167-183).  Here J is extracted
once per problem from fvm_jvp probes over a distance-2 colouring of that pattern (one
probe per colour, about a dozen on a triangle mesh; exact for an affine f), stored in
ELL form, and fvm_trbdf2_affine integrates the whole problem in one launch of resident
workgroups (no host round trip per Krylov iteration).  Problems above 65,536 unknowns (or
what the visible part of the chip holds at once), with a user callback, without save times
or outside the affine forms keep the host-driven integrator (solve.py).
"""
import ctypes

import numpy as np

from . import _lib
from .equations import csr_pattern

MAX_N = 65536


class AffineOp(ctypes.Structure):
    _fields_ = [("n", ctypes.c_int64), ("width", ctypes.c_int32), ("d_col", _lib._vp), ("d_val", _lib._vp),
                ("d_diag", _lib._vp), ("d_ovf_rp", _lib._vp), ("d_ovf_col", _lib._vp), ("d_ovf_val", _lib._vp),
                ("d_c", _lib._vp), ("n_dirichlet", ctypes.c_int32), ("d_dir_nodes", _lib._vp),
                ("d_dir_values", _lib._vp)]


class TrbOpts(ctypes.Structure):
    _fields_ = [("t0", ctypes.c_double), ("tf", ctypes.c_double), ("dt", ctypes.c_double),
                ("abstol", ctypes.c_double), ("reltol", ctypes.c_double), ("maxiters", ctypes.c_int64),
                ("newton_kappa", ctypes.c_double), ("max_newton", ctypes.c_int32),
                ("krylov_restart", ctypes.c_int32), ("krylov_rtol", ctypes.c_double),
                ("smooth_est", ctypes.c_int32), ("n_save", ctypes.c_int64), ("save_t", _lib._dp),
                ("d_saves", _lib._vp)]


class TrbStats(ctypes.Structure):
    _fields_ = [("nf", ctypes.c_int64), ("njvp", ctypes.c_int64), ("naccept", ctypes.c_int64),
                ("nreject", ctypes.c_int64), ("nnewton", ctypes.c_int64), ("nkrylov", ctypes.c_int64),
                ("nnewton_fail", ctypes.c_int64), ("nsaved", ctypes.c_int64), ("retcode", ctypes.c_int32),
                ("reserved", ctypes.c_int32), ("t", ctypes.c_double)]


_RETCODES = {0: "Success", 1: "MaxIters", 2: "Unstable", 3: "ConvergenceFailure"}


def is_affine(prob):
    """Whether the problem's traced right-hand side is affine in u and constant in t."""
    from .problem import FVMProblem

    if not isinstance(prob, FVMProblem):
        return False
    ph = prob.device_context().physics
    fk = ph["flux_kind"]
    if fk == _lib.FLUX_D_POLY_U:
        if any(ph.get("dpoly", [0.0] * 4)[1:]):
            return False
    elif fk not in (_lib.FLUX_D_NODAL, _lib.FLUX_D_EDGE, _lib.FLUX_LINEAR):
        return False
    sp = ph.get("spoly", [0.0] * 4)
    if sp[2] != 0.0 or sp[3] != 0.0 or ph.get("st", 0.0) != 0.0:
        return False
    fn = ph["fn"]
    ct, lam = np.asarray(fn[2]), (np.asarray(fn[5]) if len(fn) > 5 else np.zeros(1))
    if np.any(ct != 0.0) or np.any(lam != 0.0):
        return False
    kind, fidx = ph["node_kind"], ph["node_fidx"]
    used = np.unique(fidx[kind == _lib.NODE_DIRICHLET])
    return not np.any(np.asarray(fn[1])[used] != 0.0)


def _colouring(rp, col, n):
    """Greedy distance-2 colouring of a symmetric pattern: columns that share a row
    get different colours (fvmh_colour_d2 in the host library)."""
    rp = np.ascontiguousarray(rp, np.int64)
    col = np.ascontiguousarray(col, np.int32)
    colour = np.empty(n, np.int32)
    nc = _lib.host_lib().fvmh_colour_d2(n, _lib.ptr(rp, _lib._i64p), _lib.ptr(col, _lib._i32p),
                                        _lib.ptr(colour, _lib._i32p))
    if nc < 0:
        raise ValueError(_lib.host_lib().fvmh_last_error().decode())
    return colour.astype(np.int64)


class _EllSlots:
    """Where the entries of a CSR pattern that holds every diagonal lie in ELL form: the
    off-diagonals of each row in CSR order, slot-major [W][n], the diagonal apart."""

    def __init__(self, rp, col, n):
        self.n, self.col = n, col
        self.off = col != np.repeat(np.arange(n, dtype=col.dtype), np.diff(rp))
        deg = np.diff(rp) - 1
        if len(col) - np.count_nonzero(self.off) != n or not np.array_equal(col[~self.off], np.arange(n)):
            raise ValueError("the pattern must hold every diagonal entry")
        self.W = int(deg.max()) if n else 0
        # entry k of the off-diagonals: slot k - (those of the rows before), at [slot n + row]
        first = rp[:-1] - np.arange(n)
        self.at = np.arange(len(col) - n) * n + np.repeat(np.arange(n) - first * n, deg)

    def diagonal(self, v):
        return v[~self.off]

    def columns(self):
        """The columns, padded with the row's own."""
        e = np.tile(np.arange(self.n, dtype=np.int32), self.W)
        e[self.at] = self.col[self.off]
        return e

    def spread(self, v, pad):
        v = np.asarray(v)
        e = np.full(self.W * self.n, pad, v.dtype)
        e[self.at] = v[self.off]
        return e


class AffineOperator:
    """J (ELL form on the device), c = f(0) and the Dirichlet values of an affine
    problem, built once."""

    def __init__(self, prob):
        ctx = prob.device_context()
        tri = prob.mesh.triangulation
        n = tri.num_points()
        t0 = prob.initial_time
        rp, col = csr_pattern(tri)
        rp = rp.astype(np.int64)
        colour = _colouring(rp, col, n)
        rows = np.repeat(np.arange(n), np.diff(rp))
        val = np.zeros(len(col))
        zero = _lib.DeviceArray(n)
        zero.fill_zero()
        jv = _lib.DeviceArray(n)
        for c in range(int(colour.max()) + 1):
            ctx.jvp(zero, _lib.DeviceArray.from_host((colour == c).astype(np.float64)), jv, t0)
            Jv = jv.to_host()
            sel = colour[col] == c
            val[sel] = Jv[rows[sel]]
        self.n_colours = int(colour.max()) + 1
        f0 = _lib.DeviceArray(n)
        ctx.rhs(zero, f0, t0)
        slots = _EllSlots(rp, col, n)
        diag, ecol, eval_ = slots.diagonal(val), slots.columns(), slots.spread(val, 0.0)
        self.W = slots.W
        self.d_col = _lib.DeviceArray.from_host(ecol, np.int32)
        self.d_val = _lib.DeviceArray.from_host(eval_)
        self.d_diag = _lib.DeviceArray.from_host(diag)
        self.d_orp = _lib.DeviceArray.from_host(np.zeros(n + 1, np.int32), np.int32)
        self.d_c = f0
        kind = ctx.physics["node_kind"]
        dn = np.nonzero(kind == _lib.NODE_DIRICHLET)[0].astype(np.int32)
        probe = _lib.DeviceArray(n)
        probe.fill_zero()
        ctx.apply_dirichlet(probe, t0)  # the Dirichlet values (constant in t and u)
        self.dir_nodes = dn
        self.d_dir_nodes = _lib.DeviceArray.from_host(dn if len(dn) else np.zeros(1, np.int32), np.int32)
        self.d_dir_values = _lib.DeviceArray.from_host(probe.to_host()[dn] if len(dn) else np.zeros(1))
        self.n = n
        self.csr = (rp, col, val)

    def op(self):
        o = AffineOp()
        o.n, o.width = self.n, self.W
        o.d_col, o.d_val, o.d_diag = self.d_col.ptr, self.d_val.ptr, self.d_diag.ptr
        o.d_ovf_rp, o.d_ovf_col, o.d_ovf_val = self.d_orp.ptr, None, None
        o.d_c = self.d_c.ptr
        o.n_dirichlet = len(self.dir_nodes)
        o.d_dir_nodes, o.d_dir_values = self.d_dir_nodes.ptr, self.d_dir_values.ptr
        return o


class FrozenJacobian:
    """J(u, t) of an FVMProblem in ELL form, taken again at each step's start, and GMRES
    on a I + b J in one launch (fvm_jacobian_ell, fvm_gmres_ell): the Newton steps of the
    host TR-BDF2 loop for problems of at most MAX_N unknowns.  The pattern's colouring and
    slots are kept on the problem."""

    MAX_COLOURS, MAX_WIDTH = 64, 32  # a hub node of a fan: matrix-free (jacobian_diagonal) instead

    @classmethod
    def of(cls, prob):
        """A FrozenJacobian for prob, or None where the pattern is not one for it."""
        from .problem import FVMProblem

        if not isinstance(prob, FVMProblem) or not resident(prob.mesh.triangulation.num_points()):
            return None
        plan = getattr(prob, "_jacobian_plan", None)
        if plan is None:
            n = prob.mesh.triangulation.num_points()
            rp, col = csr_pattern(prob.mesh.triangulation)
            colour = _colouring(rp, col, n)
            slots = _EllSlots(rp, col, n)
            nc = int(colour.max()) + 1
            plan = prob._jacobian_plan = (nc, slots.W, None) if nc > cls.MAX_COLOURS or slots.W > cls.MAX_WIDTH else (
                nc, slots.W, [_lib.DeviceArray.from_host((colour == c).astype(np.float64)) for c in range(nc)],
                _lib.DeviceArray.from_host(np.concatenate([slots.spread(colour.astype(np.uint8)[col], 255),
                                                           colour.astype(np.uint8)]), np.uint8),
                _lib.DeviceArray.from_host(slots.columns(), np.int32),
                _lib.DeviceArray.from_host(np.zeros(n + 1, np.int32), np.int32))
        return cls(prob, plan) if plan[2] is not None else None

    def __init__(self, prob, plan):
        self.ctx = prob.device_context()
        self.n = n = prob.mesh.triangulation.num_points()
        self.n_colours, self.W, self.probes, self.d_colour, self.d_col, self.d_orp = plan
        self.probe_ptrs = (_lib._vp * self.n_colours)(*[p.ptr for p in self.probes])
        self.products = _lib.DeviceArray(self.n_colours * n)
        self.d_val, self.d_diag = _lib.DeviceArray(self.W * n), _lib.DeviceArray(n)
        self.work = _lib.DeviceArray.zeros(_lib.hip_lib().fvm_gmres_work_bytes(n) // 8)
        o = self.op = AffineOp()
        o.n, o.width = n, self.W
        o.d_col, o.d_val, o.d_diag, o.d_ovf_rp = self.d_col.ptr, self.d_val.ptr, self.d_diag.ptr, self.d_orp.ptr

    def take(self, u, t):
        """J at (u, t)."""
        _lib.check(_lib.hip_lib().fvm_jacobian_ell(self.ctx.handle, self.n_colours, self.probe_ptrs, self.d_colour.ptr,
                                                   self.W, u.ptr, float(t), self.products.ptr, self.d_val.ptr,
                                                   self.d_diag.ptr, None), "fvm_jacobian_ell")

    def solve(self, a, b, rhs, x, rtol, restart, maxiter, jacobi):
        """x = (a I + b J)^-1 rhs; does not wait for it."""
        _lib.check(_lib.hip_lib().fvm_gmres_ell(ctypes.byref(self.op), float(a), float(b), int(jacobi), rhs.ptr, x.ptr,
                                                float(rtol), int(restart), int(maxiter), self.work.ptr, None),
                   "fvm_gmres_ell")

    def iterations(self):
        k = ctypes.c_int64()
        _lib.check(_lib.hip_lib().fvm_gmres_iterations(self.work.ptr, ctypes.byref(k), None), "fvm_gmres_ell")
        return k.value


def affine_operator(prob):
    op = getattr(prob, "_affine_op", None)
    if op is None:
        op = AffineOperator(prob)
        prob._affine_op = op
    return op


def resident(n):
    """Whether the device holds the one-launch solvers' workgroups for n unknowns at once
    (65,536 on a whole MI355X; fewer where fewer CUs are visible)."""
    fits = ctypes.c_int32()
    _lib.check(_lib.hip_lib().fvm_ell_resident(n, ctypes.byref(fits)), "fvm_ell_resident")
    return bool(fits.value)


def eligible(prob, alg, saveat, user_callback):
    from .problem import FVMProblem

    return (isinstance(prob, FVMProblem) and getattr(alg, "device_loop", True) and user_callback is None
            and saveat is not None and len(prob.initial_condition) <= MAX_N and 1 <= alg.krylov_restart <= 30
            and resident(len(prob.initial_condition)) and is_affine(prob))


def trbdf2_affine(prob, alg, saveat, abstol, reltol, dt, maxiters, save_start):
    """solve(prob, TRBDF2(); saveat) through fvm_trbdf2_affine (see the module
    docstring); the same ODESolution as the host integrator."""
    from .solve import ODESolution, _initial_dt, _Saver

    A = affine_operator(prob)
    ctx = prob.device_context()
    n = A.n
    t0, tf = prob.initial_time, prob.final_time
    u = _lib.DeviceArray.from_host(np.asarray(prob.initial_condition, np.float64))
    fn = _lib.DeviceArray(n)
    nf = 1
    ctx.rhs(u, fn, t0)
    sol = ODESolution()
    saver = _Saver(saveat, t0, tf)
    while saver.k < len(saver.times) and saver.times[saver.k] <= t0 + 1e-14 * max(1, abs(t0)):
        sol.t.append(saver.times[saver.k])
        sol.u.append(u.to_host())
        saver.k += 1
    if dt is None:
        def f(x, out, tt):
            ctx.rhs(x, out, tt)
        dt = _initial_dt(f, u, fn, t0, tf, abstol, reltol, n, exponent=1 / 3)
        nf += 1
    times = np.ascontiguousarray(saver.times[saver.k:], np.float64)
    d_saves = _lib.DeviceArray(max(1, len(times) * n))
    o = TrbOpts()
    o.t0, o.tf, o.dt, o.abstol, o.reltol, o.maxiters = t0, tf, float(dt), abstol, reltol, int(maxiters)
    o.newton_kappa, o.max_newton = alg.newton_kappa, alg.max_newton
    o.krylov_restart, o.krylov_rtol, o.smooth_est = alg.krylov_restart, alg.krylov_rtol, int(alg.smooth_est)
    o.n_save, o.save_t, o.d_saves = len(times), _lib.ptr(times), d_saves.ptr
    st = TrbStats()
    opd = A.op()
    _lib.check(_lib.hip_lib().fvm_trbdf2_affine(ctypes.byref(opd), ctypes.byref(o), u.ptr, ctypes.byref(st), None),
               "fvm_trbdf2_affine")
    if st.nsaved:
        S = d_saves.to_host()[: st.nsaved * n].reshape(st.nsaved, n)
        for k in range(st.nsaved):
            sol.t.append(float(times[k]))
            sol.u.append(S[k].copy())
    sol.retcode = _RETCODES.get(st.retcode, "Failure")
    sol.stats = dict(nf=nf + st.nf, njvp=st.njvp, naccept=st.naccept, nreject=st.nreject, nnewton=st.nnewton,
                     nkrylov=st.nkrylov, nnewton_fail=st.nnewton_fail, device_loop=True,
                     jacobian_colours=A.n_colours)
    sol.final_device = u
    return sol

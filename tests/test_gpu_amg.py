"""The steady templates' default solver (FVM_SOLVE_AUTO): CG preconditioned by the
smoothed-aggregation multigrid of fvm_amg.hip, against SuperLU on the same A and b.

Both stop at |b - A x| <= 1e-10 |b|; the solutions then differ by at most
|A^-1| 1e-10 |b|, measured here as 1e-10 |b| times the norm of A^-1 (power iteration on
the factorisation), and the same call twice gives the same bits."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

import finitevolumemethod as FVM
from finitevolumemethod import CG

pytestmark = pytest.mark.gpu


def _hub(k, rings):
    """A node with k neighbours inside rings of k points each and one of 60: rows longer than
    the strength mask's 64 entries, transposed lists longer than the 128 of a wave."""
    pts = [(0.0, 0.0)]
    for m, r, ph in [(k, 1.0 + 3.0 * q / k, 0.5 * q) for q in range(rings)] + [(60, 1.6, 0.2)]:
        th = 2 * np.pi * (np.arange(m) + ph) / m
        pts += list(zip(r * np.cos(th), r * np.sin(th)))
    P = np.array(pts)
    return FVM.triangulate(P[:, 0], P[:, 1])


def _mesh(kind):
    if kind[0] == "hub":
        return _hub(*kind[1:])
    if kind[0] == "stretched":  # triangles 30 times longer than wide
        return FVM.jittered_rectangle(0.0, 30.0, 0.0, 1.0, *kind[1:], jitter=0.2, seed=4, single_boundary=False)
    if kind == "graded":
        t = FVM.jittered_rectangle(0.0, 1.0, 0.0, 1.0, 71, 67, jitter=0.2, seed=4, single_boundary=False)
        return FVM.Triangulation(t.x * (0.1 + 0.9 * t.x), t.y * (0.3 + 0.7 * t.y), t.triangles, t.boundary_edges, t.boundary_segments)
    nx, ny = kind
    return FVM.jittered_rectangle(0.0, 1.0, 0.0, 1.0, nx, ny, jitter=0.25, seed=11, single_boundary=False)


# up to 3,072 unknowns one workgroup's CG (two, four and six rows a thread: (3, 3), (31, 33),
# (32, 33), (64, 32) and (48, 64), the most; hub of 300: rows far beyond the eight slots), then
# the cycle: (439, 7) just over, (200, 170) four levels; hubs: a row and a list of 300 in a mesh
# of 3,361, of 2,000 in one of 4,061
@pytest.mark.parametrize("kind", [(3, 3), (31, 33), (32, 33), (64, 32), (48, 64), ("hub", 300, 2), ("stretched", 41, 43),
                                  (439, 7), (200, 170), ("stretched", 81, 83), "graded", ("hub", 300, 11),
                                  ("hub", 2000, 2)], ids=str)
@pytest.mark.parametrize("D", ["one", "varying"])
def test_default_steady_solve_matches_a_direct_solution(gpu, kind, D):
    tri = _mesh(kind)
    mesh = FVM.FVMGeometry(tri)
    segs = tri.num_boundary_segments()
    zero = lambda x, y, t, u, p: 0.0 * x  # noqa: E731
    types = tuple(FVM.Dirichlet if k % 2 == 0 else FVM.Neumann for k in range(segs))
    Dfun = (lambda x, y, p: 1.0 + 0.0 * x) if D == "one" else (lambda x, y, p: np.exp(1.5 * np.sin(3 * x / tri.x.max()) * np.cos(4 * y)))
    f = np.random.default_rng(3).uniform(-1, 1, tri.num_points())
    prob = FVM.PoissonsEquation(mesh, FVM.BoundaryConditions(mesh, (zero,) * segs, types),
                                FVM.InternalConditions(lambda x, y, t, u, p: 1.0 + 0.0 * x, dirichlet_nodes={7: 0}),
                                diffusion_function=Dfun, source_function=lambda x, y, p: p, source_parameters=f)
    a = FVM.solve(prob, maxiter=1000)
    assert a.retcode == "Success" and a.resid <= 1e-10, a.stats
    A, b = prob.A.tocsc(), prob.b
    lu = spla.splu(A)
    v = np.random.default_rng(1).standard_normal(len(b))
    for _ in range(20):  # |A^-1|_2
        v /= np.linalg.norm(v)
        v = lu.solve(lu.solve(v), trans="T")
    bound = 1.1 * np.sqrt(np.linalg.norm(v)) * 1e-10 * np.linalg.norm(b)
    x = lu.solve(b)
    assert np.linalg.norm(a.u - x) <= bound + 1e-12 * np.linalg.norm(x)
    if len(b) > 3072:  # the cycle met the target, not the Jacobi-preconditioned CG behind it
        assert FVM.solve(prob, CG(), maxiter=2 * a.iters).retcode == "MaxIters", a.stats
    if kind == (200, 170):
        assert a.iters <= 60, a.stats  # Jacobi-preconditioned CG takes hundreds
    assert np.array_equal(FVM.solve(prob, maxiter=1000).u, a.u)


@pytest.mark.parametrize("k", [127, 129, 4000, 8190, 8192, 20000])
def test_a_row_with_many_entries(gpu, k):
    """A node joined to k others across the mesh: its aggregate's column is in the transposed
    lists of k rows and more, sorted by a wave up to 128 entries, by a workgroup in LDS up to
    8,192 and in memory beyond."""
    from finitevolumemethod.templates import DeviceTemplate

    tri = FVM.triangulate_rectangle(0.0, 1.0, 0.0, 1.0, 150, 140, single_boundary=True)
    mesh = FVM.FVMGeometry(tri)
    n = tri.num_points()
    edges = np.unique(np.sort(np.concatenate([tri.triangles[:, [0, 1]], tri.triangles[:, [1, 2]], tri.triangles[:, [2, 0]]]), axis=1), axis=0)
    hub, others = 75 + 150 * 70, np.random.default_rng(k).permutation(n)[:k]
    i = np.concatenate([edges[:, 0], np.full(k, hub)])
    j = np.concatenate([edges[:, 1], others])
    w = np.concatenate([np.ones(len(edges)), np.full(k, 0.1)]) * (i != j)
    L = sp.coo_matrix((np.concatenate([w, w]), (np.concatenate([i, j]), np.concatenate([j, i]))), shape=(n, n)).tocsr()
    L = sp.diags(np.asarray(L.sum(1)).ravel() + 1e-3) - L
    A = (sp.diags(-1.0 / mesh.cv_volumes) @ L).tocsr()
    A.sort_indices()
    b = np.random.default_rng(1).standard_normal(n) / mesh.cv_volumes
    make = lambda: DeviceTemplate.from_csr(mesh, A.indptr, A.indices, A.data, b, np.zeros(n, bool))  # noqa: E731
    T = make()
    x, st = T.solve(maxiter=200)
    # sorted lists: the same hierarchy bit for bit, though they arrive in the order of atomics
    assert np.array_equal(make().solve(maxiter=200)[0].to_host(), x.to_host())
    assert st["converged"] and st["residual"] <= 1e-10, st
    assert not T.solve(CG(), maxiter=2 * st["iterations"])[1]["converged"]
    ref = spla.spsolve(A.tocsc(), b)
    # |A^-1 r| <= |L^-1| |V r| <= 1e3 max(V) 1e-10 |b|
    bound = 1e3 * mesh.cv_volumes.max() * 1e-10 * np.linalg.norm(b)
    assert np.linalg.norm(x.to_host() - ref) <= bound + 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("n", [30, 60])  # one workgroup's CG, the cycle
def test_a_singular_system_ends_as_it_does_with_jacobi(gpu, n):
    """Zero flux everywhere and a source that does not sum to zero: no solution."""
    tri = FVM.triangulate_rectangle(0.0, 1.0, 0.0, 1.0, n, n, single_boundary=True)
    mesh = FVM.FVMGeometry(tri)
    prob = FVM.PoissonsEquation(mesh, FVM.BoundaryConditions(mesh, lambda x, y, t, u, p: 0.0 * x, FVM.Neumann),
                                source_function=lambda x, y, p: 1.0 + 0.0 * x)
    a, b = FVM.solve(prob, maxiter=500), FVM.solve(prob, CG(), maxiter=500)
    assert a.retcode == b.retcode == "MaxIters" and np.all(np.isfinite(a.u))


def test_a_source_of_one_mode_needs_no_cycle(gpu):
    """sin(pi x) sin(pi y) on a uniform grid is an eigenvector of the scaled operator: the
    Jacobi-preconditioned steps before the cycle meet the target, as CG() does."""
    tri = FVM.triangulate_rectangle(0.0, 1.0, 0.0, 1.0, 70, 70, single_boundary=True)
    mesh = FVM.FVMGeometry(tri)
    prob = FVM.PoissonsEquation(mesh, FVM.BoundaryConditions(mesh, lambda x, y, t, u, p: 0.0 * x, FVM.Dirichlet),
                                source_function=lambda x, y, p: -np.sin(np.pi * x) * np.sin(np.pi * y))
    a, b = FVM.solve(prob), FVM.solve(prob, CG())
    assert a.retcode == "Success" and a.resid <= 1e-10 and a.iters <= 3
    # both residuals are below 1e-10 |b| and |A^-1| <= 1 / (2 pi^2) here, up to the grid's error
    assert np.linalg.norm(a.u - b.u) <= 2e-10 * np.linalg.norm(prob.b) / 19.0 + 1e-12 * np.linalg.norm(b.u)


@pytest.mark.parametrize("nx,ny,cycle", [(1100, 3, False), (1100, 6, False), (1100, 7, True), (30000, 4, False)])
def test_strips_within_two_edges_of_fixed_rows_need_no_cycle(gpu, nx, ny, cycle):
    """Some twenty Jacobi-preconditioned iterations an edge of distance: CG() bit for bit,
    without setting up the multigrid hierarchy."""
    tri = FVM.jittered_rectangle(0.0, nx - 1.0, 0.0, ny - 1.0, nx, ny, jitter=0.25, seed=5, single_boundary=True)
    mesh = FVM.FVMGeometry(tri)
    prob = FVM.PoissonsEquation(mesh, FVM.BoundaryConditions(mesh, lambda x, y, t, u, p: 0.0 * x, FVM.Dirichlet),
                                diffusion_function=lambda x, y, p: 1.0 + 0.0 * x, source_function=lambda x, y, p: p,
                                source_parameters=np.random.default_rng(1).random(tri.num_points()))
    a, b = FVM.solve(prob), FVM.solve(prob, CG())
    assert a.retcode == b.retcode == "Success" and a.resid <= 1e-10
    assert (a.iters < b.iters) == cycle and np.array_equal(a.u, b.u) != cycle, (a.stats, b.stats)

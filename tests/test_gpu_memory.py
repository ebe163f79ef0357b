"""Device memory of fvm_alloc / fvm_free: blocks of 1 to 128 MiB are kept for the next
allocation of their size (at most 512 MiB, none longer than 64 frees), and what happens
when the device has no memory left (the library asks HIP for more than it holds:
fvm_test_fail_allocations)."""
import contextlib
import ctypes
import threading

import numpy as np
import pytest
import torch

import finitevolumemethod as FVM
from finitevolumemethod import _lib

pytestmark = pytest.mark.gpu
MiB = 1 << 20


def _free_bytes():
    _lib.synchronize()
    return torch.cuda.mem_get_info()[0]


@pytest.mark.parametrize("n", [1, MiB // 8 - 1, MiB // 8, MiB // 8 + 1, 16 * MiB, 16 * MiB + 1])
def test_a_block_is_reused_only_after_its_work(gpu, n):
    """Writes to a freed block, queued on a stream of their own, end before the block's
    next owner has it (sizes around both ends of the kept range)."""
    src = FVM.DeviceArray.from_host(np.full(n, 7.0))
    stream = torch.cuda.Stream().cuda_stream
    for _ in range(3):
        a = FVM.DeviceArray(n)
        for _ in range(20):
            _lib.lincomb(a, (1.0,), (src,), stream=stream)
        del a
        b = FVM.DeviceArray.from_host(np.arange(n, dtype=np.float64))
        assert np.array_equal(b.to_host(), np.arange(n, dtype=np.float64))
        del b


def test_threads_get_blocks_of_their_own(gpu):
    bad = []

    def work(k):
        rng = np.random.default_rng(k)
        for r in range(20):
            n = int(rng.choice([MiB // 8, MiB // 8 + 5, MiB // 4]))
            d = FVM.DeviceArray.from_host(np.full(n, 100.0 * k + r))
            e = FVM.DeviceArray.from_host(np.full(n, -100.0 * k - r))
            if not (np.all(d.to_host() == 100.0 * k + r) and np.all(e.to_host() == -100.0 * k - r)):
                bad.append((k, r))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(1, 5)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_kept_memory_is_bounded_and_given_back(gpu):
    torch.cuda.init()
    for _ in range(65):  # what earlier tests left
        FVM.DeviceArray(MiB // 8)
    start = _free_bytes()
    blocks = [FVM.DeviceArray(16 * MiB) for _ in range(8)]  # 1 GiB
    held = start - _free_bytes()
    del blocks
    # HIP accounts for memory in granules and chunks of its own: within 64 MiB
    assert held >= 1024 * MiB - 64 * MiB
    assert start - _free_bytes() <= 512 * MiB + 64 * MiB
    for _ in range(64):
        FVM.DeviceArray(MiB // 8)
    assert start - _free_bytes() <= 64 * MiB


@contextlib.contextmanager
def _failing(after, count):
    f = _lib.hip_lib().fvm_test_fail_allocations
    f.argtypes, f.restype = [ctypes.c_int64, ctypes.c_int64], None
    f(after, count)
    try:
        yield
    finally:
        f(0, 0)


def _poisson(nx, ny):
    tri = FVM.jittered_rectangle(0.0, 1.0, 0.0, 1.0, nx, ny, jitter=0.25, seed=3)
    mesh = FVM.FVMGeometry(tri)
    f = np.random.default_rng(1).random(tri.num_points())
    return FVM.PoissonsEquation(mesh, FVM.BoundaryConditions(mesh, lambda x, y, t, u, p: 0.0 * x, FVM.Dirichlet),
                                diffusion_function=lambda x, y, p: 1.0 + x, source_function=lambda x, y, p: p,
                                source_parameters=f)


# the hierarchy's allocations one after the other: the scratch, the first level, the next ones
@pytest.mark.parametrize("after", [0, 1, 2, 4])
def test_no_room_for_the_hierarchy(gpu, after):
    """The default steady solve without memory for the multigrid hierarchy is the
    Jacobi-preconditioned one, not an error, and the next solve uses the cycle again."""
    from finitevolumemethod import CG

    prob = _poisson(80, 70)
    n = len(prob.b)
    x = FVM.DeviceArray.from_host(np.zeros(n))
    with _failing(after, 1000):
        _, st = prob.problem.solve(x=x)
    ref = FVM.solve(prob, CG())
    assert st["converged"] and st["iterations"] > 60  # the cycle takes under 60, Jacobi some 150
    # both residuals are below 1e-10 |b|; |A^-1| <= 1 / (2 pi^2) for D >= 1, 0.06 with the mesh's error
    bound = 2e-10 * 0.06 * np.linalg.norm(prob.b)
    assert np.linalg.norm(x.to_host() - ref.u) <= bound
    again = FVM.solve(prob)
    assert again.retcode == "Success" and again.iters < 60 and np.linalg.norm(again.u - ref.u) <= bound


@pytest.mark.parametrize("what", ["mesh", "template", "context", "hierarchy"])
def test_kept_blocks_are_given_back_to_every_allocation(gpu, what):
    """An allocation that fails once has the kept blocks' memory the second time."""
    prob = _poisson(80, 70)
    x = FVM.DeviceArray.from_host(np.zeros(len(prob.b)))
    tri = FVM.triangulate_rectangle(0.0, 1.0, 0.0, 1.0, 9, 9, single_boundary=True)
    mesh = FVM.FVMGeometry(tri)
    mesh.handle
    zero = FVM.BoundaryConditions(mesh, lambda x, y, t, u, p: 0.0 * x, FVM.Dirichlet)
    make = {"mesh": lambda: FVM.FVMGeometry(tri).handle,
            "template": lambda: FVM.PoissonsEquation(mesh, zero, diffusion_function=lambda x, y, p: 1.0 + x,
                                                     source_function=lambda x, y, p: x).problem,
            "context": lambda: FVM.FVMProblem(mesh, zero, diffusion_function=lambda x, y, t, u, p: 0.1 + u ** 2,
                                              initial_condition=tri.x, final_time=1.0).device_context(),
            "hierarchy": lambda: prob.problem.solve(x=x)}[what]
    for _ in range(65):  # what earlier work left
        FVM.DeviceArray(MiB // 8)
    blocks = [FVM.DeviceArray(8 * MiB) for _ in range(4)]  # 256 MiB
    del blocks
    before = _free_bytes()
    with _failing(0, 1):
        made = make()
    assert _free_bytes() - before >= 192 * MiB  # HIP accounts for memory in chunks of its own
    if what == "hierarchy":
        assert made[1]["converged"] and made[1]["iterations"] < 60


def test_a_reported_failure_leaves_no_error_behind(gpu):
    """What a caller does after a failed allocation is not taken for that failure."""
    u = FVM.DeviceArray.from_host(np.ones(100))
    with _failing(0, 1000), pytest.raises(_lib.FVMError, match="memory"):
        FVM.DeviceArray(16 * MiB)
    assert _lib.dot(u, u) == 100.0

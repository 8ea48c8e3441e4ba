"""BiCGSTAB solves of a few iterations run no iteration past their last one.

A solve that ends after k iterations is timed with the iteration limit at k,
where nothing can be queued beyond it, and far above k: the solutions are equal
bit for bit, and the times differ by less than half an iteration (one queued
past the end would add a whole one)."""
import ctypes as C
import time

import numpy as np
import pytest

from channel3d_parallel_amd import Channel, ib_geometry
from channel3d_parallel_amd._lib import ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,nth,nzb,graphs", [(66, 65, 66, 48, 64, True), (66, 65, 66, 48, 64, False),
                                                     (34, 33, 34, 24, 16, True)])
def test_short_solves_run_no_idle_iteration(nx, ny, nz, nth, nzb, graphs):
    print(f"\n[case] short solves {nx}x{ny}x{nz} graphs={graphs}", flush=True)
    with Channel(nx, ny, nz, grid_type=0, nu=1e-3) as ch:
        ch.setup_IB(ib_geometry.two_cylinders(ch.grid(11)[9], nzb=nzb, nth=nth))
        ch.set_IB_graphs(graphs)
        n = 4 * ch.nb
        b = ch.schur(np.random.default_rng(3).standard_normal(n), 5e-3)
        x = np.empty(n)
        it, err = C.c_int(), C.c_double()

        def solve(tol, maxit):
            x[:] = 0.0
            t = time.perf_counter()
            ch.L.c3d_ib_bicgstab(ch.h, ptr(x), ptr(b), tol, maxit, 5e-3, 2, C.byref(it), C.byref(err))
            return time.perf_counter() - t

        def best(tol, maxit):
            return min(solve(tol, maxit) for _ in range(20))

        iteration = (best(1e-300, 9) - best(1e-300, 1)) / 8
        for k in (1, 2, 3, 5):
            solve(1e-300, k)
            tol = err.value ** 0.5 * (1 + 1e-6)
            solve(tol, 500)
            ends = it.value  # k, or before where the residual rose in between
            limited = best(tol, ends)
            xl = x.copy()
            free = best(tol, 500)
            assert it.value == ends and np.array_equal(x, xl)
            print(f"  {ends} iterations: {1e6 * limited:.0f} us limited, {1e6 * free:.0f} us free, "
                  f"one iteration {1e6 * iteration:.0f} us", flush=True)
            assert free - limited < 0.5 * iteration

"""The boundary cells that a time step's own kernels write: bitwise what
apply_boundary_conditions makes of the interior, and P's ghosts the copies of
their neighbours, at the smallest grids, odd row counts and with each kind of
projection."""
import numpy as np
import pytest

from channel3d_parallel_amd import Channel, fields, ib_geometry
from channel3d_parallel_amd._lib import PREC_FP64, PREC_MIXED

pytestmark = pytest.mark.gpu

CASES = [(18, 4, 18, "fp64"), (18, 5, 34, "exact"), (34, 38, 18, "fp64"), (66, 66, 50, "fp64"),
         (34, 65, 18, "mixed"), (18, 34, 18, "refined"), (34, 33, 34, "body")]


@pytest.mark.parametrize("nx,ny,nz,kind", CASES)
def test_time_step_boundary_cells(nx, ny, nz, kind):
    print(f"\n[case] boundary cells after a step {nx}x{ny}x{nz} {kind}", flush=True)
    gt = 0 if kind == "body" else 1
    U, V, W = fields.channel_ic(nx, ny, nz, grid_type=gt)
    with Channel(nx, ny, nz, grid_type=gt, nu=1e-3,
                 precision=PREC_MIXED if kind == "mixed" else PREC_FP64) as ch:
        if kind == "body":
            ch.setup_IB(ib_geometry.two_cylinders(ch.grid(11)[9], nzb=16, nth=24))
            ch.set_IB_solver(tol=1e-8, maxit=200)
        if kind == "refined":
            ch.set_refinement(2)
        ch.set_rhs_exact(kind == "exact")
        nan = [np.full(s, np.nan, order="F") for s in (ch.shape_u, ch.shape_v, ch.shape_w, ch.shape_p)]
        for a, b in zip(nan, (U, V, W)):
            a[...] = b
        ch.set_fields(*nan)  # P starts as NaN: every cell has to be written
        ch.apply_boundary_conditions()
        q0 = ch.mean_mass_flow_u()
        for mass in (0, 1):
            ch.compute_time_step_RK3(1e-3, mass, q0 + 1e-3)
            a = ch.get_fields()
            ch.apply_boundary_conditions()
            b = ch.get_fields()
            for k in "UVW":
                assert np.array_equal(a[k], b[k]), (mass, k)
            P = a["P"]
            i = np.clip(np.arange(P.shape[0]), 1, P.shape[0] - 2)
            j = np.clip(np.arange(P.shape[1]), 1, P.shape[1] - 2)
            k = np.clip(np.arange(P.shape[2]), 1, P.shape[2] - 2)
            assert np.isfinite(P).all()
            assert np.array_equal(P, P[np.ix_(i, j, k)])
            assert np.array_equal(P[-2], P[1]) and np.array_equal(P[:, :, -2], P[:, :, 1])

"""Whole-field reductions (compute_dt, monitor, plane statistics) and the
right-hand sides' runs of 2, 4 and 8 planes against the oracle, at sizes around
their tiles: x extents around 64 and 256, plane counts that leave part runs,
3 rows.

Tolerances: maxima, quotients and right-hand sides are exact; sums 1e-13 of
their magnitude (summation order)."""
import numpy as np
import pytest

from channel3d_parallel_amd import Channel, fields
from oracle import orc

pytestmark = pytest.mark.gpu

NU = 1e-3
# the last two: right-hand sides in runs of 4 and of 8 planes
CASES = [(18, 4, 18), (34, 33, 50), (66, 18, 18), (258, 7, 34), (386, 6, 18), (66, 258, 66), (66, 260, 130)]


@pytest.mark.parametrize("nx,ny,nz", CASES)
def test_field_sums(nx, ny, nz):
    print(f"\n[case] field sums {nx}x{ny}x{nz}", flush=True)
    g = orc.Grid(nx, ny, nz)
    U, V, W = fields.white_faces(nx, ny, nz, seed=ny)
    g.apply_bc(U, V, W)
    with Channel(nx, ny, nz, nu=NU) as ch:
        ch.set_fields(U, V, W)
        for k in (0.4, 0.1):
            assert ch.compute_dt(k) == g.compute_dt(U, V, W, k, NU)
        m, st = ch.monitor(), ch.plane_statistics()
        ch.compute_rhs(1)
        F = ch.get_rhs(1)
    r = g.monitor(U, V, W)
    for k in ("maxU", "maxV", "maxW", "nonfinite"):
        assert m[k] == r[k], k
    for k, f in (("meanU", U), ("meanV", V), ("meanW", W)):
        assert abs(m[k] - r[k]) <= 1e-13 * np.abs(f).mean(), k
    for k, v in g.plane_statistics(U, V, W).items():
        assert np.abs(st[k] - v).max() <= 1e-13 * max(np.square(a).max() for a in (U, V, W)), k
    for a, b in zip(F, g.rhs(U, V, W, NU, 0.0, 0.0, 0.0)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("nx,ny,nz", CASES)
def test_fused_stage_matches_bitwise_form(nx, ny, nz):
    print(f"\n[case] fused stages {nx}x{ny}x{nz}", flush=True)
    U, V, W = fields.white_faces(nx, ny, nz, seed=nz)
    out = []
    for exact in (False, True):
        with Channel(nx, ny, nz, nu=NU) as ch:
            ch.set_fields(U, V, W)
            ch.apply_boundary_conditions()
            ch.set_rhs_exact(exact)
            ch.compute_time_step_RK3(1e-5)
            out.append(ch.get_fields())
    for k in "UVW":
        a, b = (o[k] for o in out)
        assert np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(b), k

"""Bulk-flow integral at row counts around its chunks of 16 rows and x extents
around its 64-wide tiles, without and with a body's mask, against the sum in
extended precision.

Tolerance: the summation tree is at most 64 additions deep (16 rows, 6 lane
steps, 4 wavefronts, the ordered sum of the partials), each rounding by half a
unit of the sum of magnitudes."""
import numpy as np
import pytest

from channel3d_parallel_amd import Channel, fields, ib_geometry

pytestmark = pytest.mark.gpu


def bulk(U, yg, H):
    L = np.longdouble
    u, h = U[1:-1, 1:-1, 1:-1].astype(L), H[1:-1, 1:-1, 1:-1].astype(L)
    d = np.diff(yg.astype(L))[1:-1][None, :, None] / 2
    s = ((h * u)[:, 1:] + (h * u)[:, :-1]) * d
    n = ((h[:, 1:] + h[:, :-1]) * d).sum()
    return s.sum() / n, abs(s).sum() / n


@pytest.mark.parametrize("nx,ny,nz", [(18, 4, 18), (34, 18, 18), (66, 19, 34), (98, 35, 18),
                                      (130, 50, 18), (18, 130, 50)])
@pytest.mark.parametrize("body", [False, True])
def test_bulk_flow(nx, ny, nz, body):
    if body and ny < 18:
        pytest.skip("no room for a body")
    print(f"\n[case] bulk flow {nx}x{ny}x{nz} body {body}", flush=True)
    U, V, W = fields.white_faces(nx, ny, nz, seed=ny)
    with Channel(nx, ny, nz, grid_type=0 if body else 1) as ch:
        yg = ch.grid(4)
        H = np.ones(ch.shape_u, order="F")
        if body:
            ch.setup_IB(ib_geometry.two_cylinders(ch.grid(11)[9], nzb=8, nth=12))
            H = ch.ib_heaviside()["Hu_int"]
        ch.set_fields(U, V, W)
        got = ch.mean_mass_flow_u()
        assert ch.mean_mass_flow_u(U) == got
    ref, mag = bulk(U, yg, H)
    assert abs(got - ref) <= 64 * 1.2e-16 * mag, (got, ref)

"""Schur products that transform only the planes near the body (rk_step other
than 1) against those that transform every plane (rk_step 1, which also
writes P): the same numbers, at row counts of each tridiagonal variant."""
import numpy as np
import pytest

from channel3d_parallel_amd import Channel, ib_geometry

pytestmark = pytest.mark.gpu

CASES = [(34, 34, 18, "body"), (34, 65, 34, "body"), (50, 98, 18, "body"), (34, 129, 34, "body"),
         (18, 193, 18, "body"), (18, 600, 18, "body"), (34, 101, 18, "walls"), (18, 33, 18, "body")]


@pytest.mark.parametrize("nx,ny,nz,kind", CASES)
def test_planes_near_the_body(nx, ny, nz, kind):
    print(f"\n[case] planes near the body {nx}x{ny}x{nz} {kind}", flush=True)
    args = dict(grid_type=2, alpha=2.6, min_buffer_width=0.1) if kind == "walls" else dict(grid_type=0)
    with Channel(nx, ny, nz, nu=1e-3, **args) as ch:
        if kind == "walls":
            ch.setup_IB_wave("standing_wave", 32, 16, 0.03, 2.0, 1.0, 0.0, 0.0)
        else:
            ch.setup_IB(ib_geometry.two_cylinders(ch.grid(11)[9], nzb=16, nth=24))
        f = np.random.default_rng(ny).standard_normal(4 * ch.nb)
        for _ in range(2):  # the second product finds the first one's spectrum and potential
            full = ch.schur(f, 0.01, rk_step=1)
            assert np.abs(full).max() > 0
            assert np.array_equal(ch.schur(f, 0.01, rk_step=2), full)
            f = full / np.abs(full).max()


# planes of more than 4608 points, which the separate x and z transforms take
BIG = [(98, 65, 66, "body"), (130, 50, 66, "body"), (50, 101, 130, "body"), (98, 101, 66, "walls"),
       (258, 129, 34, "walls")]


@pytest.mark.parametrize("nx,ny,nz,kind", BIG)
def test_planes_near_the_body_with_separate_transforms(nx, ny, nz, kind):
    print(f"\n[case] planes near the body {nx}x{ny}x{nz} {kind}", flush=True)
    args = dict(grid_type=2, alpha=2.6, min_buffer_width=0.1) if kind == "walls" else dict(grid_type=0)
    with Channel(nx, ny, nz, nu=1e-3, **args) as ch:
        if kind == "walls":
            ch.setup_IB_wave("standing_wave", 32, 16, 0.03, 2.0, 1.0, 0.0, 0.0)
        else:
            ch.setup_IB(ib_geometry.two_cylinders(ch.grid(11)[9], nzb=16, nth=24))
        stages = ch.time_projection(1, 1e-3)[1]
        assert stages["fft_z_fwd"] > 0 and stages["fft_z_inv"] > 0
        f = np.random.default_rng(ny).standard_normal(4 * ch.nb)
        for _ in range(2):  # the second product finds the first one's spectrum and potential
            full = ch.schur(f, 0.01, rk_step=1)
            assert np.abs(full).max() > 0
            assert np.array_equal(ch.schur(f, 0.01, rk_step=2), full)
            f = full / np.abs(full).max()

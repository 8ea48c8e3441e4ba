"""Both transforms of a plane in one kernel: Poisson solves of a host array
and projections against the oracle, for lengths of each radix sequence and
planes from the smallest to the largest that take it.

Tolerance: relative L2 1e-12, as for every projection (test_gpu_projection.py)."""
import numpy as np
import pytest

from channel3d_parallel_amd import Channel, fields
from oracle import orc

pytestmark = pytest.mark.gpu

CASES = [(18, 34, 18), (18, 4, 130), (130, 37, 18), (34, 65, 34), (50, 40, 98), (98, 50, 50),
         (66, 33, 130), (130, 65, 66), (98, 66, 66), (34, 45, 130)]


def rel(a, b):
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


@pytest.mark.parametrize("nx,ny,nz", CASES)
def test_planes(nx, ny, nz):
    print(f"\n[case] plane transforms {nx}x{ny}x{nz}", flush=True)
    g = orc.Grid(nx, ny, nz)
    U, V, W = fields.white_faces(nx, ny, nz, seed=nx + nz)
    g.apply_bc(U, V, W)
    for rk_step in (1, 2):
        u, v, w = (a.copy(order="F") for a in (U, V, W))
        with Channel(nx, ny, nz) as ch:
            ch.set_fields(u, v, w)
            ch.compute_non_IB_projection(1e-3, rk_step=rk_step)
            out = ch.get_fields()
            div = ch.divergence(U, V, W) if rk_step == 1 else None
            if div is not None:
                phi = np.asfortranarray(div.copy())
                ch.solve_poisson_equation(phi)
        P = g.zeros("p")
        ref = g.projection(u, v, w, rk_step=rk_step, dt=1e-3, P=P)
        for name, b in (("U", u), ("V", v), ("W", w), ("P_interim", ref["P_interim"])):
            assert rel(out[name], b) <= 1e-12, name
        if rk_step == 1:
            c = np.s_[1:-1, 1:-1, 1:-1]
            assert rel(out["P"][c], P[c]) <= 1e-12
            # P_interim = solution/dt off the plane that the divergence leaves zero
            assert rel(phi[:, :, :-1], 1e-3 * ref["P_interim"][:, :, :-1]) <= 1e-12


# every pair of lengths that has such a kernel: planes of up to 4608 points
LENGTHS = (16, 32, 48, 64, 96, 128)
PAIRS = [(n, m) for n in LENGTHS for m in LENGTHS if n * m <= 4608]


@pytest.mark.parametrize("nxp,nzp", PAIRS)
def test_every_plane_kernel(nxp, nzp):
    # rows: the fewest of the shape, and up to 12 more
    ny = 129 if nzp == 128 else 65 if (nxp, nzp) == (48, 96) else 34
    nx, ny, nz = nxp + 2, ny + (nxp + 3 * nzp) // 16 % 13, nzp + 2
    print(f"\n[case] plane kernels {nx}x{ny}x{nz}", flush=True)
    g = orc.Grid(nx, ny, nz)
    U, V, W = fields.white_faces(nx, ny, nz, seed=nx + nz)
    g.apply_bc(U, V, W)
    with Channel(nx, ny, nz) as ch:
        ch.set_fields(U, V, W)
        ch.compute_non_IB_projection(1e-3, rk_step=1)
        out = ch.get_fields()
        phi = ch.solve_poisson_equation(np.asfortranarray(ch.divergence(U, V, W)))
        stages = ch.time_projection(1, 1e-3)[1]
    assert stages["fft_z_fwd"] == stages["fft_z_inv"] == 0  # the plane's own kernels ran
    P = g.zeros("p")
    ref = g.projection(U, V, W, rk_step=1, dt=1e-3, P=P)
    for name, b in (("U", U), ("V", V), ("W", W), ("P_interim", ref["P_interim"])):
        assert rel(out[name], b) <= 1e-12, name
    c = np.s_[1:-1, 1:-1, 1:-1]
    assert rel(out["P"][c], P[c]) <= 1e-12
    assert rel(phi[:, :, :-1], 1e-3 * ref["P_interim"][:, :, :-1]) <= 1e-12

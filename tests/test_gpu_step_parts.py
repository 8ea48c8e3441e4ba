"""A time step against its parts called one by one: bitwise.  The step takes
the boundary values of the divergence from the interior, the parts read the
cells that apply_boundary_conditions wrote, so each source of the forward x
transform is compared with and without: cached and streamed FP64 fields (below
and above 128 MB), FP64 with refinement, and FP32 spectra with and without a
sweep.  The two forms do the same operations in the same order, so no
tolerance."""
import numpy as np
import pytest

from channel3d_parallel_amd import Channel, fields
from channel3d_parallel_amd._lib import PREC_FP64, PREC_MIXED

pytestmark = pytest.mark.gpu

CASES = [(18, 4, 130, PREC_FP64, None), (34, 33, 34, PREC_FP64, None), (98, 66, 66, PREC_FP64, None),
         (514, 65, 258, PREC_FP64, None), (50, 34, 18, PREC_FP64, 1), (34, 65, 34, PREC_MIXED, 0),
         (258, 65, 34, PREC_MIXED, 1)]


@pytest.mark.parametrize("nx,ny,nz,precision,sweeps", CASES)
def test_step_equals_its_parts(nx, ny, nz, precision, sweeps):
    print(f"\n[case] step and parts {nx}x{ny}x{nz} precision={precision} sweeps={sweeps}", flush=True)
    U, V, W = fields.white_faces(nx, ny, nz, seed=ny)
    dt = 1e-4
    out = []
    for whole in (True, False):
        with Channel(nx, ny, nz, nu=1e-3, precision=precision) as ch:
            if sweeps is not None:
                ch.set_refinement(sweeps)
            ch.set_rhs_exact(True)
            ch.set_fields(U, V, W)
            ch.apply_boundary_conditions()
            if whole:
                ch.compute_time_step_RK3(dt)
            else:
                ch.save_state()
                for stage in (1, 2, 3):
                    ch.compute_rhs(stage)
                    ch.rk3_update(stage, dt)
                    ch.apply_boundary_conditions()
                    ch.compute_non_IB_projection(dt, rk_step=stage)
                    ch.apply_boundary_conditions()
            out.append(ch.get_fields())
    for k in ("U", "V", "W", "P_interim", "P"):
        assert np.isfinite(out[0][k]).all(), k
        assert np.array_equal(out[0][k], out[1][k]), k

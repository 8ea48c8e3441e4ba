"""Stage times of c3d_time_projection are those of the kernels that a
projection runs: where one kernel does both transforms of a plane (up to 4608
points, FP64 without refinement, 33 rows or more, for long z columns only from
the row count on where it is the faster), the x stages hold them and the z
stages are 0; elsewhere every transform has its stage."""
import pytest

from channel3d_parallel_amd import Channel, fields
from channel3d_parallel_amd._lib import PREC_FP64, PREC_MIXED

pytestmark = pytest.mark.gpu

CASES = [(34, 65, 34, PREC_FP64, None, True), (98, 40, 50, PREC_FP64, None, True), (34, 65, 34, PREC_FP64, 1, False),
         (34, 65, 34, PREC_MIXED, 0, False), (34, 33, 34, PREC_FP64, None, False),
         (98, 65, 66, PREC_FP64, None, False), (34, 45, 130, PREC_FP64, None, False),
         (34, 129, 130, PREC_FP64, None, True), (18, 128, 130, PREC_FP64, None, False),
         (50, 64, 98, PREC_FP64, None, False), (50, 65, 98, PREC_FP64, None, True)]


@pytest.mark.parametrize("nx,ny,nz,precision,sweeps,one", CASES)
def test_stages(nx, ny, nz, precision, sweeps, one):
    print(f"\n[case] stage times {nx}x{ny}x{nz} precision={precision} sweeps={sweeps}", flush=True)
    with Channel(nx, ny, nz, precision=precision) as ch:
        if sweeps is not None:
            ch.set_refinement(sweeps)
        ch.set_fields(*fields.white_faces(nx, ny, nz, seed=1))
        ch.apply_boundary_conditions()
        total, stages = ch.time_projection(5, 1e-3)
    assert total > 0
    for name, ms in stages.items():
        assert (ms == 0) if one and name.startswith("fft_z") else ms > 0, name

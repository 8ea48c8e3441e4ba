"""Field summaries and plane statistics of short x rows, which share a
wavefront (16, 32 or 64 lanes a row), around those lengths and around the rows
of a unit, against sums in extended precision and the oracle.

Tolerances as in test_gpu_field_sums.py: maxima and counts exact, sums 1e-13 of
their magnitude (summation order)."""
import ctypes as C

import numpy as np
import pytest
import torch

from channel3d_parallel_amd import Channel, _lib, fields
from oracle import orc

pytestmark = pytest.mark.gpu

SIZES = [(3, 3, 3), (4, 20, 5), (16, 18, 7), (17, 33, 4), (18, 5, 19), (32, 12, 9), (33, 19, 5),
         (34, 6, 34), (64, 9, 11), (65, 5, 6), (66, 4, 5), (258, 5, 4), (259, 4, 3), (18, 300, 40)]


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_monitor_rows(nx, ny, nz):
    print(f"\n[case] monitor rows {nx}x{ny}x{nz}", flush=True)
    r = np.random.default_rng(nx * ny + nz)
    # (z, y, x) C-ordered is (x, y, z) Fortran-ordered
    F = [r.standard_normal(s) for s in ((nz + 1, ny + 1, nx), (nz + 1, ny, nx + 1), (nz, ny + 1, nx + 1))]
    F[0][1, 1, 1] = np.nan
    for a in F:  # boundary cells do not count
        for ax in range(3):
            b = np.moveaxis(a, ax, 0)
            b[0] = b[-1] = np.inf
    L = _lib.load()
    L.c3d_monitor_noalloc.restype = C.c_int
    L.c3d_monitor_noalloc.argtypes = [C.c_int, C.c_int, C.c_int] + [C.c_void_p] * 5
    d = [torch.from_numpy(a).cuda() for a in F]
    out = torch.full((7,), -1.0, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    assert L.c3d_monitor_noalloc(nx, ny, nz, *(t.data_ptr() for t in d), out.data_ptr(), None) == 0
    torch.cuda.synchronize()
    o = out.cpu().numpy()
    vol = (nx - 1) * (ny - 1) * (nz - 1)
    assert o[6] == 1
    for c, a in enumerate(F):
        i = a[1:-1, 1:-1, 1:-1]
        assert o[c] == (np.nanmax(i) if i.size > 1 or c else -np.inf)
        if c == 0:
            assert np.isnan(o[3])
        else:
            s = i.astype(np.longdouble).sum() / vol
            assert abs(o[3 + c] - s) <= 1e-13 * np.abs(i).sum() / vol


@pytest.mark.parametrize("nx,ny,nz", [(18, 300, 18), (18, 40, 66), (34, 300, 34), (34, 9, 130), (50, 30, 34)])
def test_statistics_rows(nx, ny, nz):
    print(f"\n[case] statistics rows {nx}x{ny}x{nz}", flush=True)
    g = orc.Grid(nx, ny, nz)
    U, V, W = fields.white_faces(nx, ny, nz, seed=ny)
    g.apply_bc(U, V, W)
    with Channel(nx, ny, nz) as ch:
        ch.set_fields(U, V, W)
        m, st = ch.monitor(), ch.plane_statistics()
    r = g.monitor(U, V, W)
    for k in ("maxU", "maxV", "maxW", "nonfinite"):
        assert m[k] == r[k], k
    for k, f in (("meanU", U), ("meanV", V), ("meanW", W)):
        assert abs(m[k] - r[k]) <= 1e-13 * np.abs(f).mean(), k
    for k, v in g.plane_statistics(U, V, W).items():
        assert np.abs(st[k] - v).max() <= 1e-13 * max(np.square(a).max() for a in (U, V, W)), k

"""Poisson solves at row counts around the edges of the partitioned
tridiagonal solver (parts of a fixed number of rows, the last ones short or
empty) against the oracle.

Tolerance: both sides are backward-stable eliminations, so their relative
difference is bounded by the unit round-off times the condition number of the
worst mode, at most max|Dyy| over the smallest |eigenvalue| (above 1)."""
import numpy as np
import pytest

from channel3d_parallel_amd import Channel
from oracle import orc

pytestmark = pytest.mark.gpu

ROWS = [3, 4, 15, 16, 17, 63, 65, 79, 80, 81, 96, 97, 113, 127, 129, 159, 161, 191, 193, 256, 257,
        320, 321, 384, 385, 512, 513, 768, 769]


@pytest.mark.parametrize("nym", ROWS)
def test_poisson_row_counts(nym):
    nx, ny, nz = (18, nym + 1, 34) if nym % 2 else (34, nym + 1, 18)
    print(f"\n[case] poisson with {nym} rows", flush=True)
    g = orc.Grid(nx, ny, nz)
    rhs = np.asfortranarray(np.random.default_rng(nym).standard_normal(g.shape_rhs))
    with Channel(nx, ny, nz) as ch:
        dmax = np.max(np.abs(ch.grid(8)))
        got = ch.solve_poisson_equation(rhs.copy(order="F"))
    ref = g.poisson(rhs.copy(order="F"))
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert err <= 2.3e-16 * max(dmax, 100.0), err

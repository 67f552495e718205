"""The snapshot's kernels at the edges of their shares of the rows: the pressure's
right-hand side in pieces of 4 and of 16 rows, the statistics and the column
energies with few rows and with columns that do not fill a block."""
import dataclasses

import numpy as np
import pytest

from conftest import deck_path
from homogenenousshearturbulence_amd import hst
from homogenenousshearturbulence_amd.deck import read_input

pytestmark = pytest.mark.gpu


def pair(oracle, nx, ny, nz, precision):
    d = dataclasses.replace(read_input(deck_path("small")), nx=nx, ny=ny, nz=nz, kpeak=2.0)
    o = oracle.Oracle(d)
    o.initial_field()
    o.fill_all_ghosts(0.3)
    o.time = 0.3
    s = hst.Solver(d, precision)
    s.set_V(o.V)
    s.time = 0.3
    return o, s


# 8,128 columns x 257 rows: pieces of 16, one row in the last.  FP64: the solve's
# condition, (ny / 2)^2, of roundings; mixed: the products' FP32 roundings
@pytest.mark.parametrize("nx,ny,nz", [(5, 8, 4), (5, 9, 4), (5, 21, 4), (63, 257, 63), (63, 271, 63)])
@pytest.mark.parametrize("precision,tol", [(hst.FP64, 1e-10), (hst.MIXED, 2e-5)])
def test_pressure(oracle_built, nx, ny, nz, precision, tol):
    o, s = pair(oracle_built, nx, ny, nz, precision)
    try:
        got = s.pressure(hst.SCRATCH)[..., 2:-2]
    finally:
        s.close()
    want = o.pressure()[..., 2:-2]
    assert float(np.abs(got - want).max() / np.abs(want).max()) <= tol


# columns: 36, 256 + 17, 65,661: one part a column
@pytest.mark.parametrize("nx,ny,nz", [(3, 8, 4), (6, 9, 19), (20, 33, 6), (128, 11, 254)])
def test_statistics(oracle_built, nx, ny, nz):
    """The statistics (sums of squares: rounding) and two samples of the energies."""
    o, s = pair(oracle_built, nx, ny, nz, hst.FP64)
    try:
        s.outstats()
        got = s.outstats()
        E, n = s.spectrum()
    finally:
        s.close()
    want, d = o.outstats(), o.deck
    assert np.allclose(got, want, rtol=1e-11, atol=1e-12 * np.abs(want).max())
    e = o.column_energy()
    e[0, d.nz] -= (want[8] ** 2 + want[9] ** 2) / o.dyl.sum()
    assert n == 2
    assert np.allclose(E, 0.5 * e, rtol=1e-12, atol=1e-13 * np.abs(e).max())

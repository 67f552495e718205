"""The line solves on both sides of the lines between their block shapes: the implicit
ones (two wavefronts while all blocks are resident, three a CU or what LDS holds; four
above) with factor tables and without, the compact ones (one wavefront while resident,
four above, the coefficients' copy up to 65,536 columns)."""
import dataclasses

import numpy as np
import pytest

from conftest import deck_path
from homogenenousshearturbulence_amd import hst
from homogenenousshearturbulence_amd.deck import read_input

pytestmark = pytest.mark.gpu


def deck(nx, ny, nz):
    return dataclasses.replace(read_input(deck_path("small")), nx=nx, ny=ny, nz=nz, exact_shift=False, kpeak=2.0,
                               ystretch=0.8)


# blocks of both systems: 766 and 776 (three a CU), 522 with two a CU (409 rows), and
# without the copy (410); against the same modes among few.  The systems are dominated
# by lambda: a few hundred roundings
@pytest.mark.parametrize("nx,nz,ny", [(155, 156, 16), (155, 158, 16), (128, 128, 409), (128, 128, 410)])
def test_pair(nx, nz, ny):
    few = (5, 4)
    rng = np.random.default_rng(11)
    rhs = rng.standard_normal((2, few[0] + 1, 2 * few[1] + 1, ny + 4, 2)) @ np.array([1.0, 1j])
    rhs[:, 0, few[1]] = 0.0
    out = []
    for x, z in (few, (nx, nz)):
        s = hst.Solver(deck(x, ny, z), hst.FP64)
        try:
            cut = np.s_[: few[0] + 1, z - few[1]: z + few[1] + 1]
            for k, fid in enumerate((hst.RHS1, hst.RHS2)):
                F = np.zeros(s.shape, dtype=np.complex128)
                F[cut] = rhs[k]
                s.upload(fid, F)
            s.linsolve(2.0e3, 0.2)
            out.append([s.download(c)[cut][..., 2:-2] for c in (hst.V1, hst.V2, hst.V3)])
        finally:
            s.close()
    for a, b in zip(*out):
        assert np.abs(a).max() > 0
        assert float(np.abs(a - b).max() / np.abs(a).max()) <= 1e-11


# 98,125 and 98,787 columns: 767 and 772 blocks of one system
@pytest.mark.parametrize("nx,nz", [(156, 312), (220, 223)])
@pytest.mark.parametrize("kind", [1, 2, 3])
def test_one_system(oracle_built, nx, nz, kind):
    d = deck(nx, 9, nz)
    o = oracle_built.Oracle(d)
    rng = np.random.default_rng(kind)
    s = hst.Solver(d, hst.FP64)
    try:
        F = rng.standard_normal(s.shape + (2,)) @ np.array([1.0, 1j])
        F[0, nz] = 0.0
        s.upload(hst.SCRATCH, F)
        s.line_solve(kind, 123.4, hst.SCRATCH, hst.RHS2, 0.3, 0.2)
        got = s.download(hst.RHS2)[..., 2:-2]
    finally:
        s.close()
    o.field(8)[...] = F
    o.line_solve(kind, 123.4, 8, 5, 0.3, 0.2)
    want = o.field(5)[..., 2:-2].copy()
    if kind in (1, 3):  # the mean mode is zero or left alone
        got[0, nz] = want[0, nz] = 0.0
    assert float(np.abs(got - want).max() / np.abs(want).max()) <= 1e-11


# 510 and 514 blocks of one wavefront, two a CU (585 rows); 857 without the copy, three
# a CU (586 rows); 65,403 and 65,703 columns; against the same modes among few.  The
# compact systems are dominated by their diagonals: a few hundred roundings
@pytest.mark.parametrize("nx,nz,ny", [(127, 127, 585), (127, 128, 585), (103, 263, 586), (168, 193, 9),
                                      (180, 181, 9)])
def test_compact(nx, nz, ny):
    few = (5, 4)
    rng = np.random.default_rng(ny)
    f = rng.standard_normal((few[0] + 1, 2 * few[1] + 1, ny + 4, 2)) @ np.array([1.0, 1j])
    out = []
    for x, z in (few, (nx, nz)):
        s = hst.Solver(deck(x, ny, z), hst.FP64)
        try:
            cut = np.s_[: few[0] + 1, z - few[1]: z + few[1] + 1]
            F = np.zeros(s.shape, dtype=np.complex128)
            F[cut] = f
            s.upload(hst.SCRATCH, F)
            got = []
            for kind in (4, 5):
                s.line_solve(kind, 0.0, hst.SCRATCH, hst.RHS2, 0.3, 0.2)
                got.append(s.download(hst.RHS2)[cut][..., 2:-2])
            for fid in (hst.RHS1, hst.RHS2):
                s.upload(fid, F)
            s.linsolve(2.0e3, 0.2)  # (dv/dy with u and w)
            got += [s.download(c)[cut][..., 2:-2] for c in (hst.V1, hst.V3)]
            out.append(got)
        finally:
            s.close()
    for a, b in zip(*out):
        assert np.abs(a).max() > 0
        assert float(np.abs(a - b).max() / np.abs(a).max()) <= 1e-11

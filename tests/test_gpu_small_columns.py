"""The column kernels of small grids: dv/dy with its columns in LDS (64 and 32 a
wavefront) and by the streamed sweep between that and the one-sweep kernel, the
three fields of the statistics in one launch, and line solves of column ranges
at the edges of a wavefront, with and without the coefficients' LDS copy."""
import dataclasses

import numpy as np
import pytest
import torch  # (first: its HIP runtime has to be the one in the process)

from conftest import deck_path
from homogenenousshearturbulence_amd import hst
from homogenenousshearturbulence_amd.deck import read_input

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


def deck(nx, ny, nz, **k):
    return dataclasses.replace(read_input(deck_path("small")), nx=nx, ny=ny, nz=nz, kpeak=2.0, **k)


# ny - 2 = 112 is the first line the one-sweep dv/dy takes; 64 columns a wavefront
# to ny = 138, 32 to 257; 300 rows: the streamed sweep on few columns; 16,471
# columns x 116 rows: the streamed sweep; 30,495: the window
@pytest.mark.parametrize("nx,ny,nz", [(3, 113, 3), (7, 114, 4), (15, 138, 15), (6, 139, 9), (5, 257, 6), (5, 300, 4),
                                      (90, 116, 90), (106, 114, 142)])
def test_steps_and_statistics(oracle_built, nx, ny, nz):
    """Two steps, then the ten statistics; tolerances: rounding of whole steps
    and of sums of squares."""
    d = deck(nx, ny, nz)
    o = oracle_built.Oracle(d)
    o.initial_field()
    o.fill_all_ghosts(0.0)
    s = hst.Solver(d, hst.FP64)
    try:
        s.set_V(o.V)
        s.reset_old()
        s.fill_all_ghosts(0.0)
        for _ in range(2):
            o.timestep(1e-3)
            s.timestep(1e-3)
        V, st = s.V, s.outstats()
    finally:
        s.close()
    for c in range(3):
        assert rel(V[c][..., 2:-2], o.V[c][..., 2:-2]) <= 1e-11, c
    want = o.outstats()
    assert np.allclose(st, want, rtol=1e-10, atol=1e-10 * np.abs(want).max())


@pytest.mark.parametrize("ny", [8, 9, 17, 65, 410, 586])
@pytest.mark.parametrize("kind", [1, 2, 3, 4, 5])
def test_line_ranges(oracle_built, ny, kind):
    """Ranges of 1, 63, 64, 65 and all columns against line_solve of the oracle."""
    d = deck(5, ny, 8)
    o = oracle_built.Oracle(d)
    rng = np.random.default_rng(ny)
    s = hst.Solver(d, hst.FP64)
    try:
        F = rng.standard_normal(s.shape) + 1j * rng.standard_normal(s.shape)
        o.field(8)[...] = F
        o.line_solve(kind, 123.4, 8, 5, 0.3, 0.2)
        want = o.field(5).transpose(2, 0, 1).reshape(ny + 4, -1)[2:-2]
        A = F.transpose(2, 0, 1).reshape(ny + 4, -1)
        ncol = A.shape[1]
        for col0, n in ((0, ncol), (1, 1), (3, 63), (0, 64), (20, 65), (ncol - 1, 1)):
            src = torch.from_numpy(np.ascontiguousarray(A[:, col0:col0 + n])).to("cuda")
            dst = torch.zeros_like(src)
            s.line_solve_noalloc(kind, 123.4, col0, n, src.data_ptr(), dst.data_ptr(), 0.3, 0.2)
            s.sync()
            got = dst.cpu().numpy()[2:-2]
            cols = np.arange(col0, col0 + n)
            if kind in (1, 3):  # the mean mode is zero or left alone
                keep = cols != d.nz
                got, cols = got[:, keep], cols[keep]
            if cols.size:
                assert np.abs(got - want[:, cols]).max() <= 1e-11 * np.abs(want).max(), (col0, n)
    finally:
        s.close()

"""The column kernels of large grids against the oracle, which thin decks do not
reach: the one-sweep dv/dy and oldrhs shift (blocks of four wavefronts) and the fused
shift and solve from checkpoints, on a stretched grid with their coefficients in LDS
and on lines too long for that."""
import dataclasses

import numpy as np
import pytest

from conftest import deck_path
from homogenenousshearturbulence_amd import hst
from homogenenousshearturbulence_amd.deck import read_input

pytestmark = pytest.mark.gpu

# name: nx, ny, nz, stretch, HST_TABLES_MB.  33,153 columns; 16,471, whose whole
# factorisation (2.4 GB) the limit leaves out and whose 690 rows exceed the copies
DECKS = {"stretched": (128, 257, 128, 2.0, None), "long": (90, 690, 90, 0.0, 400)}


@pytest.fixture(scope="module", params=DECKS)
def case(request, oracle_built):
    """A deck, its table limit, the field after a step and the time, by the oracle."""
    nx, ny, nz, stretch, limit = DECKS[request.param]
    d = dataclasses.replace(read_input(deck_path("small")), nx=nx, nz=nz, ny=ny, kpeak=3.0, alfa0=1.0, beta0=1.0,
                            ly=2 * np.pi, re=1000.0, amplitude=0.002, deltat=0.001, exact_shift=True,
                            ystretch=stretch)
    o = oracle_built.run_deck(d, nsteps=1)
    return d, limit, o.V.copy(), o.time


@pytest.mark.parametrize("precision,tol", [(hst.FP64, 1e-11), (hst.MIXED, 2e-5)])
def test_one_step(case, monkeypatch, precision, tol):
    d, limit, want, time = case
    if limit is not None:
        monkeypatch.setenv("HST_TABLES_MB", str(limit))
    s = hst.Solver(d, precision)
    try:
        before = s.memory()[0]
        hst.run_deck(d, precision, nsteps=1, solver=s)
        assert s.time == time
        # checkpoints, and the one-sweep dv/dy (two fields)
        assert s.memory()[0] - before == 6 * (d.nx + 1) * (d.nz + 1) * 2 * ((d.ny - 2 + 7) // 8) * 32
        V = s.V
        s.profile(True)
        s.timestep(d.deltat)
        row = next(r for r in s.profile_table() if r["kernel"] == "dvdy")
        s.profile(False)
        assert row["bytes"] / row["launches"] == 2 * 16.0 * (d.nx + 1) * (2 * d.nz + 1) * d.ny
    finally:
        s.close()
    for c in range(3):
        a, b = V[c][..., 2:-2], want[c][..., 2:-2]
        assert float(np.abs(a - b).max() / np.abs(b).max()) <= tol, c

"""The right-hand sides of a time step at the edges of their row chunks (2, 4,
8 or 16 rows a lane, by the grid's size), vs the oracle: rows that are no
multiple of the chunk, a single row in the last one, every size of chunk."""
import dataclasses

import numpy as np
import pytest

from conftest import deck_path
from homogenenousshearturbulence_amd import hst
from homogenenousshearturbulence_amd.deck import read_input

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


# chunks of 2 (4 x 7 columns), 4 (33 x 65), 8 (86 x 183) and 16 rows (101 x 255:
# 101 blocks a chunk, 41 chunks)
@pytest.mark.parametrize("nx,ny,nz", [(3, 9, 3), (3, 17, 4), (32, 65, 32), (32, 62, 32), (85, 49, 91), (100, 641, 127)])
@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("precision,tol", [(hst.FP64, 1e-11), (hst.MIXED, 2e-5)])
def test_one_step(oracle_built, nx, ny, nz, exact, precision, tol):
    if ny > 600 and exact != (precision == hst.MIXED):
        pytest.skip("the largest grid once per precision")
    d = dataclasses.replace(read_input(deck_path("small")), nx=nx, ny=ny, nz=nz, exact_shift=exact, kpeak=3.0,
                            s2_mean=0.2, s2_amplitude=0.3, s2_period=1.0)
    o = oracle_built.Oracle(d)
    o.initial_field()
    o.fill_all_ghosts(0.0)
    s = hst.Solver(d, precision)
    try:
        s.set_V(o.V)
        s.reset_old()
        s.fill_all_ghosts(0.0)
        o.timestep(1e-3)
        s.timestep(1e-3)
        V = s.V
    finally:
        s.close()
    for c in range(3):
        assert rel(V[c][..., 2:-2], o.V[c][..., 2:-2]) <= tol, c

"""The right-hand sides of a time step in chunks of 64 rows (grids of which 16 rows of
the fields read exceed 256 MB), the last chunk of two rows, vs the oracle."""
import dataclasses

import numpy as np
import pytest

from conftest import deck_path
from homogenenousshearturbulence_amd import hst
from homogenenousshearturbulence_amd.deck import read_input

pytestmark = pytest.mark.gpu


# 150,405 columns of 112 B a row in FP64, 233,585 of 72 B in the mixed form
@pytest.mark.parametrize("nx,nz,precision,tol", [(270, 277, hst.FP64, 1e-11), (340, 342, hst.MIXED, 2e-5)])
def test_one_step(oracle_built, nx, nz, precision, tol):
    d = dataclasses.replace(read_input(deck_path("small")), nx=nx, ny=66, nz=nz, kpeak=3.0, s2_mean=0.2,
                            s2_amplitude=0.3, s2_period=1.0)
    o = oracle_built.Oracle(d)
    o.initial_field()
    o.fill_all_ghosts(0.0)
    s = hst.Solver(d, precision)
    try:
        s.set_V(o.V)
        s.reset_old()
        s.fill_all_ghosts(0.0)
        o.timestep(1e-4)
        s.timestep(1e-4)
        V = s.V
    finally:
        s.close()
    for c in range(3):
        a, b = V[c][..., 2:-2], o.V[c][..., 2:-2]
        assert float(np.abs(a - b).max() / np.abs(b).max()) <= tol, c

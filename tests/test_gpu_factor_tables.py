"""The line solves' factor tables: the whole factorisation on small grids (the
columns at and above which a time step keeps checkpoints instead, with and
without the exact shift), lines shorter than the rows loaded ahead, a step
length that changes every step, and tables taken by the pieces between steps."""
import dataclasses

import numpy as np
import pytest

from conftest import deck_path
from homogenenousshearturbulence_amd import hst
from homogenenousshearturbulence_amd.deck import read_input

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


def start(oracle, d, precision):
    o = oracle.Oracle(d)
    o.initial_field()
    o.fill_all_ghosts(0.0)
    s = hst.Solver(d, precision)
    s.set_V(o.V)
    s.reset_old()
    s.fill_all_ghosts(0.0)
    return o, s


# 8 .. 19 rows; 26,741 columns: checkpoints without the exact shift, the whole
# factorisation with it; 33,981: checkpoints in both
@pytest.mark.parametrize("nx,ny,nz", [(3, 8, 3), (5, 9, 4), (15, 11, 15), (20, 18, 9), (31, 19, 5), (120, 12, 110),
                                      (140, 9, 120)])
@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("precision,tol", [(hst.FP64, 1e-11), (hst.MIXED, 2e-5)])
def test_two_steps(oracle_built, nx, ny, nz, exact, precision, tol):
    d = dataclasses.replace(read_input(deck_path("small")), nx=nx, ny=ny, nz=nz, exact_shift=exact, kpeak=2.0,
                            ystretch=1.0)
    o, s = start(oracle_built, d, precision)
    try:
        for _ in range(2):
            o.timestep(1e-3)
            s.timestep(1e-3)
        V = s.V
    finally:
        s.close()
    for c in range(3):
        assert rel(V[c][..., 2:-2], o.V[c][..., 2:-2]) <= tol, c


@pytest.mark.parametrize("nx,nz", [(15, 15), (120, 110)])
@pytest.mark.parametrize("exact", [False, True])
def test_changing_step_length(oracle_built, nx, nz, exact):
    """Steps of different lengths, the same again, and a linsolve of its own at
    another lambda between them (which takes one of the tables' places)."""
    d = dataclasses.replace(read_input(deck_path("small")), nx=nx, ny=16, nz=nz, exact_shift=exact, kpeak=2.0)
    o, s = start(oracle_built, d, hst.FP64)
    try:
        for dt in (1e-3, 7e-4, 7e-4, 1.3e-3, 1e-3):
            o.timestep(dt)
            s.timestep(dt)
        V = s.V
        rhs = s.download(hst.RHS1), s.download(hst.RHS2)
        s.linsolve(123.4, s.time)
        s.upload(hst.RHS1, rhs[0])
        s.upload(hst.RHS2, rhs[1])
        s.set_V(V)
        for dt in (1e-3, 5e-4):
            o.timestep(dt)
            s.timestep(dt)
        W = s.V
    finally:
        s.close()
    for c in range(3):
        assert rel(W[c][..., 2:-2], o.V[c][..., 2:-2]) <= 1e-11, c

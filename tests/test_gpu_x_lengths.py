"""The x pass at every line length it is built for, vs the oracle: the longest
and the shortest set of kept modes of a length, lengths with a factor three
(the lanes of a line that hold no elements, the radix-3 stage) among them."""
import dataclasses

import numpy as np
import pytest

from conftest import deck_path
from homogenenousshearturbulence_amd import hst
from homogenenousshearturbulence_amd.deck import read_input

pytestmark = pytest.mark.gpu

# nx, nxd: the lengths' first and last nx
LENGTHS = [(7, 12), (8, 16), (10, 16), (11, 24), (15, 24), (16, 32), (20, 32), (21, 48), (31, 48), (43, 96), (63, 96),
           (86, 192), (127, 192), (171, 384), (255, 384), (511, 768), (700, 1536)]


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("nx,nxd", LENGTHS)
@pytest.mark.parametrize("precision,tol", [(hst.FP64, 1e-12), (hst.MIXED, 2e-5)])
def test_products_and_cfl(oracle_built, nx, nxd, precision, tol):
    """The six products with their ghost rows and the CFL number; tolerances:
    the rounding of one transform pass, as for the other lengths."""
    d = dataclasses.replace(read_input(deck_path("small")), nx=nx, nz=5, ny=9, kpeak=3.0)
    assert d.nxd == nxd
    o = oracle_built.Oracle(d)
    o.initial_field()
    o.fill_all_ghosts(0.17)
    cfl = o.nonlinear(mode=0, want_cfl=True)
    P0 = o.products()
    s = hst.Solver(d, precision)
    try:
        s.set_V(o.V)
        got = s.nonlinear(want_cfl=True)
        P = [s.product(p + 1) for p in range(6)]
        assert s.compute_cfl() == got
    finally:
        s.close()
    assert abs(got - cfl) <= tol * cfl
    for p in range(6):
        assert rel(P[p], P0[p]) <= tol, p


@pytest.mark.parametrize("nx", [15, 31, 63, 127, 255, 511])
@pytest.mark.parametrize("precision,tol", [(hst.FP64, 1e-11), (hst.MIXED, 2e-5)])
def test_two_steps(oracle_built, nx, precision, tol):
    """Two time steps (the five combinations) vs the oracle."""
    d = dataclasses.replace(read_input(deck_path("small")), nx=nx, nz=5, ny=17, kpeak=3.0)
    o = oracle_built.Oracle(d)
    o.initial_field()
    o.fill_all_ghosts(0.0)
    s = hst.Solver(d, precision)
    try:
        s.set_V(o.V)
        s.reset_old()
        s.fill_all_ghosts(0.0)
        for _ in range(2):
            o.timestep(1e-3)
            s.timestep(1e-3)
        V = s.V
    finally:
        s.close()
    for c in range(3):
        assert rel(V[c][..., 2:-2], o.V[c][..., 2:-2]) <= tol, c

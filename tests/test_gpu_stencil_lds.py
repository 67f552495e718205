"""The line solves whose stencil rows are copied to LDS (up to 409 rows) and those
that read them from global memory (from 410 on): the pressure of a small grid
against the oracle, and the implicit solves of a grid with checkpoint tables
against those of a grid with the same modes among fewer."""
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


# the Poisson solve's condition is about (ny / 2)^2: 4e4 roundings, with a factor
# of ten for the stencils' large entries 1e-10
@pytest.mark.parametrize("ny", [9, 409, 410])
def test_pressure(oracle_built, ny):
    d = deck(5, ny, 4)
    o = oracle_built.Oracle(d)
    o.initial_field()
    o.fill_all_ghosts(0.3)
    o.time = 0.3
    want = o.pressure()[..., 2:-2]
    s = hst.Solver(d, hst.FP64)
    try:
        s.set_V(o.V)
        s.time = 0.3
        got = s.pressure(hst.SCRATCH)[..., 2:-2]
    finally:
        s.close()
    assert float(np.abs(got - want).max() / np.abs(want).max()) <= 1e-10


# 24,295 columns: checkpoints; the small grid takes the whole factorisation.  The
# systems are dominated by lambda: a few hundred roundings
@pytest.mark.parametrize("ny", [16, 409, 410])
def test_linsolve(ny):
    big, small = (112, 107), (5, 4)
    rng = np.random.default_rng(11)
    rhs = rng.standard_normal((2, small[0] + 1, 2 * small[1] + 1, ny + 4)) + 0j
    rhs += 1j * rng.standard_normal(rhs.shape)
    rhs[:, 0, small[1]] = 0.0
    out = {}
    for nx, nz in (small, big):
        s = hst.Solver(deck(nx, ny, nz), hst.FP64)
        try:
            cut = np.s_[: small[0] + 1, nz - small[1] : nz + small[1] + 1]
            for k, fid in enumerate((hst.RHS1, hst.RHS2)):
                F = np.zeros(s.shape, dtype=np.complex128)
                F[cut] = rhs[k]
                s.upload(fid, F)
            s.linsolve(2.0e3, 0.2)
            out[nx] = [s.download(c)[cut][..., 2:-2] for c in (hst.V1, hst.V2, hst.V3)]
        finally:
            s.close()
    for a, b in zip(out[big[0]], out[small[0]]):
        assert np.abs(b).max() > 0
        assert float(np.abs(a - b).max() / np.abs(b).max()) <= 1e-11

"""Field transfers through the pinned pieces (16 MiB): downloads below a piece, of
one and 4 KB, of several with a remainder, uploads below and above three pieces,
FP64 and the mixed form's FP32 oldrhs."""
import dataclasses

import numpy as np
import pytest

from conftest import deck_path
from homogenenousshearturbulence_amd import hst
from homogenenousshearturbulence_amd.deck import read_input

pytestmark = pytest.mark.gpu


# (nx + 1)(2 nz + 1)(ny + 4) 16 bytes: 7 kB, 8.4 MB, 16 MiB + 4 KB, 3.4 pieces
@pytest.mark.parametrize("nx,ny,nz", [(3, 12, 3), (127, 237, 8), (127, 478, 8), (63, 401, 69)])
@pytest.mark.parametrize("precision", [hst.FP64, hst.MIXED])
def test_fields_come_back(nx, ny, nz, precision):
    d = dataclasses.replace(read_input(deck_path("small")), nx=nx, ny=ny, nz=nz)
    s = hst.Solver(d, precision)
    try:
        rng = np.random.default_rng(nx)
        fields = {f: rng.standard_normal(s.shape) + 1j * rng.standard_normal(s.shape)
                  for f in (hst.V1, hst.SCRATCH, hst.OLD1)}
        for f, a in fields.items():
            s.upload(f, a)
        for f, a in fields.items():
            want = a
            if precision == hst.MIXED and f == hst.OLD1:
                want = a.astype(np.complex64).astype(np.complex128)
            for _ in range(2):
                assert np.array_equal(s.download(f), want), f
    finally:
        s.close()

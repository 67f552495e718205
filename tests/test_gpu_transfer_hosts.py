"""Field transfers of other host memory than an ordinary array, on both sides of the
sizes from which several threads copy (16 MiB down, 48 MiB up)."""
import dataclasses
import time

import numpy as np
import pytest
import torch  # (first: its HIP runtime has to be the one in the process)

from conftest import deck_path
from homogenenousshearturbulence_amd import hst
from homogenenousshearturbulence_amd.deck import read_input

pytestmark = pytest.mark.gpu

SIZES = [(3, 12, 3), (127, 478, 8), (63, 401, 69)]  # 7 kB, 16 MiB + 4 KB, 54 MiB


def solver(nx, ny, nz):
    return hst.Solver(dataclasses.replace(read_input(deck_path("small")), nx=nx, ny=ny, nz=nz), hst.FP64)


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_null_is_refused(nx, ny, nz):
    s = solver(nx, ny, nz)
    try:
        f = np.random.default_rng(1).standard_normal(s.shape) + 0j
        s.upload(hst.V1, f)
        for call in (hst.lib().hst_gpu_upload_field, hst.lib().hst_gpu_download_field):
            assert call(hst.V1, None) != 0
            assert "NULL" in hst.last_error()
        assert np.array_equal(s.download(hst.V1), f)
    finally:
        s.close()


def cpu_share(call):
    """The processors that a call keeps busy on average."""
    c, w = time.process_time(), time.perf_counter()
    call()
    c, w = time.process_time() - c, time.perf_counter() - w
    return c / w, w


def test_waiting_for_queued_steps_is_idle():
    """Steps queued, then a transfer that has to wait for them: of the copying
    threads none is busy meanwhile (the caller's own wait is)."""
    d = dataclasses.replace(read_input(deck_path("small")), nx=127, ny=257, nz=127)
    s = hst.Solver(d, hst.FP64)
    try:
        f = np.zeros(s.shape, dtype=np.complex128)
        s.download(hst.V1)
        s.timestep(1e-4)
        for call in (lambda: s.download(hst.V1), lambda: s.upload(hst.V1, f)):
            s.sync()
            for _ in range(120):
                s.timestep(1e-4)
            share, wall = cpu_share(call)
            assert wall > 0.1  # (the queue was not empty)
            assert share < 2.0
    finally:
        s.close()


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_pinned_arrays_go_straight(nx, ny, nz):
    """The caller's pinned arrays come back the same, at one processor's cost."""
    s = solver(nx, ny, nz)
    try:
        a = torch.randn(s.shape + (2,), dtype=torch.float64, pin_memory=True)
        b = torch.zeros(s.shape + (2,), dtype=torch.float64, pin_memory=True)
        up, down = hst.lib().hst_gpu_upload_field, hst.lib().hst_gpu_download_field

        def there_and_back():
            for _ in range(20):
                assert up(hst.V1, a.data_ptr()) == 0 and down(hst.V1, b.data_ptr()) == 0

        there_and_back()
        share, _ = cpu_share(there_and_back)
        assert torch.equal(a, b)
        assert share < 2.0
    finally:
        s.close()

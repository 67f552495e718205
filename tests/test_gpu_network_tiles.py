"""The network's kernels at the edges of their tiles (16 samples a wavefront,
64 a pass, 128 a training block) and the operand image they read, which is
written from given parameters and by every update.

Tolerance against the bfloat16-rounded oracle: FP32 sums in another order can
turn the rounding of an activation, 2^-8 of one operand (4e-3), the most that a
result of a single sample can move by in norm."""
import numpy as np
import pytest

from homogenenousshearturbulence_amd import closure
from test_gpu_closure import coarse_deck, norm_of, random_params, rel, synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 8191, 40001])
def test_forward(oracle_built, n):
    c = closure.Closure(coarse_deck(), 0)
    try:
        x, y = synthetic(max(n, 100), 1)
        nm, p = norm_of(x, y), random_params(2)
        c.set_params(p)
        c.set_norm(nm)
        got = c.predict(x[:n])
        want = oracle_built.mlp_forward(p, nm, x[:n], bf16=True) * nm[24:30] + nm[18:24]
        assert rel(got, want) < 4e-3
    finally:
        c.close()


@pytest.mark.parametrize("first,n", [(0, 1), (3, 16), (0, 63), (5, 64), (0, 65), (0, 127), (7, 128), (0, 129), (1, 4095)])
def test_gradient(oracle_built, first, n):
    c = closure.Closure(coarse_deck(), 4096)
    try:
        x, y = synthetic(4096, 3)
        c.set_dataset(x, y)
        nm = c.normalise()
        c.init_params(7)
        p = c.params()
        g, loss = c.grad(first, n)
        lo, go = oracle_built.mlp_grad(p, nm, x[first:first + n], y[first:first + n], bf16=True)
        assert rel(g, go) < 4e-3
        assert abs(loss - lo) < 4e-3 * lo
    finally:
        c.close()


def test_updates_keep_the_operands_in_step():
    """After training, the network that runs is the one of the parameters read back."""
    x, y = synthetic(4096, 9)
    a, b = closure.Closure(coarse_deck(), 4096), closure.Closure(coarse_deck(), 0)
    try:
        a.set_dataset(x, y)
        nm = a.normalise()
        a.init_params(3)
        before = a.predict(x)
        a.train(2, 1024, 1e-2, seed=4)
        b.set_norm(nm)
        b.set_params(a.params())
        got = a.predict(x)
        assert np.array_equal(got, b.predict(x))
        assert not np.array_equal(got, before)
    finally:
        a.close()
        b.close()

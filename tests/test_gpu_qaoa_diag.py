"""What a batched-QAOA handle finds out about its cost diagonals when it is made, wherever in them it lies: whether
C(x) = C(~x) for every x, which sends a state to the half-state kernels, and whether a phase may be too large for the
register kernels."""
import numpy as np
import pytest

import engines
import orkan_amd
from orkan_amd import batch
from test_gpu_qaoa import oracle_eval

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 9, 13, 14, 20])
def test_one_entry_breaks_the_symmetry(n):
    """A symmetric cost with one entry raised by 50, at the ends, the middle and between: taken for symmetric the mean
    would be off by far more than the bound of 1e-12 of the largest cost."""
    lib, orc = orkan_amd.load(5), engines.oracle(5)
    rng = np.random.default_rng(n)
    N = 1 << n
    base = rng.uniform(-3, 5, N)
    base = base + base[::-1]
    at = sorted({0, N // 2 - 1, N // 2, N - 1, int(rng.integers(N)), int(rng.integers(N))})
    diags = [base] + [base + 50.0 * (np.arange(N) == x) for x in at]
    gam, bet = [np.array([0.3])] * len(diags), [np.array([0.4])] * len(diags)
    b = batch.QaoaBatch(lib, [n] * len(diags), diags, max_evals=len(diags), max_p=1)
    got = b.eval(list(range(len(diags))), [1] * len(diags), gam, bet)
    b.close()
    for k, d in enumerate(diags):
        want = oracle_eval(orc, n, d, 1, gam[k], bet[k])
        assert abs(got[k] - want) <= 1e-12 * 64, (n, k, got[k], want)


@pytest.mark.parametrize("n", [1, 12, 13, 20])
@pytest.mark.parametrize("big", [np.inf, -np.inf, np.nan, 4e15])
def test_one_entry_beyond_the_register_kernels(n, big):
    """The bits of the LDS kernel, which takes such lists, wherever the entry lies."""
    lib = orkan_amd.load(5)
    rng = np.random.default_rng(n)
    N = 1 << n
    diags = []
    for x in sorted({0, N // 2, N - 1, int(rng.integers(N))}):
        diags.append(rng.uniform(0, 2, N))
        diags[-1][x] = big
    for d in diags:
        b = batch.QaoaBatch(lib, [n], [d], max_evals=1, max_p=2)
        args = ([0], [2], [np.array([0.7, 0.9])], [np.array([0.3, 1.1])])
        got = b.eval(*args)
        b.set_config(12, 512)
        assert np.array_equal(got, b.eval(*args), equal_nan=True)
        b.close()


@pytest.mark.parametrize("n", [5, 13, 16])
def test_phases_just_below_the_limit(n):
    """Phases of 2^49 to just below 2^50 in the register kernels, against the LDS kernels, whose sincos takes any argument:
    both phases are the same rounded product, off by 2^-52.6 at most, so that the means differ by rounding only.  Bound:
    (2 n + 8) p 2^-53 of max |C| for each side."""
    lib = orkan_amd.load(5)
    rng = np.random.default_rng(n)
    d = rng.uniform(0.5, 1.0, 1 << n)
    d[0] = 1.0
    g = [np.array([2.0 ** 49 * 1.5, np.nextafter(2.0 ** 50, 0.0)])]
    b = batch.QaoaBatch(lib, [n], [d], max_evals=1, max_p=2)
    args = ([0], [2], g, [np.array([0.3, 1.2])])
    got = b.eval(*args)[0]
    b.set_config(12, 512)
    want = b.eval(*args)[0]
    b.close()
    assert abs(got - want) <= 2 * (2 * n + 8) * 2 * 2.0 ** -53, (got, want)

"""Batched QAOA circuits deep enough for the scaled mixers to leave the number range: every rx runs without its scalar
factor, so that the squared norm grows by up to 2 per qubit and layer and, without a scaling on the way, overflows past
n p = 1024 (an infinite sum times a factor of 0)."""
import numpy as np
import pytest

import engines
import orkan_amd
from orkan_amd import batch
from test_gpu_qaoa import oracle_eval

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1200), (6, 200), (12, 100), (13, 90), (16, 70), (18, 50)]


@pytest.mark.parametrize("config", [None, (12, 512), (11, 256)])
@pytest.mark.parametrize("symmetric", [False, True])
def test_deep_circuits(config, symmetric):
    """One-tile and swept states, whole and half, and the LDS kernels, with mixers at, around and away from pi / 4 (the
    largest growth), against the oracle.  Bound: each layer multiplies every amplitude 2 n + 4 times, on both sides, with
    an error of 2^-53 each, of a mean of at most max |C|: 4 (2 n + 4) p 2^-53 max |C|.  Shallow circuits of the same
    list keep the bits they have in a list of their own."""
    lib, orc = orkan_amd.load(5), engines.oracle(5)
    rng = np.random.default_rng(768 + symmetric)
    ns, ps, diags, gam, bet = [], [], [], [], []
    for n, p in SHAPES:
        for spread in (0.0, 0.1, 1.5):
            d = rng.uniform(-3, 5, 1 << n)
            ns.append(n)
            ps.append(p)
            diags.append(d + d[::-1] if symmetric else d)
            gam.append(rng.uniform(0, np.pi, p))
            bet.append(np.pi / 4 + spread * rng.uniform(-1, 1, p))
    deep = len(ns)
    for n in (5, 12, 15):
        d = rng.uniform(-3, 5, 1 << n)
        ns.append(n)
        ps.append(3)
        diags.append(d + d[::-1] if symmetric else d)
        gam.append(rng.uniform(0, np.pi, 3))
        bet.append(rng.uniform(0, np.pi, 3))
    b = batch.QaoaBatch(lib, ns, diags, max_evals=len(ns), max_p=max(ps))
    if config:
        b.set_config(*config)
    got = b.eval(list(range(len(ns))), ps, gam, bet)
    alone = b.eval(list(range(deep, len(ns))), ps[deep:], gam[deep:], bet[deep:])
    b.close()
    assert np.array_equal(got[deep:], alone)
    for k in range(deep):
        n, p = ns[k], ps[k]
        want = oracle_eval(orc, n, diags[k], p, gam[k], bet[k])
        bound = 4 * (2 * n + 4) * p * 2.0 ** -53 * np.abs(diags[k]).max()
        assert abs(got[k] - want) <= bound, (n, p, got[k], want, bound)

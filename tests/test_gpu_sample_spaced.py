"""sample_matrix on vectors long enough to be held 64 amplitudes further apart than their length, and in workspaces whose
scratch takes the leaves in several batches, against every leaf built in numpy; all workspaces give the same bits."""
import ctypes as C

import numpy as np
import pytest

import orkan_amd
from linalg_np import PURE, mat1, random_psi
from orkan_amd import _ffi

pytestmark = pytest.mark.gpu


def _apply(psi, name, q, th):
    v = psi.reshape(-1, 2, 1 << q)
    return np.einsum("ab,ibj->iaj", mat1(name, th), v).reshape(-1)


@pytest.mark.parametrize("n", [11, 12, 14])
@pytest.mark.parametrize("K,others", [(2, (2,)), (17, (3, 2)), (65, (2,)), (70, (3,))])
def test_spaced_vectors(n, K, others):
    """Lengths beside and beyond 2^12, from which the vectors are spaced; one to three operations per combination; more
    leaves than a block of 64.  Workspaces: four vectors (leaves one by one, no spacing), blocks of some leaves with
    scratch for fewer, just too small and just large enough for the spacing of everything, and ample.  Bound as for the
    shorter vectors: 1e-12 of the largest entry."""
    lib = orkan_amd.load(5)
    rng = np.random.default_rng(100 * n + K)
    sizes = [2, K] + list(others)
    table, keep, chans = [], [], []
    for m in sizes:
        specs = [(["rx", "ry", "rz"][int(rng.integers(3))], int(rng.integers(n)), float(rng.uniform(0, 6))) for _ in range(m)]
        cbs = [_ffi.QOP(lambda st, f=getattr(lib, s), q=q, th=th: f(st, q, th)) for s, q, th in specs]
        w = np.ascontiguousarray((rng.standard_normal(m) + 1j * rng.standard_normal(m)) / np.sqrt(m))
        arr = (_ffi.QOP * m)(*cbs)
        keep += [cbs, arr, w]
        table.append(_ffi.AnsatzChannelT(m, arr, w.ctypes.data))
        chans.append((specs, w))
    tab = (_ffi.AnsatzChannelT * len(table))(*table)
    psi0, obs = random_psi(n, rng), rng.uniform(-1, 1, 1 << n)

    def combine(psi, c):
        return sum(w * _apply(psi, *s) for s, w in zip(*c))

    prefix = combine(psi0, chans[0])
    leaves = []
    for s in chans[1][0]:
        v = _apply(prefix, *s)
        for c in chans[2:]:
            v = combine(v, c)
        leaves.append(v)
    M = np.array(leaves)
    want = (M.conj() * obs) @ M.T
    vec, spaced = 16 << n, (16 << n) + 1024
    B = min(K, 64)
    held = (B if B == K else 2 * B) + 2 * B
    got = []
    for budget in (4 * vec, 9 * vec, 13 * spaced, (2 * B + 5) * vec, (2 * B + 5) * spaced, held * spaced - 1, held * spaced,
                   1 << 30):
        st = _ffi.StateT(PURE, None, 0)
        lib.state_init(C.byref(st), n, None)
        assert lib.orkan_state_upload(C.byref(st), psi0.ctypes.data) == 0
        S = np.zeros((K, K), np.complex128)
        assert lib.sample_matrix(C.byref(st), obs.ctypes.data, tab, len(sizes), 1, budget, S.ctypes.data) == 0
        after = np.empty(1 << n, np.complex128)
        assert lib.orkan_state_download(C.byref(st), after.ctypes.data) == 0
        lib.state_free(C.byref(st))
        assert np.abs(after - prefix).max() <= 1e-12
        got.append(S.T.copy())
    assert np.abs(got[0] - want).max() <= 1e-12 * max(1.0, np.abs(want).max())
    assert all(np.array_equal(g, got[0]) for g in got[1:])

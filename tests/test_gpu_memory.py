"""State storage is kept for the next state of nearly the same size: a reused block never shows through (a new state
reads zeros, a copy, a conversion and a |+> state exactly their own values, the padding of a small tile included),
live states never share storage, and a caller's own device buffer is adopted and released as before.  Moves and fills
are exact, so every comparison is for equality."""
import ctypes as C
import threading

import numpy as np
import pytest

import orkan_amd
from linalg_np import random_rho, to_layout
from orkan_amd._ffi import MIXED_PACKED, MIXED_TILED, PURE, StateT

pytestmark = pytest.mark.gpu


def _read(lib, st, dtype=np.complex128):
    out = np.empty(lib.state_len(C.byref(st)), dtype)
    assert lib.orkan_state_download(C.byref(st), out.ctypes.data) == 0
    return out


def _dirty(lib, kind, n):
    """leaves a block of this size full of values behind"""
    st = StateT(kind, None, 0)
    lib.state_init(C.byref(st), n, None)
    junk = np.full(lib.state_len(C.byref(st)), 7.5 - 3j, np.complex64 if kind & orkan_amd.ORKAN_FP32 else np.complex128)
    assert lib.orkan_state_upload(C.byref(st), junk.ctypes.data) == 0
    lib.state_free(C.byref(st))
    assert not st.data


@pytest.mark.parametrize("kind", [PURE, MIXED_PACKED, MIXED_TILED])
@pytest.mark.parametrize("n", [1, 3, 5, 8])
def test_reused_blocks_do_not_show(kind, n):
    lib = orkan_amd.load(5)
    D = 1 << n
    _dirty(lib, kind, n)
    st = StateT(kind, None, 0)
    lib.state_init(C.byref(st), n, None)
    assert not _read(lib, st).any()
    _dirty(lib, kind, n)
    lib.state_plus(C.byref(st), n)
    got = _read(lib, st)
    if kind == MIXED_TILED and n < 5:
        want = np.zeros((32, 32), complex)
        want[:D, :D] = 1.0 / D
        want = want.reshape(-1)
    else:
        want = np.full(got.size, 1.0 / np.sqrt(D) if kind == PURE else 1.0 / D, complex)
    assert np.array_equal(got, want)
    _dirty(lib, kind, n)
    cp = lib.state_cp(C.byref(st))
    assert cp.data != st.data and np.array_equal(_read(lib, cp), want)
    _dirty(lib, kind | orkan_amd.ORKAN_FP32, n)
    half = lib.orkan_state_convert(C.byref(st), 1)
    assert np.array_equal(_read(lib, half, np.complex64), want.astype(np.complex64))
    for s in (st, cp, half):
        lib.state_free(C.byref(s))


@pytest.mark.parametrize("n", [2, 5, 7])
def test_relayout_into_a_reused_block(n):
    lib = orkan_amd.load(5)
    rho = random_rho(n, np.random.default_rng(n))
    st = StateT(MIXED_PACKED, None, 0)
    lib.state_init(C.byref(st), n, None)
    assert lib.orkan_state_upload(C.byref(st), to_layout(rho, MIXED_PACKED, 5).ctypes.data) == 0
    low = np.tril(rho)
    full = low + np.tril(rho, -1).conj().T
    for layout in (MIXED_TILED, MIXED_PACKED):
        _dirty(lib, layout, n)
        out = StateT()
        assert lib.orkan_state_relayout(C.byref(st), C.byref(out), layout) == 0
        assert np.array_equal(_read(lib, out), to_layout(full, layout, 5))
        lib.state_free(C.byref(out))
    lib.state_free(C.byref(st))


def test_adopted_buffers_and_moved_pointers():
    lib = orkan_amd.load(5)
    buf = lib.orkan_dev_alloc(2 << 6)
    p = C.c_void_p(buf)
    st = StateT(PURE, None, 0)
    lib.state_init(C.byref(st), 6, C.byref(p))
    assert st.data == buf and not p.value
    lib.state_free(C.byref(st))
    # a state's storage handed to another state
    a, b = StateT(PURE, None, 0), StateT(PURE, None, 0)
    lib.state_plus(C.byref(a), 6)
    p = C.c_void_p(a.data)
    lib.state_init(C.byref(b), 6, C.byref(p))
    assert np.array_equal(_read(lib, b), np.full(64, 0.125, complex))
    lib.state_free(C.byref(b))
    # ... or released as a device array
    lib.state_plus(C.byref(b), 6)
    lib.orkan_dev_free(b.data)
    b.data = None
    lib.state_plus(C.byref(b), 6)
    assert np.array_equal(_read(lib, b), np.full(64, 0.125, complex))
    lib.state_free(C.byref(b))


def test_live_states_never_share_storage():
    lib = orkan_amd.load(5)
    errors = []

    def work(k):
        try:
            for r in range(20):
                states = []
                for j in range(4):
                    s = StateT(PURE, None, 0)
                    lib.state_plus(C.byref(s), 6 + (k + j) % 3)
                    lib.x(C.byref(s), 0)
                    lib.p(C.byref(s), 1, 0.1 * (k + 1) + j)
                    states.append((s, j))
                for s, j in states:
                    got = _read(lib, s)
                    want = np.full(got.size, 1.0 / np.sqrt(got.size), complex)
                    want[(np.arange(got.size) >> 1) & 1 == 1] *= np.exp(1j * (0.1 * (k + 1) + j))
                    # one product of a unit phase: 2 rounding errors of 2^-53 on values <= 1
                    assert np.abs(got - want).max() <= 4 * 2.0 ** -53
                for s, _ in states:
                    lib.state_free(C.byref(s))
        except AssertionError as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not errors and not any(t.is_alive() for t in threads)

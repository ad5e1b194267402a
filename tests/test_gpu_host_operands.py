"""Operands in host memory are read as work already on the library's stream leaves them: a pinned buffer that a copy on
the stream is still filling holds the operand only when that copy has run."""
import ctypes as C

import numpy as np
import pytest

import engines
import known_answers as ka
import orkan_amd
from linalg_np import MIXED_TILED, random_rho, superop, to_layout
from orkan_amd import _ffi

pytestmark = pytest.mark.gpu

DEVICE_TO_HOST = 2


@pytest.mark.parametrize("n", [3, 6])
def test_superoperator_written_by_the_stream(n):
    """channel_2q with a pinned superoperator: milliseconds of queued gates and a device-to-host copy lie between the call
    and the values it must use.  Against the oracle, 1e-12 per stored entry as in every parity test."""
    dev, orc = engines.DeviceEngine(orkan_amd.lib_path(5), 5), engines.oracle(5)
    hip = dev.api.lib     # symbols of the HIP runtime the library is linked with
    hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    hip.hipHostFree.argtypes = [C.c_void_p]
    hip.hipMemcpyAsync.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int, C.c_void_p]
    rng = np.random.default_rng(n)
    old, new = (np.ascontiguousarray(superop(ka.kraus_2q_sets(rng)[2])).reshape(256) for _ in range(2))
    pin, src = C.c_void_p(), dev.api.orkan_dev_alloc(512)
    assert hip.hipHostMalloc(C.byref(pin), 4096, 0) == 0
    assert np.abs(old - new).max() > 0.01
    C.memmove(pin, old.ctypes.data, 4096)
    assert dev.api.orkan_copy_to_device(src, new.ctypes.data, 4096) == 0
    data = to_layout(random_rho(n, rng), MIXED_TILED, 5)
    sd, so = dev.new(MIXED_TILED, n, data), orc.new(MIXED_TILED, n, data)
    busy = dev.plus(MIXED_TILED, 13)
    assert dev.api.orkan_sync() == 0
    for _ in range(100):
        dev.gate(busy, "h", 3)
    assert hip.hipMemcpyAsync(pin, src, 4096, DEVICE_TO_HOST, dev.api.orkan_stream()) == 0
    s = _ffi.SuperopT(2, pin.value)
    dev.api.channel_2q(C.byref(sd), C.byref(s), 0, n - 1)
    orc.channel2(so, new, 0, n - 1)
    assert np.abs(dev.read(sd) - orc.read(so)).max() <= 1e-12
    for e, st in ((dev, sd), (dev, busy), (orc, so)):
        e.free(st)
    dev.api.orkan_dev_free(src)
    assert hip.hipHostFree(pin) == 0


@pytest.mark.parametrize("nonzero", [0, 1, 127, 128, 129, 255, 256])
def test_superoperators_of_every_density(nonzero):
    """Host superoperators travel by their nonzero entries, 128 to a launch: counts at and beside that, with a zero of
    either sign among them.  1e-12 per stored entry, as in every parity test."""
    dev, orc = engines.DeviceEngine(orkan_amd.lib_path(5), 5), engines.oracle(5)
    rng = np.random.default_rng(nonzero)
    # maps of Hermitian matrices to Hermitian ones: S[ij,kl] = conj(S[ji,lk]); entries of i = j, k = l are their own partners
    i, j, k, l = np.unravel_index(rng.permutation(256), (4, 4, 4, 4))
    at, partner = (i * 4 + j) * 16 + k * 4 + l, (j * 4 + i) * 16 + l * 4 + k
    S = np.full(256, -0.0 if nonzero == 129 else 0.0, np.complex128)
    singles, pairs = at[at == partner], [(a, b) for a, b in zip(at, partner) if a < b]
    own = nonzero % 2 if nonzero <= 240 else nonzero - 240
    S[singles[:own]] = rng.standard_normal(own) / 16
    for a, b in pairs[:(nonzero - own) // 2]:
        S[a] = (rng.standard_normal() + 1j * rng.standard_normal()) / 16
        S[b] = np.conj(S[a])
    assert np.count_nonzero(S) == nonzero
    full = np.full(256, 0.25 + 0.0j)
    for n in (2, 5):
        data = to_layout(random_rho(n, rng), MIXED_TILED, 5)
        sd, so = dev.new(MIXED_TILED, n, data), orc.new(MIXED_TILED, n, data)
        for T in (full, S):      # the entries of an earlier one must not stay
            dev.channel2(sd, T, 0, n - 1)
            orc.channel2(so, T, 0, n - 1)
        assert np.abs(dev.read(sd) - orc.read(so)).max() <= 1e-12
        dev.free(sd)
        orc.free(so)

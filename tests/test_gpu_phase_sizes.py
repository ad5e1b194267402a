"""Diagonal gates and exp_diag on density matrices below and above the size from which a thread takes several entries (10
and 11 qubits), and on the smallest ones, against the oracle; and the packed superoperator kernel's mirror entries at the
same sizes."""
import ctypes as C

import numpy as np
import pytest

import engines
import orkan_amd
from linalg_np import MIXED_PACKED, MIXED_TILED, to_layout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [MIXED_PACKED, MIXED_TILED])
@pytest.mark.parametrize("n", [2, 5, 9, 10, 11])
def test_phases_against_the_oracle(kind, n):
    dev, orc = engines.DeviceEngine(orkan_amd.lib_path(5), 5), engines.oracle(5)
    rng = np.random.default_rng(40 + n)
    a = rng.standard_normal((1 << n, 2)) + 1j * rng.standard_normal((1 << n, 2))
    a /= np.linalg.norm(a)
    data = to_layout(a @ a.conj().T, kind, 5)
    diag = rng.uniform(-2, 2, 1 << n)
    sd, so = dev.new(kind, n, data), orc.new(kind, n, data)
    half = dev.api.orkan_state_convert(C.byref(sd), 1)
    for e, st in ((dev, sd), (orc, so), (dev, half)):
        e.gate(st, "cz", 0, n - 1)
        e.gate(st, "t", n // 2)
        e.exp_diag(st, diag, 0.7)
        e.gate(st, "h", n - 1)
    want = orc.read(so)
    assert np.abs(dev.read(sd) - want).max() <= 1e-12
    got = np.empty(want.size, np.complex64)
    assert dev.api.orkan_state_download(C.byref(half), got.ctypes.data) == 0
    # entries of modulus <= 1 rounded to complex64 at the start and by four updates, h doubling what came before at most
    assert np.abs(got - want).max() <= 9 * 2.0 ** -24
    for e, st in ((dev, sd), (orc, so), (dev, half)):
        e.free(st)

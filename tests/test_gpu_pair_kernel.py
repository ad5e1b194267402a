"""Two-qubit superoperators and unitaries on density matrices of 5 qubits and more (one wave per 32 x 32 group) against
the oracle, on every ordered qubit pair, both layouts, both tile sizes and both precisions; and the same bits with
streaming accesses as without."""
import ctypes as C

import numpy as np
import pytest

import engines
import known_answers as ka
import orkan_amd
from linalg_np import MIXED_PACKED, MIXED_TILED, random_rho, superop, to_layout

pytestmark = pytest.mark.gpu
TOL = 1e-12          # per stored entry, as in every parity test
# complex64: an update rounds each stored entry once, 2^-24 of an entry of modulus <= 1; entries below cover the sum of
# the updates of one pair each
TOL32 = 2.0 ** -23


def _unitary(rng):
    return np.linalg.qr(rng.standard_normal((4, 4)) + 1j * rng.standard_normal((4, 4)))[0]


@pytest.mark.parametrize("log_tile", [5, 3])
@pytest.mark.parametrize("kind", [MIXED_PACKED, MIXED_TILED])
@pytest.mark.parametrize("n", [5, 6, 8])
def test_every_pair_against_the_oracle(kind, n, log_tile):
    dev, orc = engines.DeviceEngine(orkan_amd.lib_path(log_tile), log_tile), engines.oracle(log_tile)
    rng = np.random.default_rng(100 * n + kind)
    S = superop(ka.kraus_2q_sets(rng)[0])
    data = to_layout(random_rho(n, rng), kind, log_tile)
    for q1 in range(n):
        for q2 in range(n):
            if q1 == q2:
                continue
            m = np.ascontiguousarray(_unitary(rng).T.reshape(-1))
            sd, so = dev.new(kind, n, data), orc.new(kind, n, data)
            half = dev.api.orkan_state_convert(C.byref(sd), 1)
            for e, st in ((dev, sd), (orc, so)):
                e.channel2(st, S, q1, q2)
                e.api.two_from_mat(C.byref(st), q1, q2, m.ctypes.data)
            dev.channel2(half, S, q1, q2)
            dev.api.two_from_mat(C.byref(half), q1, q2, m.ctypes.data)
            want = orc.read(so)
            assert np.abs(dev.read(sd) - want).max() <= TOL, (q1, q2)
            got = np.empty(want.size, np.complex64)
            assert dev.api.orkan_state_download(C.byref(half), got.ctypes.data) == 0
            # the start rounded once, then two updates: three roundings
            assert np.abs(got - want).max() <= 3 * TOL32, (q1, q2)
            for e, st in ((dev, sd), (orc, so), (dev, half)):
                e.free(st)


def test_streaming_accesses_change_no_value():
    dev = engines.DeviceEngine(orkan_amd.lib_path(5), 5)
    rng = np.random.default_rng(5)
    n = 8
    S = superop(ka.kraus_2q_sets(rng)[0])
    m = np.ascontiguousarray(_unitary(rng).T.reshape(-1))
    data = to_layout(random_rho(n, rng), MIXED_TILED, 5)
    out = []
    for least in (0, 1):     # smallest state that streams: the default, one byte
        assert dev.api.orkan_set_launch_shape(13, 0, least) == 0
        st = dev.new(MIXED_TILED, n, data)
        for q1, q2 in ((0, 1), (4, 2), (3, 6), (7, 0), (5, 7)):
            dev.channel2(st, S, q1, q2)
            dev.api.two_from_mat(C.byref(st), q1, q2, m.ctypes.data)
        out.append(dev.read(st))
        dev.free(st)
    assert dev.api.orkan_set_launch_shape(14, 0, 0) == 0
    assert np.array_equal(out[0], out[1])

"""The surrogate's GEMM tiles (128 x 64 up to one per CU, 128 x 128, 256 x 256) on both sides of the lines between them:
every tile multiplies in the same order, so predictions and gradients have the same bits whichever is chosen, also the
transposed copies that the weight gradients read; and batches of more rows than one slice of those against the oracle."""
import ctypes as C

import numpy as np
import pytest

import orkan_amd
from orkan_amd import surrogate
from oracle import mlp_np

pytestmark = pytest.mark.gpu


def _net(lib, rng, hidden, layers, rows):
    W, b, wo, _ = mlp_np.init_params(rng, 128, hidden, layers)
    W, wo = [w.astype(np.float32) for w in W], wo.astype(np.float32)
    b = [(0.1 * rng.standard_normal(hidden)).astype(np.float32) for _ in b]
    m = surrogate.Mlp(lib, hidden=hidden, layers=layers, max_batch=rows)
    m.set_weights(W, b, wo, 0.25)
    return m, (W, b, wo, 0.25)


@pytest.mark.parametrize("hidden,layers,rows", [
    (512, 3, 4096), (512, 3, 4097), (128, 2, 16384), (128, 2, 16385), (384, 2, 5376), (384, 2, 5400), (512, 2, 32640),
    (512, 2, 32768), (1024, 2, 16384)])
def test_every_tile_gives_the_same_bits(hidden, layers, rows):
    lib = orkan_amd.load(5)
    rng = np.random.default_rng(rows + hidden)
    m, _ = _net(lib, rng, hidden, layers, rows)
    x = rng.standard_normal((rows, 128)).astype(np.float32)
    t = rng.standard_normal(rows).astype(np.float32)
    res = []
    try:
        for variant in (2, 0, 1):     # the rule, 128 x 128 throughout, 256 x 256 staged through registers where it divides
            assert lib.orkan_set_launch_shape(11, variant, 0) == 0
            y = m.forward(x)
            loss, (dW, db, dwo, dbo) = m.grads(x, t)
            res.append([y, np.float32(loss), np.float32(dbo), dwo, *dW, *db])
    finally:
        assert lib.orkan_set_launch_shape(14, 0, 0) == 0
    for other in res[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(res[0], other))
    m.close()


@pytest.mark.parametrize("rows,hidden", [(1300, 256), (2176, 128), (4224, 512)])
def test_gradients_of_many_rows(rows, hidden):
    """Bounds as in test_gradients_at_tile_edges: bf16 rounding of activations and gradients (2^-9 per value)."""
    lib = orkan_amd.load(5)
    rng = np.random.default_rng(rows)
    m, (W, b, wo, bo) = _net(lib, rng, hidden, 3, rows)
    x = rng.standard_normal((rows, 128)).astype(np.float32)
    t = rng.standard_normal(rows).astype(np.float32)
    params = ([w.astype(np.float64) for w in W], [v.astype(np.float64) for v in b], wo.astype(np.float64), bo)
    loss, (dW, db, dwo, dbo) = m.grads(x, t)
    lref, (rW, rb, rwo, rbo) = mlp_np.loss_and_grads(params, x.astype(np.float64), t.astype(np.float64), exact=False)
    assert abs(loss - lref) <= 1e-2 * lref
    for l in range(3):
        assert np.linalg.norm(dW[l] - rW[l]) <= 2e-2 * np.linalg.norm(rW[l]), l
        assert np.linalg.norm(db[l] - rb[l]) <= 2e-2 * np.linalg.norm(rb[l]), l
    assert np.linalg.norm(dwo - rwo) <= 2e-2 * np.linalg.norm(rwo)
    assert abs(dbo - rbo) <= 1e-2 * max(1.0, abs(rbo))
    m.close()


@pytest.mark.parametrize("hidden,layers", [(128, 1), (128, 4), (256, 3), (512, 3)])
@pytest.mark.parametrize("ncand", [1, 64, 1000])
def test_screening_in_one_kernel_and_layer_by_layer(hidden, layers, ncand):
    """8 angles run through one kernel, 9 layer by layer: with the last graph feature handed over as the first angle the
    two compute the same values, and in the same order."""
    lib = orkan_amd.load(5)
    rng = np.random.default_rng(hidden + layers + ncand)
    m, _ = _net(lib, rng, hidden, layers, 256)
    gf = rng.uniform(0, 1, 120).astype(np.float32)
    ang = rng.uniform(0, 1, (ncand, 8)).astype(np.float32)
    nine = np.ascontiguousarray(np.concatenate([np.full((ncand, 1), gf[119], np.float32), ang], 1))
    out = []
    for g, a in ((gf, ang), (gf[:119], nine)):
        da, dy = lib.orkan_dev_alloc((a.size + 1) // 2), lib.orkan_dev_alloc((ncand + 1) // 2)
        assert lib.orkan_copy_to_device(da, a.ctypes.data, a.nbytes) == 0
        m.forward_candidates(g, da, ncand, dy)
        y = np.empty(ncand, np.float32)
        assert lib.orkan_copy_to_host(y.ctypes.data, dy, y.nbytes) == 0
        out.append(y)
        lib.orkan_dev_free(da)
        lib.orkan_dev_free(dy)
    assert np.array_equal(out[0], out[1])
    m.close()


def test_weights_set_after_a_diverged_step():
    """set_weights stores what it is given, also where a batch has left the weights and Adam's moments without values."""
    lib = orkan_amd.load(5)
    rng = np.random.default_rng(3)
    m, (W, b, wo, bo) = _net(lib, rng, 128, 2, 128)
    x = rng.standard_normal((100, 128)).astype(np.float32)
    y = m.forward(x)
    m.train_step(np.full((100, 128), np.nan, np.float32), np.zeros(100, np.float32), 1e-3)
    assert np.isnan(m.get_weights()[0][0]).all()
    m.set_weights(W, b, wo, bo)
    got = m.get_weights()
    assert all(np.array_equal(a, c) for a, c in zip(got[0] + got[1], W + b)) and np.array_equal(got[2], wo)
    assert np.array_equal(m.forward(x), y)
    m.close()


@pytest.mark.parametrize("n,k", [(40, 31), (40, 33), (300, 65), (70000, 65536)])
def test_topk_order(n, k):
    """Beside the sorting runs of 32, and the largest k: values descending, ties by index, zeros of either sign alike."""
    lib = orkan_amd.load(5)
    rng = np.random.default_rng(k)
    y = rng.integers(-50, 50, n).astype(np.float32) / 8
    y[rng.integers(0, n, n // 10)] = -0.0
    y[: n // 3] += rng.standard_normal(n // 3).astype(np.float32)
    dev = lib.orkan_dev_alloc((n + 1) // 2)
    assert lib.orkan_copy_to_device(dev, y.ctypes.data, y.nbytes) == 0
    idx, val = np.empty(k, np.int32), np.empty(k, np.float32)
    assert lib.orkan_topk_f32(dev, n, k, idx.ctypes.data_as(C.POINTER(C.c_int)), val.ctypes.data_as(surrogate.FP)) == 0
    lib.orkan_dev_free(dev)
    want = np.lexsort((np.arange(n), -y))[:k]
    assert np.array_equal(val, y[want]) and np.array_equal(y[idx], val)
    tie = np.flatnonzero(val[1:] == val[:-1])
    assert np.all(idx[tie] < idx[tie + 1]) and len(set(idx.tolist())) == k

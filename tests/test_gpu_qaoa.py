"""Batched QAOA launcher against per-instance runs of the reference call
sequence on the CPU oracle (state_plus, exp_diag, rx(q, 2 beta), mean) at
1e-12, plus the device-side MaxCut diagonal against numpy."""
import numpy as np
import pytest

import engines
import orkan_amd
from linalg_np import PURE
from orkan_amd import batch

pytestmark = pytest.mark.gpu


def oracle_eval(orc, n, diag, p, gamma, beta):
    st = orc.plus(PURE, n)
    for l in range(p):
        orc.exp_diag(st, diag, gamma[l])
        for q in range(n):
            orc.gate(st, "rx", q, 2 * beta[l])
    m = orc.mean(st, diag)
    orc.free(st)
    return m


@pytest.mark.parametrize("config", [None, (11, 256), (12, 1024), (13, 512)])
def test_batch_matches_per_instance_runs(config):
    lib = orkan_amd.load(5)
    orc = engines.oracle(5)
    rng = np.random.default_rng(44)
    inst = batch.maxcut_instances(48, rng, n_lo=2, n_hi=18)
    diags = [batch.maxcut_diag(i["n"], i["edges"], i["w"]) for i in inst]
    b = batch.QaoaBatch(lib, [i["n"] for i in inst], diags, max_evals=64, max_p=8)
    if config:
        b.set_config(*config)
    got = b.eval(list(range(len(inst))), [i["p"] for i in inst], [i["gamma"] for i in inst],
                 [i["beta"] for i in inst])
    for k, i in enumerate(inst):
        want = oracle_eval(orc, i["n"], diags[k], i["p"], i["gamma"], i["beta"])
        assert abs(got[k] - want) <= 1e-12, (k, i["n"], i["p"], got[k], want)
    # repeated launches of the captured graph give identical results
    again = b.eval(list(range(len(inst))), [i["p"] for i in inst], [i["gamma"] for i in inst],
                   [i["beta"] for i in inst])
    assert np.array_equal(got, again)
    b.close()


def test_device_maxcut_diag():
    lib = orkan_amd.load(5)
    rng = np.random.default_rng(3)
    for n in (3, 11, 17):
        i = batch.maxcut_instances(1, rng, n_lo=n, n_hi=n)[0]
        out = lib.orkan_dev_alloc(1 << n)
        e = np.ascontiguousarray(i["edges"])
        ei = np.ascontiguousarray(e[:, 0]); ej = np.ascontiguousarray(e[:, 1])
        w = np.ascontiguousarray(i["w"])
        rc = lib.orkan_maxcut_diag_dev(n, len(w), ei.ctypes.data_as(batch.IP), ej.ctypes.data_as(batch.IP),
                                       w.ctypes.data_as(batch.DP), out)
        assert rc == 0
        host = np.empty(1 << n)
        assert lib.orkan_copy_to_host(host.ctypes.data, out, host.nbytes) == 0
        assert np.abs(host - batch.maxcut_diag(n, i["edges"], i["w"])).max() <= 1e-12
        lib.orkan_dev_free(out)


def test_autotuner_picks_a_valid_config():
    lib = orkan_amd.load(5)
    rng = np.random.default_rng(5)
    inst = batch.maxcut_instances(32, rng, n_lo=10, n_hi=16)
    diags = [batch.maxcut_diag(i["n"], i["edges"], i["w"]) for i in inst]
    b = batch.QaoaBatch(lib, [i["n"] for i in inst], diags, max_evals=32, max_p=8)
    args = (list(range(len(inst))), [i["p"] for i in inst], [i["gamma"] for i in inst], [i["beta"] for i in inst])
    ref = b.eval(*args)
    ms, cfg = b.autotune(*args, reps=2)
    assert ms > 0 and cfg["lt"] in (11, 12, 13)
    assert np.abs(b.eval(*args) - ref).max() <= 1e-12
    b.close()


def test_largest_states_n19_n20():
    """States of 19 and 20 qubits (the top of the 10..20 range of the 4096-instance workload) stream
    through HBM in p + 1 LDS-tiled sweeps; each against its per-instance oracle run."""
    lib = orkan_amd.load(5)
    orc = engines.oracle(5)
    rng = np.random.default_rng(1920)
    inst = batch.maxcut_instances(6, rng, n_lo=19, n_hi=20)
    diags = [batch.maxcut_diag(i["n"], i["edges"], i["w"]) for i in inst]
    b = batch.QaoaBatch(lib, [i["n"] for i in inst], diags, max_evals=8, max_p=8)
    got = b.eval(list(range(len(inst))), [i["p"] for i in inst], [i["gamma"] for i in inst],
                 [i["beta"] for i in inst])
    for k, i in enumerate(inst):
        print(f"n {i['n']} p {i['p']}", flush=True)
        want = oracle_eval(orc, i["n"], diags[k], i["p"], i["gamma"], i["beta"])
        assert abs(got[k] - want) <= 1e-12, (k, i["n"], i["p"], got[k], want)
    b.close()


def test_full_4096_batch_sample():
    """The 4096-instance workload itself (cost diagonals built on the device), autotuned, one
    launch; a seeded sample of its evaluations, always including the largest states, against
    per-instance oracle runs at 1e-12."""
    from benchmarks import qaoa as bq
    lib = orkan_amd.load(5)
    orc = engines.oracle(5)
    inst = bq.make(4096)
    dptrs = bq.device_diags(lib, inst)
    b = batch.QaoaBatch(lib, [i["n"] for i in inst], dptrs, max_evals=len(inst), max_p=8)
    for p in dptrs:
        lib.orkan_dev_free(p)
    args = (list(range(len(inst))), [i["p"] for i in inst], [i["gamma"] for i in inst], [i["beta"] for i in inst])
    _, cfg = b.autotune(*args, reps=1)
    print(f"autotuned {cfg}", flush=True)
    got = b.eval(*args)
    b.close()
    order = np.argsort([-(i["n"] * 8 + i["p"]) for i in inst], kind="stable")
    sample = list(order[:4]) + list(np.random.default_rng(4096).choice(len(inst), 20, replace=False))
    for k in sample:
        i = inst[k]
        want = oracle_eval(orc, i["n"], batch.maxcut_diag(i["n"], i["edges"], i["w"]), i["p"], i["gamma"], i["beta"])
        assert abs(got[k] - want) <= 1e-12, (k, i["n"], i["p"], got[k], want)


@pytest.mark.parametrize("lo,hi", [(1, 8), (9, 13), (14, 17), (18, 20), (21, 22)])
@pytest.mark.parametrize("flips", [False, True])
def test_register_tiles(lo, hi, flips):
    """The register kernel at every qubit count of its range: states of one tile, with and without empty registers, and
    every split of the tile bits between contiguous and gathered tiles; 1 to 4 layers (both layouts a one-tile state may
    end in), mixers of |cos| >= |sin| only and of both forms (where the cost diagonal is read complemented)."""
    lib = orkan_amd.load(5)
    orc = engines.oracle(5)
    rng = np.random.default_rng(lo + flips)
    ns, ps = [], []
    for n in range(lo, hi + 1):
        for p in ((1, 2, 3, 4) if n < 18 else (2, 3) if n < 21 else (2,)):
            ns.append(n)
            ps.append(p)
    diags = [rng.uniform(-3, 5, 1 << n) for n in ns]
    gam = [rng.uniform(0, np.pi, p) for p in ps]
    bet = [rng.uniform(0, np.pi, p) if flips else rng.uniform(-0.7, 0.7, p) for p in ps]
    b = batch.QaoaBatch(lib, ns, diags, max_evals=len(ns), max_p=4)
    assert b.config()["lt"] == 12 and b.config()["threads"] == 256
    got = b.eval(list(range(len(ns))), ps, gam, bet)
    assert np.array_equal(got, b.eval(list(range(len(ns))), ps, gam, bet))
    for k, n in enumerate(ns):
        want = oracle_eval(orc, n, diags[k], ps[k], gam[k], bet[k])
        assert abs(got[k] - want) <= 1e-12, (n, ps[k], got[k], want)
    b.close()


@pytest.mark.parametrize("lo,hi", [(1, 8), (9, 13), (14, 17), (18, 20), (21, 24)])
def test_flip_symmetric_costs(lo, hi):
    """Costs with C(x) = C(~x) run on half of the state: every qubit count of the range (one tile up to 13 qubits, every
    place of the bit that the gathered tiles share with the contiguous ones), mixers of both forms, in one list with a
    cost of each size whose last bit differs in one entry and which must take the general kernels."""
    lib = orkan_amd.load(5)
    orc = engines.oracle(5)
    rng = np.random.default_rng(70 + lo)
    ns, ps, diags = [], [], []
    for n in range(lo, hi + 1):
        for p in ((1, 2, 3, 4) if n < 18 else (2, 3) if n < 21 else (2,)):
            d = rng.uniform(-3, 5, 1 << n)
            ns.append(n)
            ps.append(p)
            diags.append(d + d[::-1])
        if n < 21:
            d = diags[-1].copy()
            d[0] = np.nextafter(d[0], 9.0)
            ns.append(n)
            ps.append(2)
            diags.append(d)
    gam = [rng.uniform(0, np.pi, p) for p in ps]
    bet = [rng.uniform(0, np.pi, p) for p in ps]
    b = batch.QaoaBatch(lib, ns, diags, max_evals=len(ns), max_p=4)
    got = b.eval(list(range(len(ns))), ps, gam, bet)
    assert np.array_equal(got, b.eval(list(range(len(ns))), ps, gam, bet))
    for k, n in enumerate(ns):
        want = oracle_eval(orc, n, diags[k], ps[k], gam[k], bet[k])
        assert abs(got[k] - want) <= 1e-12, (n, ps[k], got[k], want)
    b.close()


@pytest.mark.parametrize("big", [3e15, 1e300, np.inf, np.nan])
def test_phases_beyond_the_register_kernel(big):
    """A phase of 2^50 or more, or one that is not finite, takes the whole list through the LDS kernel: the bits of that
    kernel's own shape, NaN where a phase has no value."""
    lib = orkan_amd.load(5)
    rng = np.random.default_rng(7)
    ns = [6, 13, 14]
    diags = [rng.uniform(0, 2, 1 << n) for n in ns]
    diags[1][5] = big
    args = ([0, 1, 2], [2, 2, 1], [rng.uniform(0.5, 1, 2) for _ in ns], [rng.uniform(0, 3, 2) for _ in ns])
    b = batch.QaoaBatch(lib, ns, diags, max_evals=3, max_p=2)
    got = b.eval(*args)
    b.set_config(12, 512)
    assert np.array_equal(got, b.eval(*args), equal_nan=True)
    assert np.isfinite(got[[0, 2]]).all() and (np.isfinite(big) or np.isnan(got[1]))
    b.close()

"""Timed cases: what a user of this library has it do, through its public entry points.

Each case names a `kind` of work and its sizes.  `listed()` holds representative ones, `draw()` takes more from the
same ranges, `prepare()` builds what a program has in hand before the call (states, observables, plans, weights),
`run()` is one pass, `work()` the bytes and operations the pass cannot do without, `exact()` the same outputs from
plain torch in 64 bits.

Kinds
  circuit      statevector brick layers gate by gate, then <O>: the library's headline workload (28 qubits) and the
               small circuits that interactive work consists of
  variational  state_plus, p x (exp_diag, rx on every qubit), mean: one energy of a QAOA optimisation loop
  fused        orkan_layer_1q, one call for a layer of rotations
  noise        density matrix: h and ry on every qubit, cz on neighbours, damping and depolarizing channels, mean
  pairs        density matrix: noisy entangling layer, cx and a two-qubit channel on every neighbour pair, a swap, a
               Toffoli and a dense two-qubit unitary across the register
  layouts      state_cp, conversion between the packed and the tiled layout, and to the other precision
  batch        QaoaBatch.eval, many QAOA circuits of uneven sizes in one call
  train        Adam steps of the energy surrogate from host minibatches, then its weights
  screen       surrogate predictions for a pool of candidate angles, and the best 64
  sample       sample_matrix of an ansatz with a linear combination after the sampled channel
"""
import ctypes as C
import math

import numpy as np
import torch

import orkan_amd
from orkan_amd import batch, surrogate
from orkan_amd._ffi import MIXED_PACKED, MIXED_TILED, PURE, QOP, AnsatzChannelT, StateT, SuperopT

FP32 = orkan_amd.ORKAN_FP32
TILE = 5                      # log2 of the tile edge of the default library
KINDS = {"packed": MIXED_PACKED, "tiled": MIXED_TILED}


def listed():
    return [
        # an interactive small circuit: every call is a launch
        {"name": "circuit-10", "kind": "circuit", "n": 10, "f32": False, "layers": 2},
        # the headline configuration: one brick layer on 28 qubits
        {"name": "circuit-28", "kind": "circuit", "n": 28, "f32": False, "layers": 1},
        # one energy evaluation inside an optimiser's loop
        {"name": "variational-17", "kind": "variational", "n": 17, "f32": False, "layers": 4},
        # a layer of general rotations in one call
        {"name": "fused-25", "kind": "fused", "n": 25, "f32": False},
        # a noisy circuit's layer, large, in the tiled layout
        {"name": "noise-tiled-13", "kind": "noise", "n": 13, "f32": False, "layout": "tiled"},
        # the same at an ordinary size, packed and in the smaller storage type
        {"name": "noise-packed-9-c64", "kind": "noise", "n": 9, "f32": True, "layout": "packed"},
        # a noisy entangling layer
        {"name": "pairs-tiled-12", "kind": "pairs", "n": 12, "f32": False, "layout": "tiled"},
        # moving a density matrix between layouts and precisions
        {"name": "layouts-packed-12", "kind": "layouts", "n": 12, "f32": False, "layout": "packed"},
        # the batched-search configuration: 4096 instances of 10 to 20 qubits, 1 to 8 layers
        {"name": "batch-4096", "kind": "batch", "count": 4096, "n_lo": 10, "n_hi": 20, "p_lo": 1, "p_hi": 8},
        # surrogate training at its configured batch
        {"name": "train-4096", "kind": "train", "rows": 4096, "hidden": 512, "layers": 3, "steps": 4},
        # screening of a pool of candidates (a million and an odd remainder)
        {"name": "screen-1000003", "kind": "screen", "rows": 1000003, "hidden": 512, "layers": 3},
        # one channel's sample matrix
        {"name": "sample-18", "kind": "sample", "n": 18, "leaves": 48, "after": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["circuit", "variational", "fused", "noise", "pairs", "layouts", "batch", "train", "screen",
                       "sample"])
    f32 = rng.random() < 0.3
    layout = rng.choice(["packed", "tiled"])
    if kind == "circuit":
        n = rng.randint(3, 27)
        return {"kind": kind, "n": n, "f32": f32, "layers": rng.randint(1, 4) if n < 24 else 1}
    if kind == "variational":
        n = rng.randint(4, 25)
        return {"kind": kind, "n": n, "f32": f32, "layers": rng.randint(1, 8) if n < 23 else 2}
    if kind == "fused":
        return {"kind": kind, "n": rng.randint(13, 28), "f32": f32}
    if kind == "noise":
        return {"kind": kind, "n": rng.randint(3, 13), "f32": f32, "layout": layout}
    if kind == "pairs":
        return {"kind": kind, "n": rng.randint(4, 13), "f32": f32, "layout": layout}
    if kind == "layouts":
        return {"kind": kind, "n": rng.randint(4, 13), "f32": f32, "layout": layout}
    if kind == "batch":
        lo = rng.randint(4, 12)
        p_lo = rng.randint(1, 4)
        return {"kind": kind, "count": _log_int(rng, 1, 4096), "n_lo": lo, "n_hi": min(20, lo + rng.randint(0, 8)),
                "p_lo": p_lo, "p_hi": p_lo + rng.randint(0, 4)}
    if kind == "train":
        return {"kind": kind, "rows": _log_int(rng, 33, 8192), "hidden": rng.choice([128, 256, 512, 512, 512]),
                "layers": rng.randint(2, 3), "steps": rng.randint(1, 6)}
    if kind == "screen":
        return {"kind": kind, "rows": _log_int(rng, 1000, 1000000), "hidden": rng.choice([256, 512, 512, 512]),
                "layers": rng.randint(2, 3)}
    n = rng.randint(6, 20)
    return {"kind": kind, "n": n, "leaves": _log_int(rng, 2, 64), "after": rng.randint(0, 2)}


# ---- inputs ------------------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _lib():
    return orkan_amd.load(TILE)


def _gen(seed):
    g = torch.Generator(device=_device())
    g.manual_seed(1000003 + seed)
    return g


def _random_psi(n, g, dtype=torch.complex128):
    v = torch.randn(1 << n, 2, generator=g, device=_device(), dtype=torch.float64)
    v /= v.norm()
    return torch.view_as_complex(v).to(dtype)


def _random_rho(n, g):
    """a rank-8 mixed state, dense D x D"""
    D = 1 << n
    a = torch.view_as_complex(torch.randn(D, 8, 2, generator=g, device=_device(), dtype=torch.float64))
    a = a / a.abs().square().sum().sqrt()
    return a @ a.conj().T.contiguous()


def _to_layout(rho, n, layout):
    """dense D x D -> stored array (tiled: row-major lower tiles, n below the tile zero-padded; packed: the lower
    triangle by columns)"""
    D = 1 << n
    if layout == "packed":
        t = rho.T.contiguous()
        return t[torch.ones(D, D, dtype=torch.bool, device=rho.device).triu()]
    T = 1 << TILE
    if D < T:
        out = torch.zeros(T, T, dtype=rho.dtype, device=rho.device)
        out[:D, :D] = rho
        return out.reshape(-1)
    nt = D // T
    tiles = rho.reshape(nt, T, nt, T).permute(0, 2, 1, 3)
    keep = torch.ones(nt, nt, dtype=torch.bool, device=rho.device).tril()
    return tiles[keep].reshape(-1)


def _stored(n, layout):
    D = 1 << n
    if layout == "packed":
        return D * (D + 1) // 2
    nt = max(1, D >> TILE)
    return nt * (nt + 1) // 2 << (2 * TILE)


def _adopt(lib, kind, n, tensor):
    """a state whose storage is this device tensor"""
    st = StateT(kind | (FP32 if tensor.dtype == torch.complex64 else 0), None, 0)
    buf = C.c_void_p(tensor.data_ptr())
    lib.state_init(C.byref(st), n, C.byref(buf))
    return st


class _Device:
    def __init__(self, ptr, count, f32):
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<c8" if f32 else "<c16",
                                         "data": (ptr, False), "version": 2}


def _view(ptr, count, f32):
    """a state's storage as a torch tensor (no copy)"""
    return torch.as_tensor(_Device(ptr, count, f32), device=_device())


def _obs(count, g):
    return torch.rand(count, generator=g, device=_device(), dtype=torch.float64) * 2 - 1


def _dp(t):
    return C.cast(t.data_ptr(), C.POINTER(C.c_double))


def _host(seed):
    return np.random.default_rng(7919 + seed)


def _maxcut(n, r):
    iu, ju = np.triu_indices(n, 1)
    w = np.where(r.random(iu.size) < 0.5, r.uniform(0.0, 1.0, iu.size), 0.0)
    W = np.zeros((n, n))
    W[iu, ju] = w
    return W


def _spins(n):
    x = torch.arange(1 << n, device=_device())
    return torch.stack([1.0 - 2.0 * ((x >> q) & 1).to(torch.float64) for q in range(n)], 1)


def _cut_diag(W, S):
    """C(x) = sum_(i<j) w_ij [x_i != x_j]"""
    w = torch.as_tensor(W, device=S.device)
    return 0.5 * (w.sum() - ((S @ w) * S).sum(1))


def _amp_damp(gm):
    k = [np.array([[1, 0], [0, math.sqrt(1 - gm)]], complex), np.array([[0, math.sqrt(gm)], [0, 0]], complex)]
    return sum(np.kron(a, a.conj()) for a in k)


PAULI = [np.eye(2, dtype=complex), np.array([[0, 1], [1, 0]], complex), np.array([[0, -1j], [1j, 0]], complex),
         np.array([[1, 0], [0, -1]], complex)]


def _depol(p):
    w = [1 - 3 * p / 4, p / 4, p / 4, p / 4]
    return sum(c * np.kron(a, a.conj()) for c, a in zip(w, PAULI))


def _depol2(p):
    """two-qubit depolarizing channel (local index x_q1 + 2 x_q2)"""
    out = np.zeros((16, 16), complex)
    for i, a in enumerate(PAULI):
        for j, b in enumerate(PAULI):
            k = np.kron(b, a)
            out += ((1 - 15 * p / 16) if i == j == 0 else p / 16) * np.kron(k, k.conj())
    return out


def _unitary(d, r):
    q, t = np.linalg.qr(r.standard_normal((d, d)) + 1j * r.standard_normal((d, d)))
    return q * (np.diag(t) / np.abs(np.diag(t)))


def _brick(case, seed):
    """gate list of the circuit kind"""
    r, n, ops = _host(seed), case["n"], []
    for layer in range(case["layers"]):
        for q in range(n):
            ops += [(g, q, float(r.uniform(0, 2 * math.pi))) for g in ("rx", "ry", "rz")]
        ops += [("cx", q, q + 1) for q in range(layer % 2, n - 1, 2)]
    return ops


def _noise_ops(case, seed):
    r, n = _host(seed), case["n"]
    ops = [("h", q) for q in range(n)] + [("ry", q, float(r.uniform(0, 2 * math.pi))) for q in range(n)]
    ops += [("cz", q, q + 1) for q in range(0, n - 1, 2)]
    return ops + [("damp", q) for q in range(n)] + [("depol", q) for q in range(n)]


def _pair_ops(case):
    n = case["n"]
    ops = []
    for q in range(n - 1):
        ops += [("cx", q, q + 1), ("depol2", q, q + 1)]
    return ops + [("swap_gate", 0, n - 1), ("ccx", n - 1, 0, n // 2), ("dense", 1, n - 2 if n > 4 else n - 1)]


def _sample_ops(case, seed):
    """the ansatz: a prefix channel, the sampled channel, `after` linear combinations of two operations"""
    r, n = _host(seed), case["n"]

    def op():
        name = ("rx", "ry", "rz", "cx", "h")[int(r.integers(5))]
        if name == "cx":
            return (name,) + tuple(int(q) for q in r.choice(n, 2, replace=False))
        q = int(r.integers(n))
        return (name, q) if name == "h" else (name, q, float(r.uniform(0, 2 * math.pi)))

    chans = [([op(), op()], 0.6 * r.standard_normal(2) + 0.6j * r.standard_normal(2))]
    chans.append(([op() for _ in range(case["leaves"])], None))
    for _ in range(case["after"]):
        chans.append(([op(), op()], 0.6 * r.standard_normal(2) + 0.6j * r.standard_normal(2)))
    return chans


def _mlp_weights(case, seed):
    r, k, W, b = _host(seed), surrogate.IN_DIM, [], []
    for _ in range(case["layers"]):
        W.append((r.standard_normal((k, case["hidden"])) * math.sqrt(2.0 / k)).astype(np.float32))
        b.append((0.02 * r.standard_normal(case["hidden"])).astype(np.float32))
        k = case["hidden"]
    return W, b, (r.standard_normal(k) * math.sqrt(1.0 / k)).astype(np.float32), 0.05


def _graph_features(r):
    return surrogate.graph_features(r.uniform(0, 1, int(r.integers(40, 80))))


def _train_data(case, seed):
    """minibatches as the search builds them: graph features and angles, standardised targets"""
    r, P = _host(seed + 50), surrogate.P
    gfs = np.stack([_graph_features(r) for _ in range(16)])
    out = []
    for _ in range(case["steps"]):
        rows = case["rows"]
        x = surrogate.features(gfs[r.integers(0, 16, rows)], r.uniform(0, math.pi, (rows, P)),
                               r.uniform(0, math.pi, (rows, P)))
        out.append((x, r.standard_normal(rows).astype(np.float32)))
    return out


def _lr(case):
    return [1e-3 * 0.9 ** s for s in range(case["steps"])]


def _batch_inputs(case, seed):
    r = _host(seed)
    ev = []
    for _ in range(case["count"]):
        n = int(r.integers(case["n_lo"], case["n_hi"] + 1))
        p = int(r.integers(case["p_lo"], case["p_hi"] + 1))
        ev.append((n, p, _maxcut(n, r), r.uniform(0, math.pi, p), r.uniform(0, math.pi, p)))
    return ev


# ---- prepare -----------------------------------------------------------------------------------
def prepare(case, seed):
    lib, kind, g = _lib(), case["kind"], _gen(seed)
    dt = torch.complex64 if case.get("f32") else torch.complex128
    s = {"kind": kind, "lib": lib, "case": case}
    if kind in ("circuit", "fused"):
        n = case["n"]
        s["psi"] = _random_psi(n, g, dt)
        s["st"] = _adopt(lib, PURE, n, s["psi"])
        if kind == "circuit":
            s["obs"] = _obs(1 << n, g)
            s["ops"] = [(getattr(lib, o[0]), (C.byref(s["st"]),) + o[1:]) for o in _brick(case, seed)]
        else:
            r = _host(seed)
            # column-major 2 x 2 matrices, one per qubit
            s["mats"] = np.ascontiguousarray(np.stack([_unitary(2, r).T for _ in range(n)]), dtype=np.complex128)
    elif kind == "variational":
        n, r = case["n"], _host(seed)
        s["diag"] = _cut_diag(_maxcut(n, r), _spins(n))
        s["angles"] = [(float(a), float(b)) for a, b in r.uniform(0, math.pi, (case["layers"], 2))]
        s["st"] = StateT(PURE | (FP32 if case["f32"] else 0), None, 0)
    elif kind in ("noise", "pairs"):
        n = case["n"]
        s["rho"] = _to_layout(_random_rho(n, g), n, case["layout"]).to(dt)
        s["st"] = st = _adopt(lib, KINDS[case["layout"]], n, s["rho"])
        s["obs"] = _obs(1 << n, g)
        s["sops"] = {"damp": np.ascontiguousarray(_amp_damp(0.05)), "depol": np.ascontiguousarray(_depol(0.02)),
                     "depol2": np.ascontiguousarray(_depol2(0.03))}
        sop = {k: SuperopT(2 if k == "depol2" else 1, v.ctypes.data) for k, v in s["sops"].items()}
        s["dense"] = np.ascontiguousarray(_unitary(4, _host(seed)).T)
        calls = []
        for o in (_noise_ops(case, seed) if kind == "noise" else _pair_ops(case)):
            if o[0] in ("damp", "depol"):
                calls.append((lib.channel_1q, (C.byref(st), C.byref(sop[o[0]]), o[1])))
            elif o[0] == "depol2":
                calls.append((lib.channel_2q, (C.byref(st), C.byref(sop[o[0]]), o[1], o[2])))
            elif o[0] == "dense":
                calls.append((lib.two_from_mat, (C.byref(st), o[1], o[2], s["dense"].ctypes.data)))
            else:
                calls.append((getattr(lib, o[0]), (C.byref(st),) + o[1:]))
        s["ops"] = calls
    elif kind == "layouts":
        n = case["n"]
        s["rho"] = _to_layout(_random_rho(n, g), n, case["layout"]).to(dt)
        s["st"] = _adopt(lib, KINDS[case["layout"]], n, s["rho"])
        s["made"] = []
    elif kind == "batch":
        ev, spins, diags = _batch_inputs(case, seed), {}, []
        for n, _, W, _, _ in ev:
            if n not in spins:
                spins[n] = _spins(n)
            diags.append(_cut_diag(W, spins[n]))
        torch.cuda.synchronize()
        s["batch"] = batch.QaoaBatch(lib, [e[0] for e in ev], [d.data_ptr() for d in diags], len(ev), max(e[1] for e in ev))
        del diags
        s["args"] = (list(range(len(ev))), [e[1] for e in ev], [e[3] for e in ev], [e[4] for e in ev])
        s["batch"].autotune(*s["args"], reps=2)
    elif kind in ("train", "screen"):
        rows = case["rows"]
        s["mlp"] = surrogate.Mlp(lib, hidden=case["hidden"], layers=case["layers"],
                                 max_batch=rows if kind == "train" else 65536)
        s["mlp"].set_weights(*_mlp_weights(case, seed))
        if kind == "train":
            s["data"] = _train_data(case, seed)
        else:
            r = _host(seed + 50)
            s["gf"] = _graph_features(r)
            s["ang"] = torch.rand(rows, 2 * surrogate.P, generator=g, device=_device())
            s["y"] = torch.empty(rows, device=_device())
    else:
        n = case["n"]
        s["psi"], s["obs"] = _random_psi(n, g), _obs(1 << n, g)
        s["src"], s["st"] = _adopt(lib, PURE, n, s["psi"]), StateT(PURE, None, 0)
        chans = _sample_ops(case, seed)
        s["keep"], table = [], []
        for ops, w in chans:
            cbs = [QOP(lambda p, f=getattr(lib, o[0]), a=o[1:]: f(p, *a)) for o in ops]
            arr = (QOP * len(cbs))(*cbs)
            wa = None if w is None else np.ascontiguousarray(w, dtype=np.complex128)
            s["keep"] += [cbs, arr, wa]
            table.append(AnsatzChannelT(len(cbs), arr, None if wa is None else wa.ctypes.data))
        s["table"] = (AnsatzChannelT * len(table))(*table)
        s["S"] = np.zeros((case["leaves"], case["leaves"]), np.complex128)
    return s


# ---- run ---------------------------------------------------------------------------------------
def run(s):
    lib, kind, case = s["lib"], s["kind"], s["case"]
    if kind == "circuit":
        for f, a in s["ops"]:
            f(*a)
        return {"psi": s["psi"], "mean": lib.mean(C.byref(s["st"]), _dp(s["obs"]))}
    if kind == "variational":
        st, n, d = C.byref(s["st"]), case["n"], _dp(s["diag"])
        lib.state_plus(st, n)
        for gamma, beta in s["angles"]:
            lib.exp_diag(st, d, gamma)
            for q in range(n):
                lib.rx(st, q, 2.0 * beta)
        e = lib.mean(st, d)
        return {"energy": e, "psi": _view(s["st"].data, 1 << n, case["f32"])}
    if kind == "fused":
        lib.orkan_layer_1q(C.byref(s["st"]), s["mats"].ctypes.data)
        return s["psi"]
    if kind == "noise":
        for f, a in s["ops"]:
            f(*a)
        return {"rho": s["rho"], "mean": lib.mean(C.byref(s["st"]), _dp(s["obs"]))}
    if kind == "pairs":
        for f, a in s["ops"]:
            f(*a)
        return s["rho"]
    if kind == "layouts":
        st = C.byref(s["st"])
        for old in s["made"]:
            lib.state_free(C.byref(old))
        other = "tiled" if case["layout"] == "packed" else "packed"
        cp, re = lib.state_cp(st), StateT()
        lib.orkan_state_relayout(st, C.byref(re), KINDS[other])
        cv = lib.orkan_state_convert(C.byref(re), 0 if case["f32"] else 1)
        s["made"] = [cp, re, cv]
        return [_view(cp.data, _stored(case["n"], case["layout"]), case["f32"]),
                _view(re.data, _stored(case["n"], other), case["f32"]),
                _view(cv.data, _stored(case["n"], other), not case["f32"])]
    if kind == "batch":
        return s["batch"].eval(*s["args"])
    if kind == "train":
        losses = [s["mlp"].train_step(x, t, lr) for (x, t), lr in zip(s["data"], _lr(case))]
        W, b, wo, bo = s["mlp"].get_weights()
        return {"losses": np.array(losses, np.float32), "W": W, "b": b, "w_out": wo, "b_out": np.float32(bo)}
    if kind == "screen":
        k = 64
        idx, vals = np.empty(k, np.int32), np.empty(k, np.float32)
        s["mlp"].forward_candidates(s["gf"], s["ang"].data_ptr(), case["rows"], s["y"].data_ptr())
        rc = lib.orkan_topk_f32(s["y"].data_ptr(), case["rows"], k, idx.ctypes.data_as(C.POINTER(C.c_int)),
                                vals.ctypes.data_as(C.POINTER(C.c_float)))
        if rc:
            raise RuntimeError(f"orkan_topk_f32 failed ({rc})")
        return {"y": s["y"], "best": vals, "index": idx}
    # sample_matrix consumes its input: it gets a copy of the starting state
    lib.state_free(C.byref(s["st"]))
    s["st"] = lib.state_cp(C.byref(s["src"]))
    rc = lib.sample_matrix(C.byref(s["st"]), s["obs"].data_ptr(), s["table"], len(s["table"]), 1, 1 << 32,
                           s["S"].ctypes.data)
    if rc:
        raise RuntimeError(f"sample_matrix failed ({rc})")
    return {"S": s["S"], "prefix": _view(s["st"].data, 1 << case["n"], False)}


# ---- work --------------------------------------------------------------------------------------
def work(case):
    """bytes: every call's inputs read once and outputs written once; flops: the arithmetic of the definition"""
    kind, e = case["kind"], 8 if case.get("f32") else 16
    if kind == "circuit":
        N, n = 1 << case["n"], case["n"]
        cx = sum(len(range(layer % 2, n - 1, 2)) for layer in range(case["layers"]))
        return {"bytes": N * (6 * e * n * case["layers"] + e * cx + e + 8), "flops": N * (3 * 14 * n * case["layers"] + 5)}
    if kind == "variational":
        N, n, p = 1 << case["n"], case["n"], case["layers"]
        return {"bytes": N * (e + p * (2 * e + 8 + 2 * e * n) + e + 8), "flops": N * p * (14 * n + 30)}
    if kind == "fused":
        return {"bytes": (2 * e) << case["n"], "flops": (14 * case["n"]) << case["n"]}
    if kind == "noise":
        n, L = case["n"], _stored(case["n"], case["layout"])
        return {"bytes": L * (4 * n * 2 * e + (n // 2) * 3 * e // 4), "flops": L * 4 * n * 32}
    if kind == "pairs":
        n, L = case["n"], _stored(case["n"], case["layout"])
        return {"bytes": L * ((n - 1) * (7 * e // 2) + 3 * e // 2 + 7 * e // 8 + 2 * e), "flops": L * ((n - 1) * 128 + 64)}
    if kind == "layouts":
        a = _stored(case["n"], case["layout"])
        b = _stored(case["n"], "tiled" if case["layout"] == "packed" else "packed")
        return {"bytes": 2 * e * a + e * (a + b) + 24 * b, "flops": 0}
    if kind == "batch":
        # the cost diagonals are read once; the states need never leave the chip's registers and LDS
        ns = range(case["n_lo"], case["n_hi"] + 1)
        amps = case["count"] * sum(1 << n for n in ns) / len(ns)
        p = 0.5 * (case["p_lo"] + case["p_hi"])
        rx = case["count"] * sum(n << n for n in ns) / len(ns)
        return {"bytes": 8 * amps, "flops": p * (8 * rx + 30 * amps)}
    h, layers = case.get("hidden", 0), case.get("layers", 0)
    if kind == "train":
        params = surrogate.IN_DIM * h + (layers - 1) * h * h + h * (layers + 1)
        return {"bytes": case["steps"] * (case["rows"] * (surrogate.IN_DIM + 1) * 4 + params * 24),
                "flops": case["steps"] * 6.0 * case["rows"] * params}
    if kind == "screen":
        macs = 2 * surrogate.P * h + (layers - 1) * h * h + h
        return {"bytes": case["rows"] * (2 * surrogate.P * 4 + 4) + 2 * (layers - 1) * h * h, "flops": 2.0 * case["rows"] * macs}
    N, K, a = 1 << case["n"], case["leaves"], case["after"]
    return {"bytes": N * (8 + 16 * 2 + K * 16 * (2 + 6 * a)), "flops": N * (4.0 * K * K + K * (14 + a * 44))}


# ---- exact -------------------------------------------------------------------------------------
GATES = {"h": lambda: np.array([[1, 1], [1, -1]]) / math.sqrt(2),
         "rx": lambda t: np.array([[math.cos(t / 2), -1j * math.sin(t / 2)], [-1j * math.sin(t / 2), math.cos(t / 2)]]),
         "ry": lambda t: np.array([[math.cos(t / 2), -math.sin(t / 2)], [math.sin(t / 2), math.cos(t / 2)]]),
         "rz": lambda t: np.diag([complex(math.cos(t / 2), -math.sin(t / 2)), complex(math.cos(t / 2), math.sin(t / 2))])}


def _mat1(psi, q, m):
    """2 x 2 matrix on bit q of the last axis, in place"""
    v = psi.view(psi.shape[:-1] + (-1, 2, 1 << q))
    a, b = v[..., 0, :].clone(), v[..., 1, :].clone()
    v[..., 0, :] = complex(m[0][0]) * a + complex(m[0][1]) * b
    v[..., 1, :] = complex(m[1][0]) * a + complex(m[1][1]) * b


def _perm_index(op, D, device):
    i = torch.arange(D, device=device)
    if op[0] == "cx":
        return torch.where((i >> op[1]) & 1 == 1, i ^ (1 << op[2]), i)
    if op[0] == "ccx":
        return torch.where(((i >> op[1]) & (i >> op[2]) & 1) == 1, i ^ (1 << op[3]), i)
    differ = ((i >> op[1]) ^ (i >> op[2])) & 1 == 1
    return torch.where(differ, i ^ ((1 << op[1]) | (1 << op[2])), i)


def _apply_sv(psi, op):
    if op[0] == "cx":
        v = psi.view([2] * int(math.log2(psi.numel()) + 0.5))
        n = v.dim()
        at = [slice(None)] * n
        at[n - 1 - op[1]] = 1
        one, zero = list(at), list(at)
        zero[n - 1 - op[2]], one[n - 1 - op[2]] = 0, 1
        t = v[tuple(zero)].clone()
        v[tuple(zero)] = v[tuple(one)]
        v[tuple(one)] = t
    else:
        _mat1(psi, op[1], GATES[op[0]](*op[2:]))


def _sop(rho, D, q, S):
    v = rho.view(-1, 2, 1 << q, D >> (q + 1), 2, 1 << q)
    old = [v[:, k, :, :, l, :].clone() for k in (0, 1) for l in (0, 1)]
    for i in range(2):
        for j in range(2):
            v[:, i, :, :, j, :] = sum(complex(S[2 * i + j, k]) * old[k] for k in range(4) if S[2 * i + j, k] != 0)


def _sop2(rho, D, q1, q2, S):
    lo, hi = min(q1, q2), max(q1, q2)
    shape = (D >> (hi + 1), 2, 1 << (hi - lo - 1), 2, 1 << lo)
    v = rho.view(shape + shape)

    def at(a, b):
        r = {q1: a & 1, q2: a >> 1}
        c = {q1: b & 1, q2: b >> 1}
        return (slice(None), r[hi], slice(None), r[lo], slice(None), slice(None), c[hi], slice(None), c[lo])

    old = [v[at(k // 4, k % 4)].clone() for k in range(16)]
    for m in range(16):
        v[at(m // 4, m % 4)] = sum(complex(S[m, k]) * old[k] for k in range(16) if S[m, k] != 0)


def _apply_dm(rho, D, op, dense):
    if op[0] in ("h", "ry"):
        m = np.asarray(GATES[op[0]](*op[2:]), complex)
        _sop(rho, D, op[1], np.kron(m, m.conj()))
    elif op[0] == "damp":
        _sop(rho, D, op[1], _amp_damp(0.05))
    elif op[0] == "depol":
        _sop(rho, D, op[1], _depol(0.02))
    elif op[0] == "depol2":
        _sop2(rho, D, op[1], op[2], _depol2(0.03))
    elif op[0] == "dense":
        _sop2(rho, D, min(op[1:]), max(op[1:]), np.kron(dense, dense.conj()))
    elif op[0] == "cz":
        i = torch.arange(D, device=rho.device)
        f = 1.0 - 2.0 * ((i >> op[1]) & (i >> op[2]) & 1).to(torch.float64)
        rho *= f[:, None] * f[None, :]
    else:
        p = _perm_index(op, D, rho.device)
        rho.copy_(rho[p][:, p])


def _gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def exact(case, seed):
    kind, g = case["kind"], _gen(seed)
    dt = torch.complex64 if case.get("f32") else torch.complex128
    dev = _device()
    if kind in ("circuit", "fused"):
        psi = _random_psi(case["n"], g, dt).to(torch.complex128)
        if kind == "fused":
            r = _host(seed)
            for q in range(case["n"]):
                _mat1(psi, q, _unitary(2, r))
            return psi
        obs = _obs(1 << case["n"], g)
        for op in _brick(case, seed):
            _apply_sv(psi, op)
        return {"psi": psi, "mean": float((psi.abs().square() * obs).sum())}
    if kind == "variational":
        n, r = case["n"], _host(seed)
        d = _cut_diag(_maxcut(n, r), _spins(n))
        psi = torch.full((1 << n,), 1.0 / math.sqrt(1 << n), dtype=torch.complex128, device=dev)
        for gamma, beta in r.uniform(0, math.pi, (case["layers"], 2)):
            psi *= torch.polar(torch.ones_like(d), -d * float(gamma))
            for q in range(n):
                _mat1(psi, q, GATES["rx"](2.0 * float(beta)))
        return {"energy": float((psi.abs().square() * d).sum()), "psi": psi}
    if kind in ("noise", "pairs", "layouts"):
        n, D = case["n"], 1 << case["n"]
        rho = _random_rho(n, g).to(dt).to(torch.complex128)
        if kind == "layouts":
            # the copy, the other layout, and that in the other precision: the same numbers, rounded once
            other = "tiled" if case["layout"] == "packed" else "packed"
            low = torch.tril(rho)
            full = low + torch.tril(rho, -1).conj().T if case["layout"] == "packed" else rho
            moved = _to_layout(full, n, other)
            return [_to_layout(rho, n, case["layout"]), moved, moved]
        obs = _obs(D, g)
        dense = _unitary(4, _host(seed))
        for op in (_noise_ops(case, seed) if kind == "noise" else _pair_ops(case)):
            _apply_dm(rho, D, op, dense)
        out = _to_layout(rho, n, case["layout"])
        if kind == "pairs":
            return out
        return {"rho": out, "mean": float((rho.diagonal().real * obs).sum())}
    if kind == "batch":
        ev = _batch_inputs(case, seed)
        out = np.zeros(len(ev))
        for n in sorted({e[0] for e in ev}):
            S, idx = _spins(n), [k for k, e in enumerate(ev) if e[0] == n]
            per = max(1, (1 << 26) >> n)
            for c in range(0, len(idx), per):
                part = idx[c:c + per]
                d = torch.stack([_cut_diag(ev[k][2], S) for k in part])
                psi = torch.full(d.shape, 1.0 / math.sqrt(1 << n), dtype=torch.complex128, device=dev)
                for layer in range(max(ev[k][1] for k in part)):
                    gb = np.array([(ev[k][3][layer], ev[k][4][layer]) if layer < ev[k][1] else (0.0, 0.0) for k in part])
                    gb = torch.as_tensor(gb, device=dev)
                    psi *= torch.polar(torch.ones_like(d), -d * gb[:, :1])
                    co, si = torch.cos(gb[:, 1])[:, None, None], -1j * torch.sin(gb[:, 1])[:, None, None]
                    for q in range(n):
                        v = psi.view(len(part), -1, 2, 1 << q)
                        a, b = v[:, :, 0, :].clone(), v[:, :, 1, :].clone()
                        v[:, :, 0, :] = co * a + si * b
                        v[:, :, 1, :] = si * a + co * b
                out[part] = (psi.abs().square() * d).sum(1).cpu().numpy()
        return out
    if kind in ("train", "screen"):
        W, b, wo, bo = _mlp_weights(case, seed)
        P = [torch.as_tensor(w, device=dev).double() for w in W + b + [wo]] + [torch.tensor(float(np.float32(bo)), device=dev).double()]
        nl = case["layers"]

        def forward(x):
            for l in range(nl):
                x = _gelu(x @ P[l] + P[nl + l])
            return x @ P[2 * nl] + P[2 * nl + 1]

        if kind == "screen":
            gf = torch.as_tensor(_graph_features(_host(seed + 50)), device=dev).double()
            ang = torch.rand(case["rows"], 2 * surrogate.P, generator=g, device=dev)
            y = torch.cat([forward(torch.cat([gf.expand(len(a), -1), a.double()], 1)) for a in ang.split(65536)])
            return {"y": y, "best": torch.topk(y, 64).values, "index": None}
        for p in P:
            p.requires_grad_(True)
        m, v, losses = [torch.zeros_like(p) for p in P], [torch.zeros_like(p) for p in P], []
        for k, ((x, t), lr) in enumerate(zip(_train_data(case, seed), _lr(case)), 1):
            loss = (forward(torch.as_tensor(x, device=dev).double()) - torch.as_tensor(t, device=dev).double()).square().mean()
            grads = torch.autograd.grad(loss, P)
            losses.append(float(loss.detach()))
            with torch.no_grad():
                for i, gr in enumerate(grads):
                    m[i] = 0.9 * m[i] + 0.1 * gr
                    v[i] = 0.999 * v[i] + 0.001 * gr * gr
                    P[i] -= lr * (m[i] / (1 - 0.9 ** k)) / ((v[i] / (1 - 0.999 ** k)).sqrt() + 1e-8)
        P = [p.detach() for p in P]
        return {"losses": np.array(losses), "W": P[:nl], "b": P[nl:2 * nl], "w_out": P[2 * nl], "b_out": float(P[2 * nl + 1])}
    psi, obs = _random_psi(case["n"], g), _obs(1 << case["n"], g)

    def combine(v, ops, w):
        out = torch.zeros_like(v)
        for op, c in zip(ops, w):
            t = v.clone()
            _apply_sv(t, op)
            out += complex(c) * t
        return out

    chans = _sample_ops(case, seed)
    prefix = combine(psi, *chans[0])
    leaves = []
    for op in chans[1][0]:
        t = prefix.clone()
        _apply_sv(t, op)
        for ch in chans[2:]:
            t = combine(t, *ch)
        leaves.append(t)
    M = torch.stack(leaves)
    S = (M.conj() * obs) @ M.T.contiguous()
    return {"S": S.T.contiguous().cpu().numpy(), "prefix": prefix}

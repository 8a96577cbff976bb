"""The work that programs have hip-mps do, as cases that can be timed and compared.

Every case goes through the Python front end (tnqvm_amd.mps) as a user's program does: a circuit
from |0...0> to its expectation values, a batch or a request loop of many circuits, a noisy circuit,
or a measurement of a state that is already there.  Circuits, bond dimensions, cutoffs and noise
channels have the shapes of this repository's own workloads (tnqvm_amd.circuits, bench.py, tests).

Results of complex128 runs are float64 / complex128.  The sites of a mixed-precision run are
complex64, so what such a run's circuits give is returned in that precision (float32); a
measurement of a complex64 state that is already there accumulates in 64 bits and is returned so.
A circuit's result is one array: <Z> of every qubit, then the norm <psi|psi>.
"""
from __future__ import annotations

import numpy as np

from tnqvm_amd import circuits as C
from tnqvm_amd import mps, noise

CUTOFF = 1e-10  # svd-cutoff of the random circuits (bench.py)

_shared = {}


def _engine():
    """The one engine that a program creates and keeps."""
    if "engine" not in _shared:
        _shared["engine"] = mps.Engine()
    return _shared["engine"]


# ---------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # a small circuit of a unit test or of one step of a variational loop: latency only
        {"name": "circuit_5q", "kind": "circuit", "gates": "u3_cnot", "n": 5, "depth": 6, "chi": 0, "precision": "fp64"},
        # the plain small case: 12-qubit U3 + CNOT line, every bond exact (up to 64)
        {"name": "line_12q", "kind": "circuit", "gates": "u3_cnot", "n": 12, "depth": 20, "chi": 0, "precision": "fp64"},
        # one ordinary truncated circuit alone, complex128, odd width
        {"name": "brickwork_27q_chi64", "kind": "circuit", "gates": "haar", "n": 27, "depth": 14, "chi": 64,
         "precision": "fp64"},
        # one circuit with large bonds (theta' up to 1536 x 1536), complex128: few, large SVDs
        {"name": "brickwork_22q_chi768", "kind": "circuit", "gates": "haar", "n": 22, "depth": 12, "chi": 768,
         "precision": "fp64"},
        # QAOA MaxCut through its swap network, exact bonds, rank-deficient theta', <ZZ> of every edge
        {"name": "qaoa_16q_p2", "kind": "qaoa", "n": 16, "p": 2, "precision": "fp64"},
        # many circuits of uneven width, depth and bond submitted together, mixed precision
        {"name": "batch_32_uneven", "kind": "batch", "count": 32, "n_min": 16, "n_max": 40, "d_min": 10, "d_max": 16,
         "chi": 128, "precision": "mixed"},
        # the request loop on circuits of the headline size: 40 qubits, chi 256, mixed precision
        {"name": "serve_8x40q_chi256", "kind": "serve", "count": 8, "n": 40, "depth": 14, "chi": 256,
         "precision": "mixed"},
        # a noisy circuit as the reference's noisy visitor runs one: outcome probabilities, full density matrix
        {"name": "noisy_8q", "kind": "noisy", "n": 8, "depth": 3, "shots": 1024, "precision": "fp64"},
        # many noisy circuits advanced together, thermal relaxation after every gate
        {"name": "noisy_batch_16x40q", "kind": "noisy_batch", "count": 16, "n": 40, "depth": 4, "precision": "fp64"},
        # amplitudes of random bit strings of a large state (the verification step of sampling experiments)
        {"name": "amplitudes_40q_chi256", "kind": "amplitudes", "n": 40, "chi": 256, "strings": 1000,
         "precision": "fp64"},
        # observables of a large state: <Z> of every qubit, <ZZ> of neighbours and of some distant pairs
        {"name": "observables_40q_chi256", "kind": "observables", "n": 40, "chi": 256, "far": 4, "precision": "mixed"},
        # bit strings drawn from a state too wide for its vector
        {"name": "sample_32q_chi64", "kind": "sample", "n": 32, "chi": 64, "shots": 1000, "precision": "fp64"},
    ]


def _log(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng):
    kind = rng.choice(["small", "line", "brickwork", "large", "qaoa", "batch", "serve", "noisy", "noisy_batch",
                       "amplitudes", "observables", "sample"])
    both = rng.choice(["fp64", "mixed"])
    if kind == "small":
        return {"kind": "circuit", "gates": rng.choice(["u3_cnot", "haar"]), "n": rng.randint(2, 8),
                "depth": rng.randint(3, 12), "chi": 0, "precision": "fp64"}
    if kind == "line":
        return {"kind": "circuit", "gates": rng.choice(["u3_cnot", "haar"]), "n": rng.randint(9, 13),
                "depth": rng.randint(8, 22), "chi": 0, "precision": "fp64"}
    if kind == "brickwork":
        return {"kind": "circuit", "gates": "haar", "n": rng.randint(16, 32), "depth": rng.randint(8, 14),
                "chi": _log(rng, 24, 128), "precision": "fp64"}
    if kind == "large":
        return {"kind": "circuit", "gates": "haar", "n": rng.randint(18, 22), "depth": rng.randint(8, 12),
                "chi": rng.randint(160, 700), "precision": "fp64"}
    if kind == "qaoa":
        return {"kind": "qaoa", "n": 2 * rng.randint(4, 8), "p": rng.randint(1, 2) if both == "fp64" else 1,
                "precision": "fp64"}
    if kind == "batch":
        lo = rng.randint(16, 28)
        d = rng.randint(10, 13)
        return {"kind": "batch", "count": rng.randint(20, 32), "n_min": lo, "n_max": rng.randint(lo + 4, 40),
                "d_min": d, "d_max": rng.randint(d + 1, 16), "chi": rng.randint(100, 128), "precision": "mixed"}
    if kind == "serve":
        return {"kind": "serve", "count": rng.randint(2, 8), "n": rng.randint(30, 40), "depth": rng.randint(11, 14),
                "chi": rng.randint(130, 256), "precision": "mixed"}
    if kind == "noisy":
        return {"kind": "noisy", "n": rng.randint(3, 8), "depth": rng.randint(2, 3), "shots": rng.randint(256, 2048),
                "precision": "fp64"}
    if kind == "noisy_batch":
        return {"kind": "noisy_batch", "count": rng.randint(1, 16), "n": rng.randint(9, 40), "depth": rng.randint(2, 4),
                "precision": "fp64"}
    if kind == "amplitudes":
        return {"kind": "amplitudes", "n": rng.randint(21, 40), "chi": _log(rng, 12, 256),
                "strings": _log(rng, 1, 1000), "precision": both}
    if kind == "observables":
        return {"kind": "observables", "n": rng.randint(21, 40), "chi": _log(rng, 12, 256), "far": rng.randint(0, 4),
                "precision": both}
    return {"kind": "sample", "n": rng.randint(20, 32), "chi": _log(rng, 8, 64), "shots": _log(rng, 16, 1000),
            "precision": both}


# ---------------------------------------------------------------------------------------- inputs
def _rng(case, seed):
    return np.random.default_rng([int(seed), sum(ord(ch) for ch in case["kind"])])


def _circuit(kind, n, depth, seed):
    return C.u3_cnot_line(n, depth, seed=seed) if kind == "u3_cnot" else C.haar_brickwork(n, depth, seed=seed)


def _seeds(case, seed, count):
    return [int(x) for x in _rng(case, seed).integers(1, 1 << 31, size=count)]


def _jobs(case, seed):
    """(n, depth, chi, gate seed) of every circuit of a batch or a request loop."""
    if case["kind"] == "serve":
        return [(case["n"], case["depth"], case["chi"], s) for s in _seeds(case, seed, case["count"])]
    rng, out = _rng(case, seed), []
    for k in range(case["count"]):
        # the widths and depths span their ranges evenly, whatever the seed, in a shuffled pairing
        f = k / max(1, case["count"] - 1)
        g = ((k * 7) % case["count"]) / max(1, case["count"] - 1)
        n = round(case["n_min"] + f * (case["n_max"] - case["n_min"]))
        d = round(case["d_min"] + g * (case["d_max"] - case["d_min"]))
        out.append((n, d, case["chi"] >> (k & 1), int(rng.integers(1, 1 << 31))))
    return out


def _qaoa(case, seed):
    gates, edges, pos, _ = C.qaoa_maxcut(case["n"], case["p"], seed=_seeds(case, seed, 1)[0])
    return gates, [(pos[a], pos[b]) for a, b in edges]


def _bonds(n, chi):
    return [min(2 ** min(k, n - k, 20), chi) for k in range(n + 1)]


def _sites(case, seed):
    """Left-canonical sites of a random state of norm 1 with bonds min(2^k, 2^(n-k), chi)."""
    rng, n = _rng(case, seed), case["n"]
    b = _bonds(n, case["chi"])
    dt = np.complex64 if case["precision"] == "mixed" else np.complex128
    out = []
    for k in range(n):
        a = rng.standard_normal((2 * b[k], b[k + 1])) + 1j * rng.standard_normal((2 * b[k], b[k + 1]))
        out.append(np.linalg.qr(a)[0].reshape(b[k], 2, b[k + 1]).astype(dt).astype(np.complex128))
    return out


def _pairs(case, seed):
    rng, n = np.random.default_rng([int(seed), 5]), case["n"]
    near = [(q, q + 1) for q in range(n - 1)]
    return near + [tuple(int(x) for x in rng.choice(n, size=2, replace=False)) for _ in range(case["far"])]


def _relaxation(n, seed):
    """A device's noise model: thermal relaxation of every qubit for the duration of its gates."""
    rng = np.random.default_rng([int(seed), 6])
    t1, t2 = rng.uniform(4e4, 7e4, n), rng.uniform(2e4, 5e4, n)
    one = {q: noise.thermal_relaxation(80.0, t1[q], t2[q]) for q in range(n)}
    two = {(q, q + 1): {x: noise.thermal_relaxation(400.0, t1[x], t2[x]) for x in (q, q + 1)} for q in range(n - 1)}
    return noise.NoiseModel(one, two, {q: (0.02, 0.01) for q in range(n)})


def _damping(n, seed):
    rng = np.random.default_rng([int(seed), 7])
    g = rng.uniform(0.01, 0.05, n)
    one = {q: noise.amplitude_damping(g[q] / 4) for q in range(n)}
    two = {(q, q + 1): {x: noise.amplitude_damping(g[x]) for x in (q, q + 1)} for q in range(n - 1)}
    return noise.NoiseModel(one, two, {q: (0.02, 0.01) for q in range(n)})


def prepare(case, seed):
    e, kind = _engine(), case["kind"]
    s = {"case": case, "engine": e, "seed": int(seed)}
    if kind == "circuit":
        s["gates"] = _circuit(case["gates"], case["n"], case["depth"], _seeds(case, seed, 1)[0])
    elif kind == "qaoa":
        s["gates"], s["edges"] = _qaoa(case, seed)
    elif kind in ("batch", "serve"):
        s["jobs"] = [{"n": n, "gates": C.haar_brickwork(n, d, seed=g),
                      "trunc": mps.trunc_opts(cutoff=CUTOFF, max_bond=chi, precision=case["precision"])}
                     for n, d, chi, g in _jobs(case, seed)]
    elif kind == "noisy":
        s["gates"] = C.u3_cnot_line(case["n"], case["depth"], seed=_seeds(case, seed, 1)[0])
        s["noise"] = _damping(case["n"], seed)
    elif kind == "noisy_batch":
        s["circuits"] = [(case["n"], C.u3_cnot_line(case["n"], case["depth"], seed=g))
                         for g in _seeds(case, seed, case["count"])]
        s["noise"] = _relaxation(case["n"], seed)
    else:
        st = mps.MpsState(e, case["n"], cutoff=CUTOFF, max_bond=case["chi"], precision=case["precision"])
        for k, a in enumerate(_sites(case, seed)):
            st.set_site(k, a)
        s["state"] = st
        if kind == "amplitudes":
            s["bits"] = C.random_bitstrings(case["n"], case["strings"], int(seed))
        elif kind == "observables":
            s["pairs"] = _pairs(case, seed)
        else:
            s["draws"] = np.random.default_rng([int(seed), 8]).random(case["shots"] * case["n"])
    return s


# ---------------------------------------------------------------------------------------- one pass
def _result(case, z, norm):
    r = np.concatenate([z, [norm]])
    return r.astype(np.float32) if case["precision"] == "mixed" else r


def run(state):
    case, e, kind = state["case"], state["engine"], state["case"]["kind"]
    if kind == "circuit":
        st = mps.MpsState(e, case["n"], cutoff=CUTOFF, max_bond=case["chi"], precision=case["precision"])
        st.run(state["gates"])
        out = _result(case, st.expval_z_all(), st.norm())
        st.close()
        return out
    if kind == "qaoa":
        st = mps.MpsState(e, case["n"], cutoff=1e-12, precision=case["precision"])
        st.run(state["gates"])
        out = _result(case, st.expval_zz(state["edges"]), st.norm())
        st.close()
        return out
    if kind == "batch":
        return [_result(case, r["expval_z"], r["norm"]) for r in e.run_batch(state["jobs"])]
    if kind == "serve":
        srv = mps.Server(e)
        tickets = [srv.submit(j["n"], j["gates"], j["trunc"]) for j in state["jobs"]]
        while any(srv.pending()):
            srv.step()
        return [_result(case, r["expval_z"], r["norm"]) for r in (srv.poll(t) for t in tickets)]
    if kind == "noisy":
        r = mps.run_noisy(e, case["n"], state["gates"], state["noise"], measured=range(case["n"]),
                          shots=case["shots"], seed=state["seed"], precision=case["precision"])
        return {"z": _result(case, r["expval_z"], r["trace"]), "probabilities": r["probabilities"],
                "density_matrix": r["density_matrix"]}
    if kind == "noisy_batch":
        rs = mps.run_noisy_batch(e, state["circuits"], state["noise"], precision=case["precision"])
        return [_result(case, r["expval_z"], r["trace"]) for r in rs]
    st = state["state"]
    if kind == "amplitudes":
        return st.amplitudes(state["bits"])
    if kind == "observables":
        return {"z": st.expval_z_all(), "zz": st.expval_zz(state["pairs"]), "norm": st.norm()}
    strings = st.sample_sequential(list(range(case["n"])), state["draws"])
    return np.frombuffer("".join(strings).encode(), dtype=np.uint8).reshape(case["shots"], case["n"]) - ord("0")


# ---------------------------------------------------------------------------------------- floors
def _gate_work(cl, cm, cr, k, es):
    """theta and the nominal SVD of one two-qubit gate (k triplets kept): flops, site bytes."""
    m, n = 2 * max(cl, cr), 2 * min(cl, cr)
    flops = 32 * cl * cm * cr + 128 * cl * cr + 4 * (14 * m * n * n + 8 * n ** 3)
    return flops, es * 2 * (cl * cm + cm * cr + cl * k + k * cr)


def _circuit_work(n, pairs, chi, es):
    """A circuit's gates on the sites `pairs` in order, bonds as generic gates grow them."""
    b, flops, nbytes = [1] * (n + 1), 0.0, 0.0
    for i in pairs:
        k = min(2 * b[i], 2 * b[i + 2], chi or 1 << 20)
        f, w = _gate_work(b[i], b[i + 1], b[i + 2], k, es)
        b[i + 1] = k
        flops, nbytes = flops + f, nbytes + w
    f, w = _env_work(n, b, es)
    return flops + 2 * f, nbytes + w


def _env_work(n, b, es):
    """One sweep of environments over the chain."""
    flops = sum(8.0 * 2 * (b[k] * b[k] * b[k + 1] + b[k] * b[k + 1] * b[k + 1]) for k in range(n))
    return flops, sum(2.0 * es * b[k] * b[k + 1] for k in range(n))


def _brick_pairs(n, depth):
    return [i for layer in range(depth) for i in range(layer % 2, n - 1, 2)]


def work(case):
    kind, es = case["kind"], 8 if case["precision"] == "mixed" else 16
    n = case.get("n", 0)
    if kind == "circuit":
        f, w = _circuit_work(n, _brick_pairs(n, case["depth"]), case["chi"], es)
    elif kind == "qaoa":
        f, w = _circuit_work(n, [i for _ in range(case["p"]) for t in range(n) for i in range(t % 2, n - 1, 2)], 0, es)
    elif kind in ("batch", "serve"):
        f = w = 0.0
        for m, d, chi, _ in _jobs(case, 0):
            a, b = _circuit_work(m, _brick_pairs(m, d), chi, es)
            f, w = f + a, w + b
    elif kind in ("noisy", "noisy_batch"):
        # gates as on a pure state; a channel per gate and qubit doubles the Kraus leg it compresses
        f, w = _circuit_work(n, _brick_pairs(n, case["depth"]), 0, es)
        f, w = case.get("count", 1) * 4 * f, case.get("count", 1) * 4 * w
        if kind == "noisy":
            f, w = f + 8.0 * 8 ** n, w + 16.0 * 4 ** n
    else:
        b = _bonds(n, case["chi"])
        f, w = _env_work(n, b, es)
        if kind == "amplitudes":
            f, w = sum(8.0 * case["strings"] * b[k] * b[k + 1] for k in range(n)), w + case["strings"] * (n + 16.0)
        elif kind == "observables":
            far = sum(abs(p - q) + 1 for p, q in _pairs(case, 0)[n - 1:])
            f = f * (2 + (3.0 + far / n) / 2)  # both environment sweeps, then a step per <Z> and per pair site
        else:
            f, w = f * (1 + 1.5 * case["shots"]), w + 8.0 * case["shots"] * n
    return {"bytes": float(w), "flops": float(f)}


# ---------------------------------------------------------------------------------------- 64-bit values
_PAULI = {"H": np.array([[1, 1], [1, -1]]) / np.sqrt(2.0)}


def _matrix(g):
    if "matrix" in g:
        return np.asarray(g["matrix"], dtype=np.complex128)
    if g["name"] == "U":
        t, p, l = g["params"]
        c, s = np.cos(t / 2), np.sin(t / 2)
        return np.array([[c, -np.exp(1j * l) * s], [np.exp(1j * p) * s, np.exp(1j * (p + l)) * c]])
    if g["name"] == "Rx":
        t = g["params"][0]
        return np.array([[np.cos(t / 2), -1j * np.sin(t / 2)], [-1j * np.sin(t / 2), np.cos(t / 2)]])
    if g["name"] == "CNOT":
        return np.array([[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 0, 1], [0, 0, 1, 0]], dtype=np.complex128)
    return _PAULI[g["name"]].astype(np.complex128)


def _apply(t, mat, qs):
    """mat on the axes qs of t."""
    k = len(qs)
    m = mat.reshape((2,) * (2 * k))
    return np.moveaxis(np.tensordot(m, t, axes=(range(k, 2 * k), qs)), range(k), qs)


def _dense(n, gates):
    v = np.zeros((2,) * n, dtype=np.complex128)
    v[(0,) * n] = 1
    for g in gates:
        v = _apply(v, _matrix(g), list(g["qubits"]))
    return v


def _signs(p, qs):
    """Sum of the probabilities p with the sign of Z on every qubit of qs."""
    for q in qs:
        p = p * np.array([1.0, -1.0]).reshape([2 if a == q else 1 for a in range(p.ndim)])
    return float(p.sum())


def _truncated(n, gates, chi):
    """Sites after a circuit with the reference's truncation, on plain LAPACK."""
    a = [np.array([1, 0], dtype=np.complex128).reshape(1, 2, 1) for _ in range(n)]
    for g in gates:
        m, q = _matrix(g), g["qubits"]
        if len(q) == 1:
            a[q[0]] = np.einsum("ij,ljr->lir", m, a[q[0]])
            continue
        i = q[0]
        t = np.tensordot(a[i], a[i + 1], axes=(2, 0))
        t = np.einsum("abcd,lcdr->labr", m.reshape(2, 2, 2, 2), t)
        cl, cr = t.shape[0], t.shape[3]
        u, s, v = np.linalg.svd(t.reshape(2 * cl, 2 * cr), full_matrices=False)
        below = np.flatnonzero(s < CUTOFF)
        k = min(below[0] + 1 if len(below) else len(s), chi or len(s))
        r = np.sqrt(s[:k])
        a[i], a[i + 1] = (u[:, :k] * r).reshape(cl, 2, k), (r[:, None] * v[:k]).reshape(k, 2, cr)
    return a


def _left(a, e, d=None):
    x = np.tensordot(e, a if d is None else a * np.asarray(d).reshape(1, 2, 1), axes=(1, 0))
    return np.tensordot(a.conj(), x, axes=([0, 1], [0, 1]))


def _rights(sites):
    r = [np.ones((1, 1), dtype=np.complex128)]
    for a in reversed(sites):
        x = np.tensordot(a, r[-1], axes=(2, 1))
        r.append(np.tensordot(a.conj(), x, axes=([1, 2], [1, 2])))
    return r[::-1]


def _expectations(sites, pairs=()):
    n, z = len(sites), [1.0, -1.0]
    lefts = [np.ones((1, 1), dtype=np.complex128)]
    for a in sites:
        lefts.append(_left(a, lefts[-1]))
    rights = _rights(sites)
    ez = np.array([np.sum(_left(sites[k], lefts[k], z) * rights[k + 1]).real for k in range(n)])
    ezz = []
    for p, q in ((min(x), max(x)) for x in pairs):
        e = lefts[p]
        for k in range(p, q + 1):
            e = _left(sites[k], e, z if k in (p, q) else None)
        ezz.append(np.sum(e * rights[q + 1]).real)
    return ez, np.array(ezz), float(lefts[n][0, 0].real)


def _rho(n, gates, model):
    """Density matrix after a noisy circuit; axes: ket qubits, then bra qubits."""
    r = np.zeros((2,) * (2 * n), dtype=np.complex128)
    r[(0,) * (2 * n)] = 1

    def both(x, m, qs):
        return _apply(_apply(x, m, list(qs)), m.conj(), [n + q for q in qs])

    for g in gates:
        r = both(r, _matrix(g), g["qubits"])
        for q, ops in model.channels(g):
            r = sum(both(r, k, (q,)) for k in ops)
    return r


def exact(case, seed):
    kind, n = case["kind"], case.get("n", 0)
    if kind == "circuit":
        gates = _circuit(case["gates"], n, case["depth"], _seeds(case, seed, 1)[0])
        if case["chi"] == 0:
            p = np.abs(_dense(n, gates)) ** 2
            return np.array([_signs(p, [q]) for q in range(n)] + [float(p.sum())])
        if case["chi"] > 128:
            return None  # LAPACK takes minutes for these SVDs
        ez, _, norm = _expectations(_truncated(n, gates, case["chi"]))
        return np.concatenate([ez, [norm]])
    if kind == "qaoa":
        gates, edges = _qaoa(case, seed)
        p = np.abs(_dense(n, gates)) ** 2
        return np.array([_signs(p, e) for e in edges] + [float(p.sum())])
    if kind == "noisy":
        gates = C.u3_cnot_line(n, case["depth"], seed=_seeds(case, seed, 1)[0])
        r = _rho(n, gates, _damping(n, seed))
        # index sum_i b_i 2^i: qubit 0 fastest
        r = r.transpose(list(range(n - 1, -1, -1)) + list(range(2 * n - 1, n - 1, -1))).reshape(1 << n, 1 << n)
        p = np.diag(r).real.copy()
        bits = (np.arange(1 << n)[:, None] >> np.arange(n)[None, :]) & 1
        z = (p[:, None] * (1 - 2 * bits)).sum(0)
        return {"z": np.concatenate([z, [p.sum()]]), "probabilities": p, "density_matrix": r}
    if kind == "amplitudes":
        sites, bits = _sites(case, seed), C.random_bitstrings(n, case["strings"], int(seed))
        v = np.ones((case["strings"], 1), dtype=np.complex128)
        for k, a in enumerate(sites):
            w = np.empty((case["strings"], a.shape[2]), dtype=np.complex128)
            for b in (0, 1):
                w[bits[:, k] == b] = v[bits[:, k] == b] @ a[:, b, :]
            v = w
        return v[:, 0]
    if kind == "observables":
        ez, ezz, norm = _expectations(_sites(case, seed), _pairs(case, seed))
        return {"z": ez, "zz": ezz, "norm": norm}
    # batches and request loops: minutes of LAPACK; noisy batches: the reference's Kraus bound drops
    # weight, so the density matrix is not what they give; bit strings are whole numbers
    return None

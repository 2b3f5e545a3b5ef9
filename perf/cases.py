"""What programs have this engine do, as measurable cases.

Each case is one call through the package's public entry points: a circuit's
probability, a projector norm (exact pair sums or sampled, with the |H^t> or
an |L> decomposition), a batch of uneven norms, shots drawn from a circuit,
inner products of given states, random states.  Sizes are those of the
repository's own configurations and tests, or generic ones in the same ranges
(t from a few qubits to 64, decompositions of 2 to 2^20 terms).
"""
import functools
import math

import numpy as np

from circuitsimulator_amd import Engine
from circuitsimulator_amd.engine import Instance, Projector, instance_array
from circuitsimulator_amd.probability import probability
from circuitsimulator_amd.sample import sampleShots
from circuitsimulator_amd.workloads import c1_circuit, commuting_paulis, random_L


def listed():
    return [
        # the joint distribution of two qubits of a small circuit, one
        # probability() call per outcome, as interactive use and parameter
        # scans repeat them: launches and host work
        {"name": "probability_small", "kind": "probability", "n": 8, "t": 8},
        # the smallest norms: one projector, a few hundred pair terms
        {"name": "exact_L_small", "kind": "exact", "H": False, "t": 13, "r": 5, "k": 5},
        # one exact norm of an |L> of ordinary rank
        {"name": "exact_L_pairs", "kind": "exact", "H": False, "t": 24, "r": 12, "k": 11},
        # one exact norm with the default decomposition, the largest t a
        # single call is used for
        {"name": "exact_H", "kind": "exact", "H": True, "t": 30, "r": 10, "k": 0},
        # a queue of unrelated norms of every size in one launch
        {"name": "exact_batch_uneven", "kind": "batch", "count": 192, "tmin": 8, "tmax": 48, "kmin": 2, "kmax": 12},
        # a norm estimated with the default number of samples, odd t
        {"name": "sampled_L_default", "kind": "sampled", "H": False, "t": 37, "r": 11, "k": 9, "M": 2000},
        # the headline norm estimation: 2^16 samples x 2^12 terms
        {"name": "sampled_L_large", "kind": "sampled", "H": False, "t": 48, "r": 24, "k": 12, "M": 65536},
        # sampling with the default decomposition
        {"name": "sampled_H", "kind": "sampled", "H": True, "t": 40, "r": 12, "k": 0, "M": 512},
        # the widest states (rows of more than 60 bits)
        {"name": "sampled_L_wide", "kind": "sampled", "H": False, "t": 63, "r": 21, "k": 10, "M": 512},
        # qubit-by-qubit sampling of a 40-qubit circuit, the shots together
        {"name": "shots", "kind": "shots", "n": 40, "gates": 400, "t": 40, "k": 8, "qubits": 8, "shots": 256},
        # inner products of states that the program holds
        {"name": "pairs", "kind": "pairs", "n": 48, "r": 24, "k": 12, "pairs": 4096},
        # random stabilizer states drawn and projected on the device
        {"name": "states", "kind": "states", "n": 33, "r": 12, "count": 3000},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["probability", "exact", "exact", "batch", "sampled", "sampled", "sampled", "shots", "pairs",
                       "states"])
    if kind == "probability":
        return {"kind": kind, "n": rng.randint(4, 10), "t": rng.randint(6, 14)}
    if kind == "exact":
        if rng.random() < 0.5:
            t = rng.randint(7, 30)
            return {"kind": kind, "H": True, "t": t, "r": rng.randint(1, min(10, t // 2)), "k": 0}
        t = rng.randint(9, 60)
        return {"kind": kind, "H": False, "t": t, "r": rng.randint(1, t // 2), "k": rng.randint(2, min(13, t - 1))}
    if kind == "batch":
        tmin = rng.randint(6, 30)
        return {"kind": kind, "count": _log_int(rng, 5, 192), "tmin": tmin, "tmax": rng.randint(tmin + 4, 56),
                "kmin": 2, "kmax": rng.randint(6, 12)}
    if kind == "sampled":
        if rng.random() < 0.4:
            t = rng.randint(9, 40)
            chi = 1 << ((t + 1) // 2)
            return {"kind": kind, "H": True, "t": t, "r": rng.randint(1, t // 2), "k": 0,
                    "M": _log_int(rng, 50, min(16000, (1 << 28) // chi))}
        t = rng.randint(9, 64)
        k = rng.randint(3, min(13, t - 1))
        return {"kind": kind, "H": False, "t": t, "r": rng.randint(1, t // 2), "k": k,
                "M": _log_int(rng, 50, min(30000, (1 << (27 if t <= 60 else 20)) >> k))}
    if kind == "shots":
        n = rng.randint(6, 40)
        return {"kind": kind, "n": n, "gates": 10 * n, "t": rng.randint(9, 40), "k": rng.randint(4, 8),
                "qubits": rng.randint(2, min(8, n)), "shots": _log_int(rng, 8, 256)}
    n = rng.randint(5, 64)
    if kind == "pairs":
        return {"kind": kind, "n": n, "r": rng.randint(1, n // 2), "k": rng.randint(1, min(12, n)),
                "pairs": _log_int(rng, 20, 4096)}
    return {"kind": "states", "n": n, "r": rng.randint(1, n // 2), "count": _log_int(rng, 20, 3000)}


@functools.lru_cache(maxsize=None)
def _engine():
    """The context that a program creates once and keeps."""
    return Engine(0)


def _chi(case):
    return 1 << ((case["t"] + 1) // 2) if case["H"] else 1 << case["k"]


def _norm_inputs(case, seed):
    """(phases, x masks, z masks) of the projector, and L."""
    rng = np.random.default_rng(seed)
    group = commuting_paulis(rng, case["t"], case["r"])
    return group, [] if case["H"] else random_L(rng, case["t"], case["k"])


def _small_circuit(case, seed):
    """Circuit of H, S, T and CX in which every T sits between Hadamards, so
    its probabilities are not those of a Clifford circuit; and y."""
    n, rng = case["n"], np.random.default_rng(seed)
    rows = []

    def add(ops):
        rows.append("".join(ops.get(q, "_") for q in range(n)))

    for q in range(n):
        add({q: "H"})
    for i in range(case["t"]):
        q = int(rng.integers(0, n)) if i >= 4 else i % 2
        add({q: "T"})
        if rng.random() < 0.5:
            add({q: "S"})
        add({q: "H"})
        other = int(rng.integers(0, n - 1))
        add({q: "C", other + (other >= q): "X"})
        if rng.random() < 0.5:
            add({q: "H"})
    return "\n".join(rows) + "\n", "".join(str(int(b)) for b in rng.integers(0, 2, size=case["t"]))


_OUTCOMES = [{0: a, 1: b} for a in (0, 1) for b in (0, 1)]


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "seed": seed}
    if kind == "probability":
        s["circ"], s["y"] = _small_circuit(case, seed)
    elif kind in ("exact", "sampled"):
        s["engine"] = _engine()
        (ph, xs, zs), s["L"] = _norm_inputs(case, seed)
        s["P"] = Projector.make(ph, xs, zs, case["t"])
    elif kind == "batch":
        s["engine"] = _engine()
        rng = np.random.default_rng(seed)
        A = instance_array(case["count"])
        for at in range(case["count"]):
            t = int(rng.integers(case["tmin"], case["tmax"] + 1))
            k = int(rng.integers(case["kmin"], min(case["kmax"], t) + 1))
            ph, xs, zs = commuting_paulis(rng, t, int(rng.integers(1, t // 2 + 1)))
            inst = Instance()
            inst.P = Projector.make(ph, xs, zs, t)
            inst.k = k
            for i, v in enumerate(random_L(rng, t, k)):
                inst.L[i] = v
            A[at] = np.frombuffer(bytes(inst), dtype=A.dtype)[0]
        s["instances"] = A
    elif kind == "shots":
        s["circ"], s["y"] = c1_circuit(seed=seed, n=case["n"], gates=case["gates"], ts=case["t"])
    else:
        s["engine"] = E = _engine()
        n = case["n"]
        rng = np.random.default_rng(seed)
        ph, xs, zs = commuting_paulis(rng, n, case["r"])
        s["P"] = Projector.make(ph, xs, zs, n)
        if kind == "pairs":
            # projected random states against decomposition states of an |L>
            L = random_L(rng, n, case["k"])
            count = case["pairs"]
            s["s2"] = E.prep_states(False, n, L, rng.integers(0, 1 << case["k"], size=count))
            s["s1"], _ = E.random_states(n, seed, 0, count, s["P"])
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "probability":
        return np.array([float(probability(s["circ"], m, {"quiet": True, "y": s["y"], "seed": s["seed"]}))
                         for m in _OUTCOMES])
    if kind == "exact":
        r, hist = s["engine"].exact_projector(s["P"], s["L"], case["k"], case["H"], want_hist=True)
        # the Kahan sums are FP32 sums: given back in their own precision
        return {"value": np.float64(r.value), "re": np.float64(r.re), "im": np.float64(r.im),
                "kahan": np.float32(r.kahan_re), "hist": hist, "terms": r.terms, "ips": r.ips}
    if kind == "batch":
        values, _ = s["engine"].batch_exact_values(s["instances"])
        return {"values": values}
    if kind == "sampled":
        r, extra = s["engine"].sampled_projector(s["P"], s["L"], case["k"], case["H"], s["seed"], 0, case["M"])
        return {"mean": np.float64(r.mean), "mean_kahan": np.float32(r.mean_kahan), "zsum": extra["zsum"],
                "sexp": extra["sexp"], "kahan": extra["kahan"].astype(np.float32), "ips": r.ips,
                "vanished": r.vanished}
    if kind == "shots":
        trace = []
        out = sampleShots(s["circ"], {}, list(range(case["qubits"])), case["shots"],
                          {"exact": False, "k": case["k"], "quiet": True, "y": s["y"], "trace": trace,
                           "rng": np.random.default_rng(s["seed"])})
        return {"bits": np.array([[int(c) for c in o] for o in out], dtype=np.int64),
                "P": np.array([v["P"] for v in trace if "round" in v])}
    if kind == "pairs":
        out, _ = s["engine"].inner_products(case["n"], s["s1"], s["s2"])
        return out
    states, sexp = s["engine"].random_states(case["n"], s["seed"], 0, case["count"], s["P"])
    return {"states": states, "sexp": sexp}


def work(case):
    """Bytes of the inputs and outputs, and of the arithmetic only what every
    method has to do: each term's exact addition to a sum of four integers and
    its addition to the FP32 pair (12 operations), each state's bit rows
    formed once."""
    kind = case["kind"]
    if kind in ("exact", "sampled"):
        chi = _chi(case)
        terms = chi * (chi + 1) // 2 if kind == "exact" else chi * case["M"]
        out = 8 * 1032 if kind == "exact" else 52 * case["M"]
        return {"bytes": 20 * case["r"] + 8 * case["k"] + out, "flops": 12 * terms}
    if kind == "batch":
        ks = range(case["kmin"], case["kmax"] + 1)
        terms = case["count"] * sum((1 << k) * ((1 << k) + 1) // 2 for k in ks) // len(ks)
        return {"bytes": 1900 * case["count"], "flops": 12 * terms}
    if kind == "shots":
        chi = 1 << case["k"]
        norms = 2 * case["shots"] * case["qubits"]
        return {"bytes": 8 * case["k"] * norms, "flops": 12 * norms * (chi * (chi + 1) // 2)}
    if kind == "probability":
        chi = 1 << ((case["t"] + 1) // 2)
        return {"bytes": 4 * case["n"] * (case["n"] + 4 * case["t"]), "flops": 4 * 12 * chi * (chi + 1)}
    words = 3 * case["n"] + 4
    if kind == "pairs":
        return {"bytes": (16 * words + 12) * case["pairs"], "flops": words * case["pairs"]}
    return {"bytes": (8 * words + 4) * case["count"], "flops": words * case["count"]}


# ------------------------------------------------------------ 64-bit values
def _circuit_probability(circ, measure):
    """P(measure) of a compiled circuit of {H, S, T, CX} by state vector."""
    rows = [ln for ln in circ.splitlines() if ln]
    n = len(rows[0])
    psi = np.zeros(1 << n, dtype=np.complex128)
    psi[0] = 1.0
    idx = np.arange(1 << n)
    for row in rows:
        ops = {c: q for q, c in enumerate(row) if c != "_"}
        if "C" in ops:
            on = ((idx >> ops["C"]) & 1) == 1
            psi[on] = psi[idx[on] ^ (1 << ops["X"])]
            continue
        (g, q), = ops.items()
        one = ((idx >> q) & 1) == 1
        if g == "H":
            other = psi[idx ^ (1 << q)]
            psi = np.where(one, other - psi, other + psi) * math.sqrt(0.5)
        else:
            psi[one] *= {"S": 1j, "T": np.exp(0.25j * math.pi)}[g]
    keep = np.ones(1 << n, dtype=bool)
    for q, b in measure.items():
        keep &= ((idx >> q) & 1) == b
    return float(np.sum(np.abs(psi[keep]) ** 2) / np.sum(np.abs(psi) ** 2))


def _magic_norm(t, group):
    """|| Pi |H^t> ||^2 scaled as the sum of the unit states of the
    decomposition: the mean over the group's elements of their expectation
    value, a product over qubits (1, 1/sqrt2 for X and Z, 0 for Y)."""
    ph, xs, zs = group
    total = 0.0
    elements = [(0, 0, 0)]
    for p, x, z in zip(ph, xs, zs):
        elements += [((q + p + 2 * bin(b & z).count("1")) & 3, a ^ z, b ^ x) for q, a, b in elements]
    for q, a, b in elements:
        if a & b == 0:
            total += (1, 0, -1, 0)[q] * 2.0 ** (-bin(a | b).count("1") / 2)
    return total / len(elements) * 2.0 ** (t // 2) * ((2 + math.sqrt(2)) if t % 2 else 1.0)


def _code_norm(t, group, L):
    """<L| Pi |L> for |L> the sum over the code words x of the product of
    |+> on supp(x) and |0> elsewhere, by state vector."""
    words = np.zeros(1, dtype=np.int64)
    for v in L:
        words = np.concatenate([words, words ^ v])
    f = np.zeros(1 << t)
    for w in words:
        f[w] += 2.0 ** (-bin(int(w)).count("1") / 2)
    for q in range(t):  # psi(y) = sum of f(x) over x containing y
        g = f.reshape(-1, 2, 1 << q)
        g[:, 0] += g[:, 1]
    psi = f.astype(np.complex128)
    out = psi.copy()
    idx = np.arange(1 << t, dtype=np.uint32)
    for p, x, z in zip(*group):
        moved = out[idx ^ np.uint32(x)]
        par = idx & np.uint32(z)
        for sh in (16, 8, 4, 2, 1):
            par ^= par >> np.uint32(sh)
        moved[(par & 1) == 1] *= -1
        out += (1, 1j, -1, -1j)[p & 3] * moved
        out *= 0.5
    return float(np.vdot(psi, out).real)


def exact(case, seed):
    if case["kind"] == "probability":
        circ, _ = _small_circuit(case, seed)
        return np.array([_circuit_probability(circ, m) for m in _OUTCOMES])
    if case["kind"] == "exact" and (case["H"] or case["t"] <= 24):
        group, L = _norm_inputs(case, seed)
        v = _magic_norm(case["t"], group) if case["H"] else _code_norm(case["t"], group, L)
        v = np.float64(v)
        return {"value": abs(v), "re": v, "im": np.float64(0), "kahan": v, "hist": None, "terms": None, "ips": None}
    return None

"""The sweep kernels (csrc/cse_sweep.h) run on the CPU (sweep_cpu.h: a block as
fibers, its waves one after the other between barriers) against every term
eliminated by itself: a block's shared tables are complete before any wave
reads them, in whatever order its waves run; the claim loop takes every item
once; partial sums are flushed whole; a lane's FP32 sums are short."""
import ctypes
import math
import os
import random
import shutil
import subprocess

import numpy as np
import pytest

TESTS = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(TESTS), "circuitsimulator_amd", "csrc")
HIST = 129 * 8
REC = 68
ASM = 'asm volatile("" : "+s"(c));'  # keeps a scalar out of sight of the compiler's hoisting
ORDERS = [(0, 1, 2, 3), (3, 2, 1, 0), (1, 3, 0, 2)]


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    d = tmp_path_factory.mktemp("sweep")
    with open(os.path.join(CSRC, "cse_sweep.h")) as f:
        src = f.read()
    assert src.count("asm volatile") == src.count(ASM) == 1
    (d / "sweep_host.h").write_text(src.replace(ASM, ""))
    (d / "sweep.cpp").write_text('#include "sweep_cpu.h"\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-ffp-contract=off", "-Wno-attributes", "-shared", "-fPIC", "-I", TESTS,
                    "-I", CSRC, "-I", str(d), "-o", str(d / "sweep.so"), str(d / "sweep.cpp")], check=True)
    return d


@pytest.fixture
def S(built, tmp_path):
    """the library, loaded anew: shared memory that nothing has written"""
    so = tmp_path / "sweep.so"
    shutil.copy(built / "sweep.so", so)
    return ctypes.CDLL(str(so))


def ptr(a, t):
    return a.ctypes.data_as(ctypes.POINTER(t))


def word(v):
    """slot x of a mask at bit 31 - x of its half"""
    return sum(1 << (31 - x if x < 32 else 95 - x) for x in range(64) if v >> x & 1)


def record(rnd, n, vanished=0, dens=None):
    dens = rnd.random() if dens is None else dens
    J = [0] * 64
    for a in range(n):
        for b in range(a):
            if rnd.random() < dens:
                J[a] |= 1 << b
                J[b] |= 1 << a
    d1, d2, F = (rnd.getrandbits(n) for _ in range(3))
    w0 = n << 8 | rnd.randrange(8) << 16 | rnd.randrange(0, n // 2 + 1) << 24 | vanished << 40
    return [w0, word(F), word(d1), word(d2)] + [word(j) for j in J]


def instance(S, rnd, mode, n, k, G, signs=0, pairs=1, lds=38, count=3, first=3, rec=None):
    """adds a random instance: index bits that move `first` slots and then one
    or two more each, or for signs slot and sign in turn"""
    LP, LT, ub, at = [], [], [0], 0
    for b in range(k):
        if signs:
            u, s = 2 * b, 2 * b + 1
            assert s < n
            LP.append(1 << s)
            LT.append(1 << u)
            at = s + 1
        else:
            up = min(n, at + (first if b == 0 else 1 + (b & 1)))
            LP.append((((1 << up) - 1) ^ ((1 << at) - 1)) ^ (rnd.getrandbits(at) if at else 0))
            LT.append(0)
            at = up
        if b < 12:
            ub.append(at)
    if mode == 1:
        count = 1 << k
    recs = rec or [record(rnd, n, vanished=int(r % 7 == 5)) for r in range(count)]
    items = S.sweep_add(mode, n, k, signs, G, (ctypes.c_uint8 * 16)(*ub), (ctypes.c_uint64 * 32)(*map(word, LP)),
                        (ctypes.c_uint64 * 32)(*map(word, LT)), pairs, lds, count,
                        (ctypes.c_uint64 * (REC * count))(*[w for r in recs for w in r]))
    return {"n": n, "k": k, "G": G, "count": count, "recs": recs, "items": items}


def terms_of(S, insts, exact=False):
    """[instance][record, j] -> (eps, p, m); for exact sums the records' phases
    are set first so that <phi_r|Pi|phi_r> is positive, as it is in earnest"""
    out = []
    if exact:
        for i, t in enumerate(terms_of(S, insts)):
            for r in range(insts[i]["count"]):
                S.sweep_phase(i, r, -int(t[r, r, 2]))
    for i, d in enumerate(insts):
        t = np.zeros((d["count"], 1 << d["k"], 3), dtype=np.int32)
        for r in range(d["count"]):
            S.sweep_terms(i, r, ptr(t[r], ctypes.c_int))
        out.append(t)
    return out


def launch(S, mode, insts, nh, ht, grid, order, flush=1 << 30, copies=0):
    nrec, ni = sum(d["count"] for d in insts), len(insts)
    nt = sum(d["count"] << d["k"] if mode == 0 else (1 << d["k"]) * ((1 << d["k"]) + 1) // 2 for d in insts)
    n = 8 if copies else 1
    words = HIST + 3 * ni
    # kahan, counts and histograms in one block a copy, as the engine lays them out
    block = np.zeros(n * words, dtype=np.uint64)
    out = {"terms": np.full(nt, -7, dtype=np.int32), "zsum": np.zeros((nrec, 4), dtype=np.int64),
           "kahan": np.zeros((nrec, 2)), "hist": np.zeros((ni, HIST), dtype=np.uint64)}
    ips = np.zeros(ni, dtype=np.uint64)
    hist, kah, cnt = out["hist"], out["kahan"], ips
    if copies:
        hist, kah, cnt = block[:HIST], block[HIST:HIST + 2].view(np.float64), block[HIST + 2:HIST + 3]
    out["err"] = S.sweep_run(mode, nh, ht, copies, grid, (ctypes.c_int * 4)(*order), ctypes.c_longlong(flush),
                ptr(out["terms"], ctypes.c_int32), ptr(out["zsum"], ctypes.c_longlong), ptr(kah, ctypes.c_double),
                ptr(hist, ctypes.c_ulonglong), ptr(cnt, ctypes.c_ulonglong), words if copies else 0)
    if copies:
        b = block.reshape(n, words)
        out["hist"][0] = b[:, :HIST].sum(axis=0)
        ips[0] = b[:, HIST + 2].sum()
        out["kahan"] = b[:, HIST:HIST + 2].copy().view(np.float64).sum(axis=0)[None]
    out["ips"] = ips
    return out


# w^m in the basis 1, w, w^2, w^3, and sqrt2 w^m = w^{m+1} - w^{m+3}
def zomega(p, m):
    z = [0, 0, 0, 0]

    def add(q, v):
        z[q & 3] += -v if q & 4 else v
    v = 1 << (32 + (p >> 1))
    if p & 1:
        add((m + 1) & 7, v)
        add((m + 3) & 7, -v)
    else:
        add(m & 7, v)
    return z


def packed(t):
    return np.where(t[..., 0] == 1, -8 * t[..., 1] + t[..., 2] + 1, 0).astype(np.int32)


def check_sampled(out, insts, ref):
    assert out["err"] == 0
    at = tat = 0
    for d, t in zip(insts, ref):
        chi = 1 << d["k"]
        assert np.array_equal(out["terms"][tat:tat + d["count"] * chi], packed(t).reshape(-1))
        for r in range(d["count"]):
            want = np.sum([zomega(int(p), int(m)) for e, p, m in t[r] if e] or [[0] * 4], axis=0)
            assert np.array_equal(out["zsum"][at + r], want)
        at += d["count"]
        tat += d["count"] * chi


def hist_of(d, t):
    h = np.zeros(HIST, dtype=np.int64)
    for r in range(d["count"]):
        sexp = int(d["recs"][r][0] >> 24 & 0xffff)
        for j in range(r, 1 << d["k"]):
            e, p, m = (int(v) for v in t[r, j])
            if e:
                h[8 * (sexp - p) + m] += 1
                if j > r:
                    h[8 * (sexp - p) + (8 - m) % 8] += 1
    return h


def check_exact(out, insts, ref):
    assert out["err"] == 0
    terms = [packed(t)[np.triu_indices(1 << d["k"])] for d, t in zip(insts, ref)]
    assert np.array_equal(out["terms"], np.concatenate(terms))
    for i, (d, t) in enumerate(zip(insts, ref)):
        assert np.array_equal(out["hist"][i].astype(np.int64), hist_of(d, t))
        live = [r for r in range(d["count"]) if not d["recs"][r][0] >> 40 & 1]
        assert int(out["ips"][i]) == sum((1 << d["k"]) - r for r in live)


# one block, so one item from its own place and the others from the queue; the
# tables of both decompositions (of one wave, two and all four), pairs and not
CASES = [(2, 1, 0, 0, 1), (20, 5, 3, 0, 1), (20, 5, 3, 0, 0), (40, 6, 2, 0, 1), (52, 5, 4, 0, 1), (20, 5, 3, 1, 0),
         (44, 6, 3, 1, 0)]


def nh_of(n):
    return 0 if n <= 32 else 16 if n <= 48 else 32


@pytest.mark.parametrize("order", ORDERS)
@pytest.mark.parametrize("n,k,G,signs,pairs", CASES)
def test_sampled_sums_whatever_wave_is_first(S, n, k, G, signs, pairs, order):
    rnd = random.Random(1000 * n + 10 * k + signs)
    S.sweep_begin()
    d = [instance(S, rnd, 0, n, k, G, signs, pairs, count=70)]
    ref = terms_of(S, d)
    check_sampled(launch(S, 0, d, nh_of(n), signs, 1, order), d, ref)


@pytest.mark.parametrize("order", ORDERS)
@pytest.mark.parametrize("n,k,G,signs,pairs", CASES)
def test_exact_sums_whatever_wave_is_first(S, n, k, G, signs, pairs, order):
    rnd = random.Random(1100 * n + 10 * k + signs)
    S.sweep_begin()
    d = [instance(S, rnd, 1, n, k, G, signs, pairs)]
    ref = terms_of(S, d, exact=True)
    check_exact(launch(S, 1, d, nh_of(n), signs, 1, order), d, ref)


# several instances and items a block: partial sums move from item to item and
# are flushed between instances and after `flush` terms of one
@pytest.mark.parametrize("flush", [1, 1000, 1 << 30])
@pytest.mark.parametrize("grid", [1, 3, 50])
def test_claims_and_flushes(S, grid, flush):
    rnd = random.Random(7 * grid)
    S.sweep_begin()
    d = [instance(S, rnd, 1, 10, 5, 0), instance(S, rnd, 1, 9, 6, 1), instance(S, rnd, 1, 4, 1, 1, first=2)]
    assert d[-1]["items"] > 3
    ref = terms_of(S, d, exact=True)
    out = launch(S, 1, d, 0, 0, min(grid, d[-1]["items"]), ORDERS[grid % 3], flush)
    check_exact(out, d, ref)


def test_copies_add_up(S):
    rnd = random.Random(5)
    S.sweep_begin()
    d = [instance(S, rnd, 1, 12, 6, 0)]
    ref = terms_of(S, d, exact=True)
    check_exact(launch(S, 1, d, 0, 0, d[0]["items"], ORDERS[1], copies=1), d, ref)


# a record that no projection gives, with more summed slots than its state has
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n,extra", [(3, 3), (3, 29)])
def test_an_exponent_out_of_range_is_flagged_and_not_added(S, mode, n, extra):
    rnd = random.Random(9)
    S.sweep_begin()
    # every summed slot a factor 2: the term of index 0 has p = extra
    bad = [n << 8, word((1 << n + extra) - 1), 0, 0] + [0] * 64
    ok = record(rnd, n)
    d = [instance(S, rnd, mode, n, 1, 0, count=2, first=n, rec=[bad, ok])]
    ref = terms_of(S, d, exact=mode == 1)
    assert tuple(ref[0][0, 0][:2]) == (1, extra)
    out = launch(S, mode, d, 0, 0, 1, ORDERS[0])
    assert out["err"] == 2
    ref[0][0, ref[0][0, :, 1] > 0, 0] = 0
    if mode == 0:
        for r in range(2):
            want = np.sum([zomega(int(p), int(m)) for e, p, m in ref[0][r] if e] or [[0] * 4], axis=0)
            assert np.array_equal(out["zsum"][r], want)
    else:
        got = out["hist"][0].astype(np.int64)
        assert got.sum() == sum(2 * (j > r) + (j == r) for r in range(2) for j in range(r, 2) if ref[0][r, j, 0])


# What the FP32 sums may be off: a term is the FP32 number nearest to its value
# (2^-24 of it), and n additions lose at most about n^2 2^-48 of the sum of
# magnitudes besides.
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("n,k,G,signs", [(20, 8, 8, 0), (16, 8, 7, 1), (52, 7, 6, 0)])
def test_fp32_sums_carry_only_their_terms_rounding(S, mode, n, k, G, signs):
    rnd = random.Random(31 * n + k)
    S.sweep_begin()
    d = [instance(S, rnd, mode, n, k, G, signs, count=4, first=1)]
    ref = terms_of(S, d, exact=mode == 1)[0]
    out = launch(S, mode, d, nh_of(n), signs, 1, ORDERS[0])

    def of(p, m):  # the nearest FP32 numbers
        zero = (m % 4 == 2, m % 4 == 0)
        return tuple(0.0 if z else float(np.float32(2.0 ** (p / 2) * f(math.pi * m / 4)))
                     for z, f in zip(zero, (math.cos, math.sin)))

    tot = [0.0, 0.0, 0.0]
    for r in range(d[0]["count"]):
        if mode == 0:
            tot = [0.0, 0.0, 0.0]
        sexp = int(d[0]["recs"][r][0] >> 24 & 0xffff) if mode == 1 else 0
        vals = [tuple((1 + (mode == 1 and j > r)) * c for c in of(int(p) - sexp, int(m)))
                for j, (e, p, m) in enumerate(ref[r]) if e and (mode == 0 or j >= r)]
        tot = [math.fsum([tot[0]] + [v[0] for v in vals]), math.fsum([tot[1]] + [v[1] for v in vals]),
               math.fsum([tot[2]] + [max(map(abs, v)) for v in vals])]
        if mode == 0:
            for q in range(2):
                assert abs(out["kahan"][r, q] - tot[q]) <= (1 << 2 * G) * 2.0 ** -48 * tot[2]
    if mode == 1:
        assert abs(out["kahan"][0, 0] - tot[0]) <= (1 << 2 * G) * 2.0 ** -48 * tot[2]

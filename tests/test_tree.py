"""The sweep's per-lane exponential sums (csrc/cse_tree.h): on the CPU, the
same header compiled by g++ against a brute-force sum, at slot counts around
the 32-slot words and with dropped, multiplier and signed slots; the basis of
a decomposition's rows (cse_chain_basis); and on the GPU every term of small
sweeps against the oracle at the widths where the kernel changes, with trees
of different depths."""
import cmath
import ctypes
import math
import os
import random
import subprocess

import numpy as np
import pytest

import orc
from gpu_util import oracle_exact_terms, oracle_sampled, random_commuting_projector

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "circuitsimulator_amd", "csrc")
SHIM = r"""
#include "cse_tree.h"
#include <string.h>
using namespace cse::tree;
template <int NH, bool HT> static void go(int n, const uint64_t *row, const uint64_t *w, int *out) {
    Form<NH> f;
    memset(&f, 0, sizeof f);
    for (int x = 0; x < 32 + NH; x++) {
        f.lo[x] = x < n ? (u32)row[x] : 0;
        if (x >= 32) f.hi[x - 32] = x < n ? (u32)(row[x] >> 32) : 0;
    }
    f.d1 = (u32)w[0]; f.d2 = (u32)w[1]; f.A = (u32)w[2]; f.T = (u32)w[3];
    f.d1h = w[0] >> 32; f.d2h = w[1] >> 32; f.Ah = w[2] >> 32; f.Th = w[3] >> 32;
    int ph = 0, cnt = 0;
    if (NH) {
        StepsHi<NH, HT, NH - 1>::run(f, n);
        fold<HT>(f.d1h, f.d2h, f.Ah, f.Th, ~0u, ph, cnt);
    }
    const int low = n < 32 ? n : 32;
    steps<NH, HT>(f, low, low / 2);   // two stretches, as a tree's levels
    if (low / 2 > 0) steps<NH, HT>(f, low / 2, 0);
    fold<HT>(f.d1, f.d2, f.A, f.T, ~0u, ph, cnt);
    out[0] = (f.z >> 31) ? 0 : 1;
    out[1] = cnt - (int)f.nb - n;
    out[2] = (ph + 2 * (int)f.q1 + 4 * TREE_POP(f.x2)) & 7;
}
extern "C" void pair_eval(int c, const uint64_t *row, const uint64_t *w, int *out) {
    Form<0> f;
    memset(&f, 0, sizeof f);
    for (int x = 0; x < c; x++) f.lo[x] = (u32)row[x];
    f.d1 = (u32)w[0]; f.d2 = (u32)w[1]; f.A = (u32)w[2];
    PairSums s;
    pair_sums(f, c, s);
    for (int k = 0; k < 2; k++) {
        out[3 * k] = s.zero[k] ? 0 : 1;
        out[3 * k + 1] = s.cnt[k];
        out[3 * k + 2] = s.ph[k] & 7;
    }
}
extern "C" void tree_eval(int nh, int ht, int n, const uint64_t *row, const uint64_t *w, int *out) {
    if (nh == 0) ht ? go<0, true>(n, row, w, out) : go<0, false>(n, row, w, out);
    else if (nh == 16) ht ? go<16, true>(n, row, w, out) : go<16, false>(n, row, w, out);
    else ht ? go<32, true>(n, row, w, out) : go<32, false>(n, row, w, out);
}
"""


@pytest.fixture(scope="module")
def tree(tmp_path_factory):
    d = tmp_path_factory.mktemp("tree")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "shim.so"), str(d / "shim.cpp")],
                   check=True)
    return ctypes.CDLL(str(d / "shim.so"))


def words(v):
    """slot x of a mask at bit 31 - x of its half, as the header keeps it"""
    return sum(1 << (31 - x if x < 32 else 95 - x) for x in range(64) if v >> x & 1)


def brute(J, d1, d2, A, F, T):
    """The term as cse_tree.h defines it: the sum over the slots of A with
    (-1)^{T z}, the others at T; 2^{-1/2} per pivot slot and per summed
    coordinate, 1/2 per summed multiplier."""
    n = len(J)
    idx = [i for i in range(n) if A >> i & 1]
    tot = 0
    for m in range(1 << len(idx)):
        z = T & ~A
        for t, i in enumerate(idx):
            z |= (m >> t & 1) << i
        ph = 4 * bin(T & A & z).count("1")
        for i in range(n):
            if z >> i & 1:
                ph += 2 * (d1 >> i & 1) + 4 * (d2 >> i & 1) + 4 * bin(J[i] & z & ((1 << i) - 1)).count("1")
        tot += cmath.exp(1j * math.pi * (ph % 8) / 4)
    half = -(n - bin(F).count("1")) - bin(A ^ F).count("1") - 2 * bin(F & A).count("1")
    return tot * 2.0 ** (half / 2)


@pytest.mark.parametrize("nh,n", [(0, 1), (0, 2), (0, 31), (0, 32), (16, 33), (16, 47), (16, 48), (32, 49), (32, 63),
                                  (32, 64)])
@pytest.mark.parametrize("signs", [0, 1])
def test_form_sums_match_brute_force(tree, nh, n, signs):
    # up to 8 coupled slots anywhere among the n (the others empty and
    # dropped): every kind of step, partners on either side of slot 32
    rnd = random.Random(100 * n + signs)
    for _ in range(150):
        nv = rnd.randint(1, min(8, n))
        pos = sorted(rnd.sample(range(n), nv))
        dens = rnd.random()
        J = [0] * nv
        for a in range(nv):
            for b in range(a):
                if rnd.random() < dens:
                    J[a] |= 1 << b
                    J[b] |= 1 << a
        d1, d2, A, F = (rnd.getrandbits(nv) for _ in range(4))
        if rnd.random() < 0.4:
            d1 = 0
        T = rnd.getrandbits(nv) if signs else 0

        def up(v):
            return sum((v >> i & 1) << p for i, p in enumerate(pos))

        rows = (ctypes.c_uint64 * 64)()
        for i, p in enumerate(pos):
            rows[p] = words(up(J[i]))
        out = (ctypes.c_int * 3)()
        tree.tree_eval(nh, signs, n, rows, (ctypes.c_uint64 * 4)(*[words(up(v)) for v in (d1, d2, A, T)]), out)
        # the n - nv empty slots are pivots without a sum: 2^{-1/2} each
        got = out[0] * 2.0 ** ((out[1] + n - nv) / 2) * cmath.exp(1j * math.pi * out[2] / 4)
        assert abs(got - brute(J, d1, d2, A, F, T)) <= 1e-9


@pytest.mark.parametrize("c", [1, 2, 3, 4, 5, 8, 9, 12, 16, 17, 18, 31, 32])
def test_two_complementary_terms_match_brute_force(tree, c):
    # up to 9 coupled slots, on both sides of the cut, among the c
    rnd = random.Random(77 * c)
    for _ in range(300):
        nv = min(c, rnd.randint(1, 9))
        pos = sorted(rnd.sample(range(c), nv))
        dens = rnd.random()
        J = [0] * nv
        for a in range(nv):
            for b in range(a):
                if rnd.random() < dens:
                    J[a] |= 1 << b
                    J[b] |= 1 << a
        d1, d2, A = (rnd.getrandbits(nv) for _ in range(3))
        if rnd.random() < 0.5:
            d1 = 0

        def up(v):
            return sum((v >> i & 1) << p for i, p in enumerate(pos))

        rows = (ctypes.c_uint64 * 64)()
        for i, p in enumerate(pos):
            rows[p] = words(up(J[i]))
        out = (ctypes.c_int * 6)()
        tree.pair_eval(c, rows, (ctypes.c_uint64 * 4)(*[words(up(v)) for v in (d1, d2, A, 0)]), out)
        for k in range(2):
            a = ~A & ((1 << nv) - 1) if k else A
            # the c - nv empty slots: 2^{-1/2} each where dropped, 1 where summed
            got = out[3 * k] * 2.0 ** ((out[3 * k + 1] - c) / 2) * cmath.exp(1j * math.pi * out[3 * k + 2] / 4)
            want = brute(J, d1, d2, a, 0, 0) * (1.0 if k else 2.0 ** (-(c - nv) / 2))
            assert abs(got - want) <= 1e-9


@pytest.mark.parametrize("t,k", [(1, 0), (1, 1), (2, 3), (13, 5), (24, 11), (48, 12), (64, 14), (60, 20)])
def test_chain_basis_keeps_the_span(t, k):
    from circuitsimulator_amd.engine import lib
    rnd = random.Random(t * 100 + k)
    for kind in range(4):
        L = [rnd.getrandbits(t) for _ in range(k)]
        if kind == 1 and k > 2:
            L[1] = L[0] ^ L[2]
        if kind == 2 and k:
            L[0] = 0
        rows, jmap = (ctypes.c_uint64 * 32)(), (ctypes.c_uint32 * 32)()
        ub, col = (ctypes.c_uint8 * 16)(), (ctypes.c_uint8 * 64)()
        lib().cse_chain_basis(t, k, (ctypes.c_uint64 * 32)(*L), 12, rows, jmap, ub, col)
        assert sorted(col[:t]) == list(range(t))
        moved, reduced = 0, []
        for g in range(k):
            x = 0
            for b in range(k):
                if jmap[g] >> b & 1:
                    x ^= L[k - 1 - b]
            assert x == rows[g]
            moved |= x
            if g < 12:
                assert sorted(col[:ub[g + 1]]) == [q for q in range(t) if moved >> q & 1]
            v = jmap[g]
            for r in reduced:
                v = min(v, v ^ r)
            assert v
            reduced.append(v)


@pytest.fixture(scope="module")
def E():
    from circuitsimulator_amd import Engine
    e = Engine(0)
    yield e
    e.close()


# widths on either side of each kernel's limit; chunk bounds a lane's terms
@pytest.mark.gpu
@pytest.mark.parametrize("t,k,exact", [(2, 1, 0), (31, 5, 0), (32, 4, 0), (33, 5, 0), (48, 5, 0), (49, 4, 0),
                                       (64, 5, 0), (9, 0, 1), (10, 0, 1)])
def test_every_sampled_term_at_the_kernels_widths(E, t, k, exact):
    from circuitsimulator_amd.engine import Projector
    rng = np.random.default_rng(31 * t + k)
    ph, xs, zs = random_commuting_projector(rng, t, max(1, t // 3))
    L = [] if exact else [orc.rand_bits(rng, t) for _ in range(k)]
    chi = 1 << ((t + 1) // 2) if exact else 1 << k
    se, zsum, terms = oracle_sampled(t, k, L, exact, ph, xs, zs, 5, 0, 3, chi)
    P = Projector.make(ph, xs, zs, t)
    for chunk in (0, 1, 4, chi):
        print(f"sampled t={t} k={k} exact={exact} chunk={chunk}", flush=True)
        _, ex = E.sampled_projector(P, L, k, exact, 5, 0, 3, chunk=chunk, want_terms=True)
        assert np.array_equal(ex["sexp"], se)
        assert np.array_equal(ex["terms"], terms)
        assert np.array_equal(ex["zsum"], zsum)


@pytest.mark.gpu
@pytest.mark.parametrize("t,k,exact", [(2, 1, 0), (32, 4, 0), (33, 4, 0), (48, 4, 0), (49, 4, 0), (64, 4, 0),
                                       (9, 0, 1), (10, 0, 1)])
def test_every_exact_term_at_the_kernels_widths(E, t, k, exact):
    from circuitsimulator_amd.engine import Instance, Projector
    rng = np.random.default_rng(37 * t + k)
    ph, xs, zs = random_commuting_projector(rng, t, max(1, t // 3))
    L = [] if exact else [orc.rand_bits(rng, t) for _ in range(k)]
    inst = Instance()
    inst.P = Projector.make(ph, xs, zs, t)
    inst.exact, inst.k = exact, k
    for i, v in enumerate(L):
        inst.L[i] = v
    chi = 1 << ((t + 1) // 2) if exact else 1 << k
    nl = chi * (chi + 1) // 2
    want = [w[0] for w in oracle_exact_terms(t, k, L, exact, ph, xs, zs)]
    for chunk in (0, 1, 4, chi):
        print(f"exact t={t} k={k} exact={exact} chunk={chunk}", flush=True)
        _, terms, _ = E.batch_exact([inst], chunk=chunk, want_terms=True, nterms=nl)
        assert want == list(terms)


# levels beyond 32 slots: rows that reach them one, two and many slots at a
# time, next to narrower instances in the same launch
@pytest.mark.gpu
@pytest.mark.parametrize("t,steps", [(49, [30, 2, 1, 16]), (56, [8, 20, 10, 9, 8]), (64, [33, 1, 15, 15]),
                                     (63, [3, 28, 1, 1, 17]), (64, [2, 40, 21])])
def test_levels_beyond_32_slots(E, t, steps):
    from circuitsimulator_amd.engine import Instance, Projector
    rng = np.random.default_rng(41 * t + len(steps))
    order = rng.permutation(t)
    L, at = [], 0
    for s in steps:
        # s new columns and some of the ones before
        L.append(sum(1 << int(q) for q in order[at:at + s]) ^ (orc.rand_bits(rng, t) & sum(1 << int(q) for q in order[:at])))
        at += s
    k = len(L)
    ph, xs, zs = random_commuting_projector(rng, t, t // 3)
    se, zsum, terms = oracle_sampled(t, k, L, 0, ph, xs, zs, 5, 0, 3, 1 << k)
    P = Projector.make(ph, xs, zs, t)
    for chunk in (0, 4, 1 << k):
        print(f"t={t} steps={steps} chunk={chunk}", flush=True)
        _, ex = E.sampled_projector(P, L, k, 0, 5, 0, 3, chunk=chunk, want_terms=True)
        assert np.array_equal(ex["sexp"], se)
        assert np.array_equal(ex["terms"], terms)
        assert np.array_equal(ex["zsum"], zsum)
    inst, want = [], []
    for n, rows in ((t, L), (9, [3, 500, 77])):
        i = Instance()
        p = (ph, xs, zs) if n == t else random_commuting_projector(rng, n, 3)
        i.P = Projector.make(*p, n)
        i.exact, i.k = 0, len(rows)
        for q, v in enumerate(rows):
            i.L[q] = v
        inst.append(i)
        want += [w[0] for w in oracle_exact_terms(n, len(rows), rows, 0, *p)]
    for chunk in (0, 1 << k):
        _, got, _ = E.batch_exact(inst, chunk=chunk, want_terms=True, nterms=len(want))
        assert want == list(got)

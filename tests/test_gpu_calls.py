"""Calls on one context, one after the other: partial sums flushed within an
instance, and results that come back in each of the three ways (polled for,
in kernel stores, in a copy), whatever the call before was."""
import numpy as np
import pytest

from circuitsimulator_amd import Engine
from circuitsimulator_amd.engine import Instance, Projector
from circuitsimulator_amd.workloads import commuting_paulis, random_L
from gpu_util import oracle_exact_terms

pytestmark = pytest.mark.gpu


def drawn(t, k, r, seed):
    rng = np.random.default_rng(seed)
    return Projector.make(*commuting_paulis(rng, t, r), t), random_L(rng, t, k)


def test_flushes_within_an_instance(monkeypatch):
    """One term a lane gives each block some 30 items of one instance; with
    bounds below that it adds its sums to the global ones in between."""
    P, L = drawn(24, 12, 12, 7)
    inst = Instance()
    inst.P = P
    inst.k = 12
    for i, v in enumerate(L):
        inst.L[i] = v
    chi = 1 << 12
    lanes = chi * (chi + 1) // 2
    got = {}
    for bound in (None, "64", "1000", "5000"):
        monkeypatch.delenv("CSE_FLUSH_TERMS", raising=False)
        if bound:
            monkeypatch.setenv("CSE_FLUSH_TERMS", bound)
        with Engine(0) as E:
            assert lanes // 256 > 20 * 4 * E.device_info()[0]
            (r,), _, _ = E.batch_exact([inst], chunk=1)
            (deep,), _, _ = E.batch_exact([inst])
        print(f"CSE_FLUSH_TERMS={bound}", flush=True)
        got[bound] = (r.re, r.im, r.ips)
        assert got[bound] == (deep.re, deep.im, deep.ips) and r.terms == lanes
        # FP32 terms of at most 2^-24 relative error, signs at random
        assert abs(r.kahan_re - r.re) <= 1e-5 * abs(r.re)
    assert len(set(got.values())) == 1


@pytest.mark.parametrize("t,r,k", [(33, 1, 0), (49, 3, 1), (64, 1, 0), (64, 5, 2), (64, 40, 1)])
def test_slots_without_rows(t, r, k):
    """Few generators leave most slots without a row in any lane, whose steps
    end early: every pair term against the oracle."""
    rng = np.random.default_rng(10 * t + r)
    ph, xs, zs = commuting_paulis(rng, t, r)
    L = random_L(rng, t, k) if k else []
    inst = Instance()
    inst.P = Projector.make(ph, xs, zs, t)
    inst.k = k
    for i, v in enumerate(L):
        inst.L[i] = v
    chi = 1 << k
    with Engine(0) as E:
        (res,), terms, _ = E.batch_exact([inst], want_terms=True, nterms=chi * (chi + 1) // 2)
    want = oracle_exact_terms(t, k, L, 0, ph, xs, zs)
    assert [w[0] for w in want] == list(terms)
    assert res.im == 0.0


def test_results_of_every_size_on_one_context():
    """Sizes on both sides of 1 MB and of 64 MB, with per-term calls and exact
    ones between them: each as on a context of its own."""
    calls = [(24, 9, 300, False), (13, 4, 40000, False), (9, 3, 1, False), (4, 1, 1400000, False),
             (24, 9, 300, True), (40, 8, 20000, False), (4, 1, 1400000, False), (64, 6, 17, False)]

    def sampled(E, i, t, k, count, terms):
        P, L = drawn(t, k, max(1, t // 3), 50 + i)
        r, x = E.sampled_projector(P, L, k, 0, 11 + i, 5, count, want_terms=terms)
        return (r.mean, r.ips, r.vanished), [x[n] for n in ("zsum", "sexp", "terms") if n in x]

    def exact(E, i, t, k):
        P, L = drawn(t, k, t // 2, 90 + i)
        r, h = E.exact_projector(P, L, k, 0, want_hist=i % 2 == 0)
        return (r.re, r.im, r.ips), [h] if h is not None else []

    def same(a, b):
        assert a[0] == b[0] and len(a[1]) == len(b[1])
        for x, y in zip(a[1], b[1]):
            assert np.array_equal(x, y)

    with Engine(0) as E:
        for i, c in enumerate(calls):
            print("call", i, c, flush=True)
            with Engine(0) as F:
                same(sampled(E, i, *c), sampled(F, i, *c))
            with Engine(0) as F:
                same(exact(E, i, 10 + 6 * i, 3 + i), exact(F, i, 10 + 6 * i, 3 + i))

"""Exact values whose sums are formed on the device (calls that do not ask
for the histogram) against cse_hist_value of the histogram: the same bits."""
import ctypes

import numpy as np
import pytest

from circuitsimulator_amd import Engine
from circuitsimulator_amd.engine import Instance, Projector, _ptr, instance_array, lib
from circuitsimulator_amd.workloads import commuting_paulis, random_L

PMIN = -128
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def E():
    with Engine(0) as e:
        yield e


def host_value(hist):
    re, im = ctypes.c_double(), ctypes.c_double()
    lib().cse_hist_value(_ptr(np.ascontiguousarray(hist, dtype=np.int64), ctypes.c_int64), PMIN,
                         ctypes.byref(re), ctypes.byref(im))
    return re.value, im.value


def drawn(t, k, r, seed):
    rng = np.random.default_rng(seed)
    return commuting_paulis(rng, t, r), random_L(rng, t, k)


@pytest.mark.parametrize("t,k,r", [(2, 1, 1), (9, 4, 3), (13, 5, 5), (33, 7, 16), (48, 9, 24), (64, 6, 1), (64, 8, 32)])
def test_single_L(E, t, k, r):
    (ph, xs, zs), L = drawn(t, k, r, 100 * t + k)
    P = Projector.make(ph, xs, zs, t)
    _, hist = E.exact_projector(P, L, k, 0, want_hist=True)
    res = E.exact_projector(P, L, k, 0)
    res = res[0] if isinstance(res, tuple) else res
    assert (res.re, res.im) == host_value(hist)


@pytest.mark.parametrize("t,r", [(1, 1), (7, 2), (16, 8), (21, 3)])
def test_single_H(E, t, r):
    (ph, xs, zs), _ = drawn(t, 0, r, t)
    P = Projector.make(ph, xs, zs, t)
    _, hist = E.exact_projector(P, [], 0, 1, want_hist=True)
    res = E.exact_projector(P, [], 0, 1)
    res = res[0] if isinstance(res, tuple) else res
    assert (res.re, res.im) == host_value(hist)


@pytest.mark.parametrize("count", [2, 3, 5, 67, 600])
def test_batches(E, count):
    """Counts that leave a wave idle, one wave and several blocks; one
    instance's projector (Z and -Z on a qubit) has no terms at all."""
    A = instance_array(count)
    want = np.zeros(count)
    for i in range(count):
        t, k = 4 + i % 37, 1 + i % 5
        (ph, xs, zs), L = drawn(t, min(k, t - 1), 1 + i % (t // 2), 1000 + i)
        if i == 1:
            ph, xs, zs = [0, 2], [0, 0], [1, 1]
        inst = Instance()
        inst.P = Projector.make(ph, xs, zs, t)
        inst.k = len(L)
        for b, v in enumerate(L):
            inst.L[b] = v
        A[i] = np.frombuffer(bytes(inst), dtype=A.dtype)[0]
        if i < 40:
            _, hist = E.exact_projector(inst.P, L, len(L), 0, want_hist=True)
            want[i] = np.hypot(*host_value(hist))
    vals, _ = E.batch_exact_values(A)
    assert np.array_equal(vals[:40], want[:40])
    assert vals[1] == 0.0


@pytest.mark.parametrize("t,k", [(24, 9), (24, 10), (40, 10), (50, 11)])
def test_copies_of_the_sums(E, t, k):
    """Calls of 256 blocks and more add to copies of the histogram: the same
    histogram, count and value as the call in the library's static array,
    which has one copy."""
    (ph, xs, zs), L = drawn(t, k, t // 3, t + k)
    P = Projector.make(ph, xs, zs, t)
    a, ha = E.exact_projector(P, L, k, 0, want_hist=True)
    b, hb = E.exact_projector_noalloc(P, L, k, 0, want_hist=True)
    c, _ = E.exact_projector(P, L, k, 0)
    assert np.array_equal(ha, hb) and a.ips == b.ips == c.ips == a.terms
    assert (a.re, a.im) == (b.re, b.im) == (c.re, c.im) == host_value(ha)
    assert abs(a.kahan_re - b.kahan_re) <= 1e-5 * abs(a.re)

"""The Morton sorts at the edges of their runs (512 keys, 16 runs, 16 x 16 runs and one more,
which the library sort takes): forces with sorted and unsorted i agree, the j-set holds every
particle once (FP64 oracle), and equal keys (a far escaper that makes the key cells wide,
repeated i) do no harm."""
import numpy as np
import pytest

import oracle as O
from helpers import vec_rel_err
from nb6 import ics, lib

pytestmark = pytest.mark.gpu
SIZES = [2, 512, 513, 8192, 8193, 131072, 131073]


@pytest.mark.parametrize("n", SIZES)
def test_sorted_sets_give_the_unsorted_results(n):
    m, x, v = ics.plummer(n, seed=n, masses=ics.kroupa_masses(n, 1))
    x[n - 1] = 1.0e5                        # key cells of 0.05
    src = np.arange(n) // 2                 # every i twice
    xi, vi = x[src].copy(), v[src].copy()
    h2, dtr = np.full(n, 1.0e-3), np.full(n, 2.0 ** -7)
    L = lib.load()
    g = lib.Gpunb(n)
    try:
        g.send(m, x, v)
        out = []
        for isort in (0, 1):
            assert L.nb6_set_regf_tuning(isort, 1) == 0
            out.append(g.regf(h2, dtr, xi, vi, 40, 35))
    finally:
        L.nb6_set_regf_tuning(2048, 1)
        g.close()
    (a0, j0, p0, l0), (a1, j1, p1, l1) = out
    assert np.array_equal(l0, l1)
    # the same pairs in FP32, summed in FP64 in another order
    assert vec_rel_err(a1, a0).max() <= 1e-10 and vec_rel_err(j1, j0).max() <= 1e-10
    assert (np.abs(p1 - p0) <= 1e-12 * p0).all()
    k = np.linspace(0, n - 1, min(n, 40)).astype(int)
    acc, _, pot, lst = O.regf(m, x, v, h2[k], dtr[k], xi[k], vi[k], 40, 35)
    assert np.array_equal(l1[k], lst)
    assert vec_rel_err(a1[k], acc).max() <= 1e-6
    assert (np.abs(p1[k] - pot) <= 1e-6 * pot).all()


def test_ordered_irregular_calls_give_the_same_bits():
    n = 3000
    m, x, v = ics.plummer(n, seed=4)
    rng = np.random.default_rng(3)
    L = lib.load()
    g, irr = lib.Gpunb(n), lib.IrrSimd(n, 64)
    try:
        g.send(m, x, v)
        for i in range(n):
            irr.set_jp(i + 1, x[i], v[i], 0.1 * v[i], 0.01 * v[i], m[i], 0.0)
            row = rng.choice(n - 1, 20, replace=False)
            irr.set_list(i + 1, np.r_[20, row + (row >= i) + 1])
        for ni in SIZES[3:] + [2048]:
            addr = rng.integers(1, n + 1, ni).astype(np.int32)
            out = []
            for order in (0, 1):
                assert L.nb6_set_irr_config(64, order) == 0
                out.append(irr.firr_vec(0.0078125, addr))
            for a, b in zip(*out):
                assert np.array_equal(a, b)
    finally:
        L.nb6_set_irr_config(64, 1)
        irr.close()
        g.close()

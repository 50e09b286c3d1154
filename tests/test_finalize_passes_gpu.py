"""The finalize's passes over 64 candidates at counts around the pass edges (hard, soft and both),
in one wavefront per i (all j in one chunk) and in four and eight (further j far away)."""
import numpy as np
import pytest

import oracle as O
from helpers import vec_rel_err
from nb6 import lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("far, ni", [(0, 9), (6000, 9), (6000, 2100)])
@pytest.mark.parametrize("hard, soft", [(1, 0), (1, 63), (63, 0), (64, 0), (65, 0), (60, 5), (64, 64),
                                        (100, 29), (1, 192), (200, 120)])
def test_candidate_counts_around_a_pass(hard, soft, far, ni):
    rng = np.random.default_rng(1000 * hard + soft)

    def shell(n, lo, hi):
        d = rng.normal(size=(n, 3))
        return d / np.linalg.norm(d, axis=1)[:, None] * rng.uniform(lo, hi, (n, 1))
    # i at the origin within 1e-3: hard candidates inside R = 1, soft ones between R and 2 R
    x = np.concatenate([shell(hard, 0.05, 0.9), shell(soft, 1.1, 1.9), shell(far, 50.0, 60.0)])
    n = len(x)
    v = rng.normal(size=(n, 3)) * 0.1
    m = rng.uniform(0.5, 1.5, n) / n
    xi, vi = rng.uniform(-1e-3, 1e-3, (ni, 3)), rng.normal(size=(ni, 3)) * 0.1
    h2, dtr = np.full(ni, 1.0), np.full(ni, 2.0 ** -10)
    g = lib.Gpunb(max(n, 16))
    try:
        g.send(m, x, v)
        acc, jrk, pot, lst = g.regf(h2, dtr, xi, vi, 300, 250)
    finally:
        g.close()
    k = np.arange(0, ni, max(1, ni // 50))
    racc, rjrk, rpot, rlst = O.regf(m, x, v, h2[k], dtr[k], xi[k], vi[k], 300, 250)
    assert np.array_equal(lst[k, 0], rlst[:, 0]) and (lst[:, 0] == hard).all()
    assert np.array_equal(lst[k, 1:hard + 1], rlst[:, 1:hard + 1])
    if soft + far:
        # soft pairs are summed in FP64, far ones in FP32
        tol = 1e-6 if far else 1e-13
        assert vec_rel_err(acc[k], racc).max() <= tol * 100
        assert (np.abs(pot[k] - rpot) / rpot).max() <= tol

"""The finalize stage of the regular force at the sizes where it changes form (one, four or
eight wavefronts per i; one chunk, 64 chunks and more per pass) and with rows that hold from
none to several passes of 64 candidates: lists equal to the FP64 oracle's, acc and pot within
1e-6 of it; with the FP64 pair kernel, which feeds the same stage, acc, jerk and pot within
1e-9 (40,000 terms, 2^-53 each, 200-fold cancellation)."""
import numpy as np
import pytest

import oracle as O
from helpers import vec_rel_err
from nb6 import ics, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ni,m_flag,nnbmax", [
    (200, 200, 0, 150),          # one chunk
    (1000, 37, 0, 350),
    (9000, 2048, 0, 200), (9000, 2049, 0, 200),
    (9000, 2048, 1, 200), (3000, 3000, 1, 300),
    (4500, 16384, 0, 200), (4500, 16385, 0, 200),
    (40000, 300, 0, 0), (40000, 300, 0, 1), (40000, 5, 0, 1500),
])
def test_finalize_forms(n, ni, m_flag, nnbmax):
    rng = np.random.default_rng(n + ni)
    m, x, v = ics.plummer(n, seed=n, masses=ics.kroupa_masses(n, 1))
    idx = rng.choice(n, size=ni, replace=ni > n)
    cnt = np.clip(np.exp(rng.normal(np.log(60.0), 0.8, ni)), 1, 0.4 * n)
    cnt[: ni // 8] = 1.0
    dens = np.sqrt(1.0 + (x[idx] ** 2).sum(1) / 0.35) ** -5 * n * 0.7
    h2 = (3.0 * cnt / (4.0 * np.pi * dens)) ** (2.0 / 3.0)
    h2 = np.minimum(h2, 0.3 + 0.1 * (x[idx] ** 2).sum(1))
    if m_flag:
        h2 = h2 / m.mean()
    dtr = np.exp(rng.uniform(np.log(2.0 ** -9), np.log(2.0 ** -4), ni))
    lmax = max(nnbmax + 1, 2)
    xi, vi = x[idx].copy(), v[idx].copy()
    g = lib.Gpunb(n)
    try:
        g.send(m, x, v)
        runs = []
        for prec in (0, 2):
            g.L.nb6_set_regf_precision(prec)
            runs.append(g.regf(h2, dtr, xi, vi, lmax, nnbmax, m_flag))
    finally:
        g.L.nb6_set_regf_precision(0)
        g.close()
    racc, rjrk, rpot, rlst = O.regf(m, x, v, h2, dtr, xi, vi, lmax, nnbmax, m_flag)
    for (acc, jrk, pot, lst), tol in zip(runs, (1e-6, 1e-9)):
        assert np.array_equal(lst[:, 0], rlst[:, 0])
        for a, b in zip(lst, rlst):
            c = max(int(b[0]), 0)
            assert np.array_equal(a[1:c + 1], b[1:c + 1])
        assert vec_rel_err(acc, racc).max() <= tol
        assert (np.abs(pot - rpot) / rpot).max() <= tol
    assert vec_rel_err(runs[1][1], rjrk).max() <= 1e-9

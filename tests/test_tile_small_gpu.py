"""The regular force's form for small calls (64 i per work-group, the pieces of a tile side by
side) against the 256-wide form on the same particles: without the FP64 pass the FP32 partial
sums are the same bits, so forces agree to the rounding of their FP64 sums (2000 partial sums
of 2^-53 each with 200-fold cancellation: 5e-11); lists are equal, overflowing rows too."""
import numpy as np
import pytest

from helpers import vec_rel_err
from nb6 import ics, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ni,m_flag,nnbmax,big", [
    (4096, 1, 0, 350, 0.0), (5000, 63, 0, 350, 0.0), (5001, 64, 1, 350, 0.0),
    (5333, 65, 0, 350, 0.1), (60000, 250, 0, 350, 0.02), (60000, 130, 1, 60, 0.05),
    (9000, 300, 0, 3, 0.3),
])
def test_small_form_equals_wide_form(n, ni, m_flag, nnbmax, big):
    rng = np.random.default_rng(n + ni)
    m, x, v = ics.plummer(n, seed=n, masses=ics.kroupa_masses(n, 2))
    m, x, v = ics.add_binaries(m, x, v, 0.3, n)
    nw = 70000                                   # the wide call's i-set
    idx = rng.integers(0, n, nw)
    rs = 0.5 * (40.0 / n) ** (1.0 / 3.0) * np.exp(rng.normal(0, 0.4, nw)) * (1 + (x[idx] ** 2).sum(1))
    # some rows with far more neighbours than slots
    rs = np.where(rng.uniform(size=nw) < big, 0.6, np.minimum(rs, 0.4))
    h2 = rs * rs / (m.mean() if m_flag else 1.0)
    dtr = np.exp(rng.uniform(np.log(2.0 ** -9), np.log(2.0 ** -4), nw))
    xi, vi = x[idx].copy(), v[idx].copy()
    pick = np.sort(rng.choice(nw, ni, replace=False))
    g = lib.Gpunb(n)
    try:
        g.L.nb6_set_regf_refine(0)
        g.send(m, x, v)
        wide = g.regf(h2, dtr, xi, vi, nnbmax + 1, nnbmax, m_flag)
        small = g.regf(h2[pick], dtr[pick], xi[pick].copy(), vi[pick].copy(), nnbmax + 1, nnbmax,
                       m_flag)
    finally:
        g.L.nb6_set_regf_refine(1)
        g.close()
    for a, b in zip(small[3], wide[3][pick]):
        c = max(int(b[0]), 0)
        assert a[0] == b[0] and np.array_equal(a[1:c + 1], b[1:c + 1])
    # rows whose soft slots fill up keep different near pairs in their FP32 sums where the
    # chunks differ; the others have the same FP32 terms
    few = np.abs(wide[3][pick][:, 0]) < 20
    assert few.any() or ni < 2
    assert vec_rel_err(small[0][few], wide[0][pick][few]).max(initial=0.0) <= 5e-11
    assert vec_rel_err(small[1][few], wide[1][pick][few]).max(initial=0.0) <= 5e-11
    assert vec_rel_err(small[0], wide[0][pick]).max() <= 1e-6

"""Rows whose soft slots are full long before their chunk ends: later tiles are tested for hard
pairs only. The far-tile test on or off and one or two i per lane give the same bits, lists are
the FP64 kernel's, forces within its bar."""
import numpy as np
import pytest

from helpers import vec_rel_err
from nb6 import ics, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m_flag", [0, 1])
@pytest.mark.parametrize("n, ni, nnb, nnbmax, threads", [
    (20000, 300, 400, 1500, 256),         # soft slots full, every list found
    (20000, 300, 400, 1500, 512),
    (20001, 130, 4000, 60, 256),          # and hard slots
    (1025, 200, 500, 1000, 128),          # the shortest chunk with that test: one tile and a record
    (30011, 70000, 300, 900, 0),          # the form of large calls
])
def test_full_soft_slots(n, ni, nnb, nnbmax, threads, m_flag):
    m, x, v = ics.plummer(n, seed=n, masses=ics.kroupa_masses(n, 3))
    rng = np.random.default_rng(ni + nnb)
    idx = rng.integers(0, n, ni)
    a = 3.0 * np.pi / 16.0                # radius of about nnb neighbours in a Plummer sphere
    rs = a * (nnb / n) ** (1 / 3) * (1.0 + (x[idx] ** 2).sum(1) / a**2) ** (5 / 6)
    h2 = rs * rs * rng.uniform(0.3, 1.2, ni) / (m.mean() if m_flag else 1.0)
    dtr = 2.0 ** rng.integers(-10, -4, ni).astype(float)
    L = lib.load()
    g = lib.Gpunb(n)
    got = []
    lmax = nnbmax + 1
    try:
        g.send(m, x, v)
        for far, ipl in ((1, 1), (0, 1), (1, 2)):
            assert L.nb6_set_regf_config(threads, ipl, 1) == 0
            assert L.nb6_set_regf_tuning(2048, far) == 0
            got.append(g.regf(h2, dtr, x[idx].copy(), v[idx].copy(), lmax, nnbmax, m_flag))
            assert L.nb6_last_regf_chunks() == 1
        L.nb6_set_regf_precision(2)
        ref = g.regf(h2, dtr, x[idx].copy(), v[idx].copy(), lmax, nnbmax, m_flag)
    finally:
        L.nb6_set_regf_precision(0)
        L.nb6_set_regf_tuning(2048, 1)
        L.nb6_set_regf_config(0, 1, 4096)
        g.close()
    for other in got[1:]:
        for q, w in zip(got[0], other):
            assert np.array_equal(q, w, equal_nan=q.dtype.kind == "f")
    full = ref[3][:, 0] >= 0              # (overflowing counts: band pairs have few slots)
    assert full.any() == (nnbmax > nnb) and np.array_equal(got[0][3][:, 0] >= 0, full)
    c = np.maximum(ref[3][:, 0], 0)[:, None]
    keep = np.arange(lmax - 1)[None] < c
    assert np.array_equal(got[0][3][full, 0], ref[3][full, 0])
    assert np.array_equal(np.where(keep, got[0][3][:, 1:], 0)[full], np.where(keep, ref[3][:, 1:], 0)[full])
    assert vec_rel_err(got[0][0], ref[0]).max() <= 1e-6
    assert vec_rel_err(got[0][2], ref[2]).max() <= 1e-6

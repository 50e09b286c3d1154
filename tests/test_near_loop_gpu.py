"""The loop with the neighbour test in one i per lane (its own code) against two i per lane
(pair by pair): the same bits, with rows whose hard or soft slots fill up, and j-sets that end inside
a 64-j piece."""
import numpy as np
import pytest

from nb6 import ics, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m_flag", [0, 1])
@pytest.mark.parametrize("threads", [128, 512])
@pytest.mark.parametrize("n, ni, nnb, nnbmax", [
    (40, 40, 10, 30),            # less than one piece
    (1000, 200, 30, 150),
    (1000, 200, 60, 3),          # hard slots fill up
    (6001, 130, 700, 900),       # soft slots fill up
    (6001, 130, 1500, 20),       # both
])
def test_one_and_two_i_per_lane_give_the_same_bits(n, ni, nnb, nnbmax, threads, m_flag):
    m, x, v = ics.plummer(n, seed=n)
    m = m * np.exp(np.random.default_rng(2).normal(0.0, 1.0, n))
    rng = np.random.default_rng(n + nnb)
    idx = rng.choice(n, ni, replace=False)
    d = np.sort(((x[idx, None] - x[None]) ** 2).sum(2), axis=1)
    h2 = d[:, min(nnb, n - 1)] * rng.uniform(0.5, 1.0, ni)
    if m_flag:
        h2 = h2 / m.mean()
    dtr = 2.0 ** rng.integers(-10, -4, ni).astype(float)
    L = lib.load()
    g = lib.Gpunb(n)
    got = []
    try:
        for ipl in (1, 2):
            assert L.nb6_set_regf_config(threads, ipl, 1) == 0
            g.send(m, x, v)
            got.append(g.regf(h2, dtr, x[idx].copy(), v[idx].copy(), 1001, nnbmax, m_flag))
    finally:
        L.nb6_set_regf_config(0, 1, 4096)
        g.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f")
    if nnbmax < nnb / 4:
        assert (got[0][3][:, 0] < 0).any()

"""The loop for tiles far from every i of a wavefront against the loop with the neighbour test
(far_test off): the same bits, at j-sets that end inside a tile, a 64-j piece and a round of 16."""
import numpy as np
import pytest

import oracle as O
from helpers import vec_rel_err
from nb6 import ics, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m_flag", [0, 1])
@pytest.mark.parametrize("threads", [0, 128, 256, 512])
@pytest.mark.parametrize("n", [1, 15, 65, 257, 1031])
def test_far_loop_gives_the_bits_of_the_test_loop(n, threads, m_flag):
    # 256-wide work-groups take the form for small calls below 1793 pieces of 64 i
    ni = 64 * 1793 + 7 if threads == 256 else 301
    m, x, v = ics.plummer(max(n, 4), seed=n)
    m, x, v = m[:n].copy(), x[:n].copy(), v[:n].copy()
    rng = np.random.default_rng(n)
    xi = 40.0 + rng.uniform(-1.0, 1.0, (ni, 3))        # every tile is far
    vi = rng.uniform(-1.0, 1.0, (ni, 3))
    h2, dtr = np.full(ni, 0.01), np.full(ni, 2.0 ** -6)
    L = lib.load()
    g = lib.Gpunb(max(n, 16))
    try:
        assert L.nb6_set_regf_config(threads, 1, 4096) == 0
        g.send(m, x, v)
        got = []
        for far in (1, 0):
            assert L.nb6_set_regf_tuning(2048, far) == 0
            got.append(g.regf(h2, dtr, xi, vi, 200, 150, m_flag))
    finally:
        L.nb6_set_regf_tuning(2048, 1)
        L.nb6_set_regf_config(0, 1, 4096)
        g.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    acc, jrk, pot, lst = got[0]
    k = np.arange(0, ni, max(1, ni // 300))
    racc, rjrk, rpot, rlst = O.regf(m, x, v, h2[k], dtr[k], xi[k], vi[k], 200, 150, m_flag)
    assert np.array_equal(lst[k, 0], rlst[:, 0])
    assert vec_rel_err(acc[k], racc).max() <= 1e-6
    assert (np.abs(pot[k] - rpot) / rpot).max() <= 1e-6

"""Ragged i-sets on many j-chunks, which take the form of small calls for the lanes that a
256-wide block would leave empty: the bits of 128-wide work-groups on the same chunks."""
import numpy as np
import pytest

from nb6 import ics, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m_flag", [0, 1])
@pytest.mark.parametrize("n, ni", [(100003, 270), (100003, 320), (100003, 321), (300000, 65)])
def test_ragged_sets_give_the_bits_of_128_wide_groups(n, ni, m_flag):
    m, x, v = ics.plummer(n, seed=n, masses=ics.kroupa_masses(n, 2))
    rng = np.random.default_rng(ni)
    idx = np.sort(rng.choice(n, ni, replace=False))
    rs = np.minimum(0.5 * (40.0 / n) ** (1.0 / 3.0) * (1 + (x[idx] ** 2).sum(1)), 0.4)
    h2 = rs * rs / (m.mean() if m_flag else 1.0)
    dtr = np.exp(rng.uniform(np.log(2.0 ** -9), np.log(2.0 ** -4), ni))
    L = lib.load()
    g = lib.Gpunb(n)
    got = []
    try:
        g.send(m, x, v)
        for threads in (0, 128):
            assert L.nb6_set_regf_config(threads, 1, 4096) == 0
            got.append(g.regf(h2, dtr, x[idx].copy(), v[idx].copy(), 400, 350, m_flag))
    finally:
        L.nb6_set_regf_config(0, 1, 4096)
        g.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)

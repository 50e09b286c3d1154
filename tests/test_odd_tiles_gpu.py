"""A j-set of an odd number of 256-j tiles in 512-wide work-groups: the second half of the last
work-group tile holds only dummy records, and its tile origin and box do not exist.  The memory
there is filled with NaN by an earlier, larger j-set in the same buffers."""
import numpy as np
import pytest

import oracle as O
from helpers import vec_rel_err
from nb6 import ics, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [200, 5333])
def test_512_wide_groups_on_an_odd_number_of_tiles(n):
    ni = 65536                            # 512-wide work-groups
    m, x, v = ics.plummer(n, seed=n)
    rng = np.random.default_rng(n)
    idx = rng.integers(0, n, ni)
    h2 = np.full(ni, 0.01)
    dtr = np.full(ni, 2.0 ** -6)
    L = lib.load()
    big = 4 * n + 1024
    g = lib.Gpunb(big)
    try:
        # positions near the largest FP64 values: their tiles' origins and boxes overflow
        far = 1.7e308 * rng.uniform(-1.0, 1.0, (big, 3))
        d = lib.DeviceArray.from_host(np.ascontiguousarray(np.vstack([far.T, far.T, np.ones(big)])))
        assert L.nb6_send_device(big, big, d.ptr, None) == 0
        L.nb6_sync()
        d.free()
        g.send(m, x, v)
        acc, jrk, pot, lst = g.regf(h2, dtr, x[idx].copy(), v[idx].copy(), 200, 150)
    finally:
        g.close()
    racc, rjrk, rpot, rlst = O.regf(m, x, v, h2[:n], dtr[:n], x, v, 200, 150)
    assert np.array_equal(lst[:, 0], rlst[idx, 0])
    assert vec_rel_err(acc, racc[idx]).max() <= 1e-6
    assert (np.abs(pot - rpot[idx]) / rpot[idx]).max() <= 1e-6

"""Results of small blocks written straight into host memory: the device arrays of the same call,
rows with no neighbour, full rows and overflowing rows (only the count of those is used)."""
import numpy as np
import pytest

from nb6 import ics, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni, lmax, nnbmax", [(1, 2, 1), (3, 65, 64), (5, 66, 65), (257, 400, 350),
                                              (1023, 512, 511)])
def test_host_results_equal_the_device_arrays(ni, lmax, nnbmax):
    n = 2048
    m, x, v = ics.plummer(n, seed=ni)
    rng = np.random.default_rng(ni)
    idx = np.sort(rng.choice(n, ni, replace=False))
    h2 = rng.choice([0.0, 0.01, 0.1, 1.0], ni)
    dtr = np.full(ni, 2.0 ** -7)
    L = lib.load()
    g = lib.Gpunb(n)
    try:
        g.send(m, x, v)
        acc, jrk, pot, lst = g.regf(h2, dtr, x[idx].copy(), v[idx].copy(), lmax, nnbmax)
        di = lib.DeviceArray.from_host(np.ascontiguousarray(
            np.concatenate([x[idx].T, v[idx].T, h2[None], dtr[None]])))
        do, dl = lib.DeviceArray(7 * ni * 8), lib.DeviceArray(ni * lmax * 4)
        assert L.nb6_regf_device(ni, ni, di.ptr, lmax, nnbmax, 0, do.ptr, dl.ptr, None) == 0
        L.nb6_sync()
        out, rows = do.to_host(np.float64, (7, ni)), dl.to_host(np.int32, (ni, lmax))
        for d in (di, do, dl):
            d.free()
    finally:
        g.close()
    assert np.array_equal(acc, out[0:3].T) and np.array_equal(jrk, out[3:6].T)
    assert np.array_equal(pot, out[6])
    for a, b in zip(lst, rows):
        assert a[0] == b[0]
        if a[0] > 0:
            assert np.array_equal(a[:a[0] + 1], b[:a[0] + 1])
        assert not a[max(a[0], 0) + 1:].any()

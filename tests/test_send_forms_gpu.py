"""The j-set's build at tile edges: a send from host arrays (bounds from the host) and one from
device arrays (bounds on the device) leave the same j-set, so a regular force gives the same
bits; the device arrays may be overwritten as soon as the send returns; and an ensemble of
clusters of those sizes agrees with the FP64 oracle."""
import numpy as np
import pytest

import oracle as O
from helpers import vec_rel_err
from nb6 import ics, lib

pytestmark = pytest.mark.gpu
SIZES = [1, 2, 255, 256, 257, 513, 4097]


def system(n):
    if n < 3:
        return np.full(n, 0.5), np.arange(3.0 * n).reshape(n, 3), np.ones((n, 3))
    return ics.plummer(n, seed=n, masses=ics.kroupa_masses(n, 1))


def soa(x, v, *rest):
    return np.ascontiguousarray(np.vstack([x.T, v.T, *rest]))


@pytest.mark.parametrize("n", SIZES + [131073, 140000])
@pytest.mark.parametrize("m_flag", [0, 1])
def test_device_send_equals_host_send(n, m_flag):
    m, x, v = system(n)
    ni = min(n, 300)
    h2 = np.full(ni, 0.04) / (m.mean() if m_flag else 1.0)
    dtr = np.full(ni, 2.0 ** -7)
    xi, vi = x[:ni].copy(), v[:ni].copy()
    g = lib.Gpunb(n)
    try:
        g.send(m, x, v)
        a = g.regf(h2, dtr, xi, vi, 400, 350, m_flag)
        d = lib.DeviceArray.from_host(soa(x, v, m))
        assert g.L.nb6_send_device(n, n, d.ptr, None) == 0
        g.L.nb6_memcpy_htod(d.ptr, np.full(7 * n, 1e30).ctypes.data, 56 * n)
        b = g.regf(h2, dtr, xi, vi, 400, 350, m_flag)
        d.free()
    finally:
        g.close()
    for p, q in zip(a, b):
        assert np.array_equal(p, q)


def test_ensemble_of_clusters_at_tile_edges():
    parts = [system(n) for n in SIZES]
    off = np.concatenate([[0], np.cumsum(SIZES)]).astype(np.int32)
    m, x, v = (np.concatenate(p) for p in zip(*parts))
    n = len(m)
    h2, dtr = np.full(n, 0.04), np.full(n, 2.0 ** -7)
    L = lib.load()
    j, i = lib.DeviceArray.from_host(soa(x, v, m)), lib.DeviceArray.from_host(soa(x, v, h2, dtr))
    o, r = lib.DeviceArray(56 * n), lib.DeviceArray(4 * n * 1000)
    assert L.nb6_ens_open(len(SIZES), n) == 0
    try:
        for graph in (0, 1, 1):
            assert L.nb6_ens_send_device(len(SIZES), off.ctypes.data_as(lib._ip), j.ptr, n, None) == 0
            assert L.nb6_ens_regf_device(i.ptr, n, 1000, 950, 0, o.ptr, r.ptr, graph, None) == 0
            L.nb6_sync()
            out, rows = o.to_host(np.float64, (7, n)), r.to_host(np.int32, (n, 1000))
            for a, b in zip(off[:-1], off[1:]):
                s = slice(a, b)
                acc, _, pot, lst = O.regf(m[s], x[s], v[s], h2[s], dtr[s], x[s], v[s], 1000, 950)
                assert np.array_equal(rows[s][:, 0], lst[:, 0])
                assert vec_rel_err(out[0:3, s].T, acc).max() <= 1e-6
                assert (np.abs(out[6, s] - pot) <= 1e-6 * pot).all()
    finally:
        L.nb6_ens_close()
        for d in (j, i, o, r):
            d.free()

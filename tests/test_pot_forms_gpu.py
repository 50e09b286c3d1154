"""The all-pairs potential at tile and block edges (one or two particles per lane), on part of
the particles, and with coincident particles and values that are not finite.  All terms are
positive, so FP32 separations and reciprocal square roots, a few 2^-24 each, hold the sum
to 8 x 2^-24 relative."""
import numpy as np
import pytest

from nb6 import ics, lib

pytestmark = pytest.mark.gpu
TOL = 8 * 2.0 ** -24


def device_pot(x, m, i0, ni):
    n = len(m)
    d = lib.DeviceArray.from_host(np.ascontiguousarray(np.vstack([x.T, m])))
    o = lib.DeviceArray(8 * ni)
    assert lib.load().nb6_pot_device(n, n, d.ptr, i0, ni, o.ptr, None) == 0
    r = o.to_host(np.float64, ni)
    d.free()
    o.free()
    return r


def exact(x, m, idx):
    out = np.empty(len(idx))
    for k, i in enumerate(idx):
        r2 = ((x - x[i]) ** 2).sum(1)
        ok = r2 > 0
        out[k] = (m[ok] / np.sqrt(r2[ok])).sum()
    return out


@pytest.mark.parametrize("n,i0,ni", [
    (1, 0, 1), (2, 1, 1), (255, 0, 255), (256, 0, 256), (257, 3, 254), (1025, 0, 1025),
    (16384, 0, 16384), (16641, 1, 16640), (20480, 0, 20480), (70001, 33, 5714),
    (70001, 33, 5715),
])
def test_pot_matches_fp64(n, i0, ni):
    m = ics.kroupa_masses(n, n)
    if n < 3:
        x = np.arange(3.0 * n).reshape(n, 3) ** 2
    else:
        _, x, v = ics.plummer(n, seed=n, masses=m)
        m, x, _ = ics.add_binaries(m, x, v, 0.2, n)
    got = device_pot(x, m, i0, ni)
    k = np.unique(np.concatenate([[0, ni - 1], np.random.default_rng(n).integers(0, ni, 200)]))
    ref = exact(x, m, i0 + k)
    assert (np.abs(got[k] - ref) <= TOL * ref).all()


@pytest.mark.parametrize("n", [3000, 20001])      # one, two particles per lane
def test_pot_leaves_out_coincident_and_not_finite(n):
    m = ics.kroupa_masses(n, 5)
    _, x, _ = ics.plummer(n, seed=5, masses=m)
    x[11] = x[10]
    x[n - 1] = x[12]                     # another tile's
    x[100, 1] = np.inf
    x[200] = np.nan
    x[300] = (1.0e25, -1.0e25, 3.0)      # r2 overflows: adds nothing
    m[12] = 0.0
    got = device_pot(x, m, 0, n)
    out = np.array([100, 200, 300])
    assert (got[out] == 0.0).all()
    keep = np.setdiff1d(np.arange(n), out)
    k = np.unique(np.concatenate([[10, 11, 12, n - 1], keep[::97]]))
    ref = exact(x[keep], m[keep], np.searchsorted(keep, k))
    assert (np.abs(got[k] - ref) <= TOL * ref).all()

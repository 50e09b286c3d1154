"""A j-set that is being built on one stream and used on another: nb6_send_device and
nb6_jp_predict_send_ followed at once by the regular force, the k-th neighbour radius and
another send on a different stream give the results of one stream; a force can be captured
while the build is still queued, and replays once its caller has waited for that."""
import ctypes

import numpy as np
import pytest

from helpers import c2_inputs
from nb6 import lib
from test_zz_no_alloc import _same_rows

pytestmark = pytest.mark.gpu

N, NI, LMAX, NNBMAX = 200000, 3000, 300, 250


class Streams:
    def __init__(self):
        self.L = lib.load()
        self.s = [ctypes.c_void_p(), ctypes.c_void_p()]
        for s in self.s:
            assert self.L.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0    # hipStreamNonBlocking

    def sync(self):
        self.L.nb6_sync()
        for s in self.s:
            assert self.L.hipStreamSynchronize(s) == 0

    def close(self):
        for s in self.s:
            self.L.hipStreamDestroy(s)


@pytest.fixture(scope="module")
def case():
    m, x, v, idx, h2, dtr = c2_inputs(n=N, ni=NI, m_flag=1)
    L = lib.load()
    sets = [(x, v), (-1.5 * x, v), (x[::-1].copy(), v)]
    d = {"j": [], "i": []}
    for a, b in sets:
        d["j"].append(lib.DeviceArray.from_host(np.ascontiguousarray(np.concatenate([a.T, b.T, m[None]]))))
        d["i"].append(lib.DeviceArray.from_host(np.ascontiguousarray(
            np.concatenate([a[idx].T, b[idx].T, h2[None], dtr[None]]))))
    out = lib.DeviceArray(7 * NI * 8)
    rows = lib.DeviceArray(NI * LMAX * 4)
    rs = lib.DeviceArray(NI * 8)
    g = lib.Gpunb(N)
    st = Streams()
    yield L, g, d, out, rows, rs, st, (m, x, v)
    st.close()
    g.close()
    for q in d["j"] + d["i"] + [out, rows, rs]:
        q.free()


def _force(c, k, s):
    L, g, d, out, rows, rs, st, _ = c
    assert L.nb6_regf_device(NI, NI, d["i"][k].ptr, LMAX, NNBMAX, 1, out.ptr, rows.ptr, s) == 0
    assert L.nb6_rs_kth_device(NI, NI, d["i"][k].ptr, rows.ptr, LMAX, 2, rs.ptr, s) == 0


def _results(c):
    L, g, d, out, rows, rs, st, _ = c
    st.sync()
    return (out.to_host(np.float64, (7, NI)), rows.to_host(np.int32, (NI, LMAX)),
            rs.to_host(np.float64, (NI,)))


def _same(a, b):
    return np.array_equal(a[0], b[0]) and _same_rows(a[1], b[1]) and np.array_equal(a[2], b[2])


@pytest.mark.parametrize("send, use", [(0, 1), (0, None), (None, 0)])
def test_send_on_one_stream_force_on_another(case, send, use):
    L, g, d, out, rows, rs, st, _ = case
    sa = None if send is None else st.s[send]
    sb = None if use is None else st.s[use]
    want = []
    for k in range(3):
        assert L.nb6_send_device(N, N, d["j"][k].ptr, None) == 0
        _force(case, k, None)
        want.append(_results(case))
    for rep in range(6):
        k = rep % 3
        assert L.nb6_send_device(N, N, d["j"][k].ptr, sa) == 0
        _force(case, k, sb)
        assert _same(_results(case), want[k]), rep
    # two sends in a row on different streams: the second one counts
    for rep in range(4):
        k = rep % 3
        assert L.nb6_send_device(N, N, d["j"][(k + 1) % 3].ptr, sa) == 0
        assert L.nb6_send_device(N, N, d["j"][k].ptr, sb) == 0
        _force(case, k, sa)
        assert _same(_results(case), want[k]), rep


def test_predicted_j_set_on_another_stream(case):
    L, g, d, out, rows, rs, st, (m, x, v) = case
    jp = lib.JPred(N)
    z = np.zeros((N, 3))
    try:
        want = []
        for sign in (1.0, -1.0):
            jp.set(np.arange(1, N + 1), sign * x, v, z, z, m, np.zeros(N))
            jp.predict_send(0.0, N)
            _force(case, 0, None)
            want.append(_results(case))
        for rep in range(4):
            jp.set(np.arange(1, N + 1), (1.0 if rep % 2 == 0 else -1.0) * x, v, z, z, m, np.zeros(N))
            jp.predict_send(0.0, N)
            _force(case, 0, st.s[0])
            assert _same(_results(case), want[rep % 2]), rep
    finally:
        jp.close()


def test_captured_force_after_a_send_on_another_stream(case):
    L, g, d, out, rows, rs, st, _ = case
    ib, s = d["i"][1], st.s[1]

    def step(stream):
        assert L.nb6_regf_device_noalloc(NI, NI, ib.ptr, LMAX, NNBMAX, 1, out.ptr, rows.ptr, stream) == 0

    assert L.nb6_send_device(N, N, d["j"][1].ptr, None) == 0
    step(None)
    want = _results(case)
    assert L.nb6_send_device(N, N, d["j"][0].ptr, None) == 0
    graph, ex = ctypes.c_void_p(), ctypes.c_void_p()
    assert L.nb6_send_device(N, N, d["j"][1].ptr, st.s[0]) == 0
    assert L.hipStreamBeginCapture(s, 1) == 0                  # hipStreamCaptureModeThreadLocal
    step(s)
    assert L.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    assert L.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    try:
        assert L.hipStreamSynchronize(st.s[0]) == 0            # (a replay is the caller's to order)
        zero = np.zeros((7, NI))
        for rep in range(3):
            L.nb6_memcpy_htod(out.ptr, zero.ctypes.data, zero.nbytes)
            assert L.hipGraphLaunch(ex, s) == 0
            got = _results(case)
            assert np.array_equal(got[0], want[0]) and _same_rows(got[1], want[1]), rep
    finally:
        L.hipGraphExecDestroy(ex)
        L.hipGraphDestroy(graph)

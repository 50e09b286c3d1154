"""nb6_ens_send_device returns with the j-set complete: a step on another stream than the
send's takes the particles just sent, at every one of repeated sends of one layout (which
keep the cluster layout and the work items, as an integration's sends do)."""
import ctypes

import numpy as np
import pytest

from nb6 import lib
from test_ensemble_gpu import _same_rows, make_ensemble

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("send_on_library_stream", [False, True])
def test_step_on_another_stream_takes_the_sent_particles(send_on_library_stream):
    sizes = [16384, 8000, 300, 12000, 64, 9000]
    ms, xs, vs, h2s, dts, off = make_ensemble(sizes, seed=31)
    lmax, nnbmax = 120, 100
    ntot = int(off[-1])
    L = lib.load()
    offp = off.ctypes.data_as(lib._ip)
    m, v = np.concatenate(ms), np.concatenate(vs)
    h2, dtr = np.concatenate(h2s), np.concatenate(dts)
    x = np.concatenate(xs)
    dev = []
    for k in range(2):      # the particles and, mirrored and drifted, the same clusters again
        xk = x if k == 0 else -(x + 0.02 * v)
        vk = v if k == 0 else -v
        dev.append((lib.DeviceArray.from_host(np.ascontiguousarray(np.concatenate([xk.T, vk.T, m[None]]))),
                    lib.DeviceArray.from_host(np.ascontiguousarray(
                        np.concatenate([xk.T, vk.T, h2[None], dtr[None]])))))
    do = lib.DeviceArray(7 * ntot * 8)
    dl = lib.DeviceArray(ntot * lmax * 4)
    other = ctypes.c_void_p()
    assert L.hipStreamCreateWithFlags(ctypes.byref(other), 1) == 0       # hipStreamNonBlocking
    sa, sb = (None, other) if send_on_library_stream else (other, None)

    def step(k, s_send, s_step):
        assert L.nb6_ens_send_device(len(sizes), offp, dev[k][0].ptr, ntot, s_send) == 0
        assert L.nb6_ens_regf_device(dev[k][1].ptr, ntot, lmax, nnbmax, 0, do.ptr, dl.ptr, 0, s_step) == 0
        L.nb6_sync()
        assert L.hipStreamSynchronize(other) == 0
        return do.to_host(np.float64, (7, ntot)), dl.to_host(np.int32, (ntot, lmax))

    try:
        assert L.nb6_ens_open(len(sizes), ntot) == 0
        want = [step(k, sb, sb) for k in range(2)]
        for rep in range(6):
            out, lst = step(rep % 2, sa, sb)
            assert np.array_equal(out, want[rep % 2][0]), f"send {rep}"
            assert _same_rows(lst, want[rep % 2][1]), f"send {rep}"
    finally:
        L.nb6_ens_close()
        L.hipStreamDestroy(other)
        for a, b in dev:
            a.free()
            b.free()
        do.free()
        dl.free()

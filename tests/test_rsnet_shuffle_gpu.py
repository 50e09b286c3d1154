"""An epoch's minibatches: the order of the seeded keys (SplitMix64), sorted stably, at sample
counts for one, two and three launches of the order and for the library's sort; weights equal
those of single steps on the same batches, bit for bit."""
import ctypes

import numpy as np
import pytest

import rsnet as R
from nb6 import lib
from nb6.rsdrive import RSNet

pytestmark = pytest.mark.gpu


def shuffled(n, seed):
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + np.uint64(0x9E3779B97F4A7C15) * np.arange(1, n + 1, dtype=np.uint64)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z ^= z >> np.uint64(31)
    return np.argsort(z >> np.uint64(32), kind="stable")


@pytest.mark.parametrize("n, batch", [(1, 1), (500, 200), (8192, 1000), (20011, 4096),
                                      (131072, 32768), (131073, 65536)])
def test_epoch_equals_steps_on_the_shuffled_batches(n, batch):
    rng = np.random.default_rng(n)
    feat = rng.normal(size=(8, n)).astype(np.float32)
    t = rng.normal(size=n).astype(np.float32)
    p = R.init_params(5).astype(np.float32)
    h = ctypes.c_float()
    got = []
    for epoch in (True, False):
        net = RSNet(seed=7)
        net.set_params(p)
        net.set_norm(np.zeros(8, np.float32), np.ones(8, np.float32))
        if epoch:
            fd, td = (lib.DeviceArray.from_host(a) for a in (feat, t))
            assert net.L.nb6_rsnet_train_epoch_device(n, fd.ptr, td.ptr, batch, ctypes.c_float(1e-3),
                                                      99, ctypes.addressof(h), None) == 0
            fd.free()
            td.free()
        else:
            o = shuffled(n, 99)
            for b in range(n // batch):
                k = o[b * batch:(b + 1) * batch]
                fd, td = (lib.DeviceArray.from_host(np.ascontiguousarray(a))
                          for a in (feat[:, k], t[k]))
                assert net.L.nb6_rsnet_train_step_device(batch, fd.ptr, td.ptr, ctypes.c_float(1e-3),
                                                         ctypes.addressof(h), None) == 0
                fd.free()
                td.free()
        got.append(net.params())
        net.close()
    assert np.array_equal(got[0], got[1])
    assert not np.array_equal(got[0], p)

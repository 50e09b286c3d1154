"""The network's gradient over batch sizes at the edges of its work-groups (64 samples) and
of the partial sums read at once (128 blocks; 8192 loss partials), and the Adam step that
follows it, against the FP64 oracle."""
import ctypes

import numpy as np
import pytest

import rsnet as R
from nb6 import lib
from nb6.rsdrive import RSNet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [63, 64, 65, 8192, 8193, 8192 * 64 + 65])
def test_gradient_and_adam_step_by_batch_size(n):
    net = RSNet(seed=7)
    rng = np.random.default_rng(n)
    p = R.init_params(3).astype(np.float32)
    net.set_params(p)
    net.set_norm(np.zeros(8, np.float32), np.ones(8, np.float32))
    feat = rng.normal(size=(n, 8)).astype(np.float32)
    t = np.full(n, -3.0, np.float32)          # residuals of one sign: no cancellation
    dev = [lib.DeviceArray.from_host(np.ascontiguousarray(a)) for a in (feat.T, t)]
    dev += [lib.DeviceArray(R.NPARAM * 4), lib.DeviceArray(4)]
    fd, td, gd, ld = (d.ptr for d in dev)
    assert net.L.nb6_rsnet_grad_device(n, fd, td, gd, ld, None) == 0
    g = dev[2].to_host(np.float32, R.NPARAM).astype(np.float64)
    loss = float(dev[3].to_host(np.float32, 1)[0])
    lr, h = 1e-3, ctypes.c_float()
    assert net.L.nb6_rsnet_train_step_device(n, fd, td, ctypes.c_float(lr), ctypes.addressof(h),
                                             None) == 0
    w = net.params().astype(np.float64)
    for d in dev:
        d.free()
    net.close()
    rl, rg = R.loss_and_grad(p, feat, t)
    # FP32 sums: 1e-5 inside a block, and one rounding (2^-24) per block partial added
    tol = 1e-5 + ((n + 63) // 64) * 2.0 ** -24
    assert abs(loss - rl) <= 1e-5 * rl and abs(h.value - rl) <= 1e-5 * rl
    assert np.linalg.norm(g - rg) <= tol * np.linalg.norm(rg)
    # first step: lr g / (|g| + 1e-8); weights below 2 hold it to 2^-23 of their size
    big = np.abs(g) > 1e-3
    step = (p - w)[big]
    assert np.abs(step - lr * np.sign(g[big])).max() <= 1e-3 * lr + 2.0 ** -22
    assert np.array_equal(w[g == 0.0], p[g == 0.0])

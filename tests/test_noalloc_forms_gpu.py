"""nb6_regf_device_noalloc with i-sets on both sides of where the whole call, were it one batch,
would take one wavefront per i in the finalize: small batches of many chunks either way.
Lists and forces against the FP64 kernel's."""
import numpy as np
import pytest

from helpers import c2_inputs
from nb6 import lib
from test_zz_no_alloc import _call, _rel, _same_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni", [16384, 16385, 30001])
def test_small_batches_of_large_calls(ni):
    L = lib.load()
    m, x, v, idx, h2, dtr = c2_inputs(n=32768, ni=ni)
    lmax, nnbmax = 500, 450
    ib = np.ascontiguousarray(np.concatenate([x[idx].T, v[idx].T, h2[None], dtr[None]]))
    g = lib.Gpunb(m.size)
    try:
        g.send(m, x, v)
        out, lst = _call(L, L.nb6_regf_device_noalloc, ib, ni, lmax, nnbmax)
        assert L.nb6_last_regf_batches() > 4 and L.nb6_last_regf_chunks() >= 16
        ref, rlst = _call(L, L.nb6_regf_device, ib, ni, lmax, nnbmax, prec=2)
    finally:
        g.close()
    assert _same_rows(lst, rlst)
    # the bar of the FP32 kernel against FP64
    for q in (slice(0, 3), slice(3, 6), slice(6, 7)):
        assert _rel(out[q], ref[q]).max() <= 1e-6

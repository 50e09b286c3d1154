"""Replays of the ensemble's graph (nb6_ens_regf_device, use_graph = 1) after a change that the
captured kernel arguments depend on: every such call gives the eager step's results."""
import numpy as np
import pytest

import oracle as O
from helpers import vec_rel_err
from nb6 import lib
from test_ensemble_gpu import _same_rows, make_ensemble

pytestmark = pytest.mark.gpu


class Ens:
    """An open ensemble with device copies of several layouts of ntot particles."""

    def __init__(self, layouts, lmax):
        self.L, self.lmax = lib.load(), lmax
        self.ntot = sum(layouts[0])
        self.parts = [make_ensemble(s, seed=17 + k) for k, s in enumerate(layouts)]
        self.dev = []
        for ms, xs, vs, h2s, dts, off in self.parts:
            m, x, v = np.concatenate(ms), np.concatenate(xs), np.concatenate(vs)
            h2, dtr = np.concatenate(h2s), np.concatenate(dts)
            self.dev.append(lib.DeviceArray.from_host(np.ascontiguousarray(
                np.concatenate([x.T, v.T, m[None]]))))
            self.dev.append(lib.DeviceArray.from_host(np.ascontiguousarray(
                np.concatenate([x.T, v.T, h2[None], dtr[None]]))))
        # one i-block array: the graph's key holds its address
        self.di = lib.DeviceArray(8 * self.ntot * 8)
        self.do = lib.DeviceArray(7 * self.ntot * 8)
        self.dl = lib.DeviceArray(self.ntot * lmax * 4)
        assert self.L.nb6_ens_open(max(len(s) for s in layouts), self.ntot) == 0

    def send(self, k):
        off = self.parts[k][5]
        assert self.L.nb6_ens_send_device(len(off) - 1, off.ctypes.data_as(lib._ip), self.dev[2 * k].ptr,
                                          self.ntot, None) == 0
        self.L.nb6_device_copy(self.di.ptr, self.dev[2 * k + 1].ptr, 8 * self.ntot * 8, None)

    def step(self, graph, lmax, nnbmax):
        assert self.L.nb6_ens_regf_device(self.di.ptr, self.ntot, lmax, nnbmax, 0, self.do.ptr,
                                          self.dl.ptr, graph, None) == 0
        self.L.nb6_sync()
        lst = self.dl.to_host(np.int32, (self.ntot * self.lmax,))[:self.ntot * lmax]
        return self.do.to_host(np.float64, (7, self.ntot)), lst.reshape(self.ntot, lmax)

    def close(self):
        self.L.nb6_ens_close()
        for d in self.dev + [self.di, self.do, self.dl]:
            d.free()


def test_layout_of_equal_totals_and_another_longest_cluster():
    """Two layouts with the same particles, slots and work items: the longest cluster of the
    second has two partial-sum segments, that of the first one.  Nearly every row takes
    the FP64 pass, which works by segments."""
    lmax, nnbmax = 120, 100
    e = Ens([[4096, 4096], [256, 7936]], lmax)
    try:
        e.L.nb6_set_ens_refine_weights(1e6, 1e6, 1e6, 0.0)
        for k in (0, 1, 0):
            e.send(k)
            got = [e.step(1, lmax, nnbmax) for _ in range(3)]
            want = e.step(0, lmax, nnbmax)
            # (an outlier of 256 particles can have all of them in its near field: no FP32 sums)
            assert e.L.nb6_ens_last_refined() > e.ntot - 256
            ms, xs, vs, h2s, dts, off = e.parts[k]
            for c in range(2):
                a, b = off[c], off[c + 1]
                racc = O.regf(ms[c], xs[c], vs[c], h2s[c], dts[c], xs[c], vs[c], lmax, nnbmax)[0]
                for q, (out, _) in enumerate(got):
                    assert vec_rel_err(out[0:3, a:b].T, racc).max() <= 1e-6, (k, c, q)
            # (which rows' items found room, and so the order of their FP64 sums, differs
            # from call to call: 8,192 terms that cancel to a thousandth leave 1e-9)
            for out, lst in got:
                assert vec_rel_err(out[0:3].T, want[0][0:3].T).max() <= 1e-9
                assert _same_rows(lst, want[1])
    finally:
        e.L.nb6_set_ens_refine_weights(0.5, 0.5, 0.5, 0.0)
        e.close()


def test_work_buffers_that_a_larger_step_outgrew():
    """A step with longer rows between two graph steps takes larger work buffers, so the graph's
    are gone; the same for the switched diagnostic output."""
    e = Ens([[3000, 900, 1500]], 600)
    dbg = lib.DeviceArray(4 * e.ntot * 8)
    try:
        e.send(0)
        first = [e.step(1, 80, 60) for _ in range(2)]
        e.step(0, 600, 560)
        after = [e.step(1, 80, 60) for _ in range(3)]
        want = e.step(0, 80, 60)
        for out, lst in first + after:
            assert np.array_equal(out, want[0])
            assert _same_rows(lst, want[1])
        # the error scales follow the switch, from eager and from replayed steps
        ref = np.full((4, e.ntot), -1.0)
        scales = []
        for ptr in (dbg.ptr, None, dbg.ptr):
            e.L.nb6_set_regf_debug_bounds(ptr)
            e.L.nb6_memcpy_htod(dbg.ptr, ref.ctypes.data, ref.nbytes)
            out, _ = e.step(1, 80, 60)
            assert np.array_equal(out, want[0])
            scales.append(dbg.to_host(np.float64, (4, e.ntot)))
        assert (scales[0] >= 0).all() and np.array_equal(scales[0], scales[2])
        assert (scales[1] == -1.0).all()
    finally:
        e.L.nb6_set_regf_debug_bounds(None)
        dbg.free()
        e.close()

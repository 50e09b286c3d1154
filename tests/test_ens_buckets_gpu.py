"""The FP64 pass of an ensemble with more (cluster, segment) buckets than its lists hold in LDS
(4096): every flagged row is recomputed from its own cluster's particles, as the FP64 oracle
has them."""
import numpy as np
import pytest

import oracle as O
from helpers import rows_as_sets, vec_rel_err
from nb6 import lib
from test_ensemble_gpu import make_ensemble, run_ensemble

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    [64] * 4096,                              # the most that have a bucket per entry
    [64] * 4097,                              # one more: runs of two buckets
    [40 + c % 50 for c in range(9000)],       # runs of three, the last one short
    [64] * 2500 + [9000] + [64] * 2500,       # three segments per cluster, most of them empty
], ids=["4096", "4097", "9000", "15003"])
def test_every_row_in_the_fp64_pass(sizes):
    base = make_ensemble(sorted(set(sizes)), seed=3, counts=20)
    of = {n: k for k, n in enumerate(sorted(set(sizes)))}
    ms, xs, vs, h2s, dts = [[q[of[n]] for n in sizes] for q in base[:5]]
    off = np.r_[0, np.cumsum(sizes)].astype(np.int32)
    L = lib.load()
    lmax, nnbmax = 64, 50
    L.nb6_set_ens_refine_weights(1e6, 1e6, 1e6, 0.0)
    try:
        (out, lst), = run_ensemble(ms, xs, vs, h2s, dts, off, lmax, nnbmax, use_graph=0)
    finally:
        L.nb6_set_ens_refine_weights(0.5, 0.5, 0.5, 0.0)
    ref = {n: O.regf(*[q[of[n]] for q in base[:5]], base[1][of[n]], base[2][of[n]], lmax, nnbmax)
           for n in of}
    for c, n in enumerate(sizes):
        a, b = off[c], off[c + 1]
        racc, rjrk, rpot, rlst = ref[n]
        assert rows_as_sets(lst[a:b]) == rows_as_sets(rlst), c
        # FP64 sums: 1e-16 times up to 9,000 terms that cancel to a thousandth
        assert vec_rel_err(out[0:3, a:b].T, racc).max() <= 1e-9, c
        assert (np.abs(out[6, a:b] - rpot) <= 1e-9 * np.abs(rpot)).all(), c

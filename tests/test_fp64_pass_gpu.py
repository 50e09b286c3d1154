"""The regular force's FP64 pass in its forms (units of four items up to 16,384 i, of 64 above,
few and many segments, short last segments): with error weights that send every row through
it, acc, jerk and pot agree with the FP64 oracle as FP64 sums do (1e-9: 40,000 terms of 2^-53
with 200-fold cancellation), lists equal it.  The calls run in one child process: the
weights are a library setting that other tests use at its defaults."""
import json
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROOT = Path(__file__).resolve().parent.parent
CASES = [(300, 1, 0), (300, 63, 0), (1000, 65, 1), (1024, 40, 0), (5000, 257, 0),
         (20011, 700, 1), (40000, 3, 0), (2000, 16384, 0), (2000, 16385, 0), (3001, 17000, 1)]


def run_case(n, ni, m_flag):
    import oracle as O
    from helpers import vec_rel_err
    from nb6 import ics, lib
    rng = np.random.default_rng(n * 7 + ni)
    m, x, v = ics.plummer(n, seed=n, masses=ics.kroupa_masses(n, 1))
    idx = rng.choice(n, size=ni, replace=ni > n)
    h2 = (0.1 + 0.3 * rng.uniform(size=ni)) ** 2 * (300.0 / n) ** (2.0 / 3.0)
    if m_flag:
        h2 = h2 / m.mean()
    dtr = np.full(ni, 2.0 ** -6)
    xi, vi = x[idx].copy(), v[idx].copy()
    g = lib.Gpunb(n)
    # every segment's share is above any allowance
    g.L.nb6_set_regf_refine_weights(1e6, 1e6, 1e6, 1e6)
    g.send(m, x, v)
    acc, jrk, pot, lst = g.regf(h2, dtr, xi, vi, 400, 350, m_flag)
    rows = g.L.nb6_last_regf_refined()
    g.close()
    racc, rjrk, rpot, rlst = O.regf(m, x, v, h2, dtr, xi, vi, 400, 350, m_flag)
    same = all(a[0] == b[0] and np.array_equal(a[1:max(b[0], 0) + 1], b[1:max(b[0], 0) + 1])
               for a, b in zip(lst, rlst))
    return {"rows": rows, "lists": same, "acc": vec_rel_err(acc, racc).max(),
            "jrk": vec_rel_err(jrk, rjrk).max(), "pot": (np.abs(pot - rpot) / rpot).max()}


def main():
    for c in CASES:
        print("CASE " + json.dumps([c, run_case(*c)]), flush=True)


@pytest.fixture(scope="module")
def results():
    path = os.pathsep.join(str(p) for p in (ROOT / "tests", ROOT / "oracle",
                                            ROOT / "nbody6ppgpu-beijing_amd"))
    p = subprocess.run([sys.executable, "-c", "import test_fp64_pass_gpu as t; t.main()"],
                       env={**os.environ, "PYTHONPATH": path}, capture_output=True, text=True,
                       timeout=100)
    assert p.returncode == 0, p.stderr[-2000:]
    got = [json.loads(s[5:]) for s in p.stdout.splitlines() if s.startswith("CASE ")]
    return {tuple(c): r for c, r in got}


@pytest.mark.parametrize("case", CASES)
def test_every_row_through_the_fp64_pass(results, case):
    r = results[case]
    assert r["rows"] == case[1] and r["lists"]
    assert r["acc"] <= 1e-9 and r["jrk"] <= 1e-9 and r["pot"] <= 1e-9

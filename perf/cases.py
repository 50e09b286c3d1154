"""The calls of libnb6gpu.so whose time matters to a program that uses it, with the sizes
they meet: regular blocks (the j-set sent, then the regular force of the block's particles,
from host arrays as the Fortran integrator calls them and on device arrays), one step of an
ensemble of small clusters, the all-pairs potential, the irregular force of a block, and one
training epoch of the neighbour-radius network.

A case is a dict of plain values; ``kind`` names the call sequence:
  host      gpunb_send_ + gpunb_regf_ on host arrays
  device    nb6_send_device + nb6_regf_device
  ensemble  nb6_ens_send_device + nb6_ens_regf_device
  pot_host  gpupot_              pot     nb6_pot_device
  irr_host  irr_simd_firr_vec_   irr     nb6_irr_firr_device
  train     nb6_rsnet_open, _set_norm, _train_epoch_device, _get_params
"""
from __future__ import annotations

import ctypes
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parent.parent / "nbody6ppgpu-beijing_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from nb6 import lib  # noqa: E402

N_MAX = 1 << 20                  # particles the library is opened for
ENS_CLUSTERS, ENS_PARTICLES = 256, 1 << 20
PAIR_FLOPS, POT_FLOPS = 60, 20   # per pair, the reference's convention and the potential's


def listed():
    return [
        # N = 1024 Plummer sphere (examples/example_1k): an ordinary small block, all launch
        # and transfer latency
        {"name": "block_1k_host", "kind": "host", "n": 1024, "ni": 40, "lmax": 400,
         "nnb": 50, "binaries": 0.0, "m_flag": 0},
        # N = 65,536: the integrator hands over blocks in pieces of up to 1024
        {"name": "block_64k_host", "kind": "host", "n": 65536, "ni": 1024, "lmax": 500,
         "nnb": 80, "binaries": 0.0, "m_flag": 0},
        # a small block of an odd-sized cluster, on device arrays
        {"name": "block_50k", "kind": "device", "n": 50021, "ni": 257, "lmax": 500,
         "nnb": 80, "binaries": 0.1, "m_flag": 0},
        # N = 100k (the N100k input), mass-weighted neighbour criterion, half in binaries
        {"name": "block_100k_mass", "kind": "device", "n": 100003, "ni": 6007, "lmax": 500,
         "nnb": 80, "binaries": 0.5, "m_flag": 1},
        # every particle of N = 65,536 at once (start-up, synchronised steps)
        {"name": "full_64k", "kind": "device", "n": 65536, "ni": 65536, "lmax": 500,
         "nnb": 80, "binaries": 0.0, "m_flag": 0},
        # the largest block of the N = 1,048,576 system with 50 % binaries
        {"name": "block_1m", "kind": "device", "n": 1048576, "ni": 131072, "lmax": 600,
         "nnb": 80, "binaries": 0.5, "m_flag": 0},
        # independent clusters of uneven N, one regular step of all particles
        {"name": "ensemble_64", "kind": "ensemble", "clusters": 64, "n_lo": 1024,
         "n_hi": 16384, "lmax": 400, "nnb": 50},
        # energy check of an N = 10k run from host arrays
        {"name": "pot_10k_host", "kind": "pot_host", "n": 10007, "binaries": 0.1},
        # and of a large one, device arrays
        {"name": "pot_256k", "kind": "pot", "n": 262144, "binaries": 0.5},
        # irregular blocks: a small one through the Fortran interface, a large one on the
        # device
        {"name": "irr_64k_host", "kind": "irr_host", "n": 65536, "ni": 100, "lmax": 256,
         "nnb": 80},
        {"name": "irr_256k", "kind": "irr", "n": 262144, "ni": 32768, "lmax": 256, "nnb": 80},
        # neighbour-radius network: one epoch of minibatch Adam
        {"name": "train_131k", "kind": "train", "samples": 131072, "batch": 8192},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("host", "device", "device", "device", "ensemble", "pot_host", "pot",
                       "irr_host", "irr", "train"))
    if kind in ("host", "device"):
        n = _log_int(rng, 1000, 200000 if kind == "host" else 400000)
        ni = _log_int(rng, 1, min(n, 1024 if kind == "host" else 65536))
        big = n >= 4096
        return {"kind": kind, "n": n, "ni": ni, "lmax": rng.choice((500, 600)) if big else 400,
                "nnb": 80 if big else 50, "binaries": rng.choice((0.0, 0.1, 0.5)),
                "m_flag": rng.choice((0, 0, 1))}
    if kind == "ensemble":
        lo = _log_int(rng, 500, 3000)
        return {"kind": kind, "clusters": _log_int(rng, 4, 128), "n_lo": lo,
                "n_hi": _log_int(rng, lo + 1, 16384), "lmax": 400, "nnb": 50}
    if kind in ("pot", "pot_host"):
        return {"kind": kind, "n": _log_int(rng, 1000, 40000 if kind == "pot_host" else 300000),
                "binaries": rng.choice((0.0, 0.1, 0.5))}
    if kind in ("irr", "irr_host"):
        n = _log_int(rng, 4000, 300000)
        ni = _log_int(rng, 1, min(n, 1024) if kind == "irr_host" else max(2, n // 4))
        return {"kind": kind, "n": n, "ni": ni, "lmax": 256, "nnb": 80}
    n = _log_int(rng, 20000, 400000)
    return {"kind": kind, "samples": n, "batch": rng.choice((2048, 4096, 8192))}


# ---------------------------------------------------------------------- inputs
def _unit(rng, n):
    z = rng.uniform(-1.0, 1.0, n)
    phi = rng.uniform(0.0, 2.0 * math.pi, n)
    s = np.sqrt(1.0 - z * z)
    return np.stack([s * np.cos(phi), s * np.sin(phi), z], axis=1)


def _masses(rng, n):
    """Kroupa-like two-segment power law, 0.08-100, total mass 1."""
    def seg(a, u, lo, hi):
        return (lo ** (1 - a) + u * (hi ** (1 - a) - lo ** (1 - a))) ** (1.0 / (1 - a))
    low = rng.uniform(0.0, 1.0, n) < 0.76
    u = rng.uniform(0.0, 1.0, n)
    m = np.where(low, seg(1.3, u, 0.08, 0.5), seg(2.3, u, 0.5, 100.0))
    return m / m.sum()


_Q = np.linspace(0.0, 1.0, 4097)
_QCDF = np.concatenate([[0.0], np.cumsum(0.5 * np.diff(_Q) * (
    (_Q ** 2 * (1 - _Q ** 2) ** 3.5)[1:] + (_Q ** 2 * (1 - _Q ** 2) ** 3.5)[:-1]))])
_QCDF /= _QCDF[-1]


def _cluster(rng, n, binaries=0.0, equal=False):
    """A Plummer sphere in N-body units (cut at ten scale radii), a share of its particles
    paired into binaries of 0.005-50 AU: m [n], x [n][3], v [n][3]."""
    m = np.full(n, 1.0 / n) if equal else _masses(rng, n)
    top = (1.0 + 1.0 / 100.0) ** -1.5                 # mass inside ten scale radii
    r = 1.0 / np.sqrt(rng.uniform(1e-9, top, n) ** (-2.0 / 3.0) - 1.0)
    x = _unit(rng, n) * r[:, None]
    q = np.interp(rng.uniform(0.0, 1.0, n), _QCDF, _Q)
    v = _unit(rng, n) * (q * math.sqrt(2.0) * (1.0 + r * r) ** -0.25)[:, None]
    a = 3.0 * math.pi / 16.0
    x *= a
    v /= math.sqrt(a)
    nb = int(0.5 * binaries * n)
    if nb:
        sep = np.exp(rng.uniform(math.log(0.005), math.log(50.0), nb)) / 206264.806
        i, j = np.arange(nb) * 2, np.arange(nb) * 2 + 1
        mt = m[i] + m[j]
        e = _unit(rng, nb)
        w = np.cross(e, _unit(rng, nb))
        w *= (np.sqrt(mt / sep) / np.linalg.norm(w, axis=1))[:, None]
        d = e * sep[:, None]
        fi, fj = (m[j] / mt)[:, None], (m[i] / mt)[:, None]
        x[j], v[j] = x[i] - fj * d, v[i] - fj * w
        x[i], v[i] = x[i] + fi * d, v[i] + fi * w
    return m, x, v


def _radii(rng, x, idx, nnb, cap):
    """Neighbour radii that give about log-normal counts of median nnb, from the mean
    density of the shell around each particle."""
    n = len(x)
    r = np.sqrt((x * x).sum(1))
    order = np.argsort(r)
    rs = r[order]
    rank = np.empty(n, np.int64)
    rank[order] = np.arange(n)
    w = max(16, n // 512)
    k = rank[idx]
    lo, hi = np.maximum(k - w, 0), np.minimum(k + w, n - 1)
    inner = np.where(k - w < 0, 0.0, rs[lo])
    dens = (hi - lo + 1) / (4.0 / 3.0 * math.pi * (rs[hi] ** 3 - inner ** 3))
    counts = np.clip(np.exp(rng.normal(math.log(nnb), 0.4, len(idx))), 2.0, cap)
    rad = (3.0 * counts / (4.0 * math.pi * dens)) ** (1.0 / 3.0)
    return np.minimum(rad, 0.3 * (r[idx] + rs[n // 2]))


def _block(case, seed):
    """One regular block: m, x, v of all particles; h2, dtr, x, v of the active ones."""
    n, ni = case["n"], case["ni"]
    rng = np.random.default_rng([seed, n, ni])
    m, x, v = _cluster(rng, n, case["binaries"], equal=n <= 2048)
    idx = np.sort(rng.choice(n, size=ni, replace=False)) if ni < n else np.arange(n)
    rs = _radii(rng, x, idx, case["nnb"], 0.6 * case["lmax"])
    h2 = rs * rs
    if case["m_flag"]:
        h2 = h2 / m.mean()
    dtr = np.exp(rng.uniform(math.log(2.0 ** -10), math.log(2.0 ** -4), ni))
    return m, x, v, idx, h2, dtr


def _soa(x, v, *rest):
    return np.concatenate([x.T, v.T, np.stack(rest)])


def _gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _ensemble(case, seed):
    """Cluster sizes (the case's own) and the particles of all clusters (the seed's)."""
    srng = np.random.default_rng([case["clusters"], case["n_lo"], case["n_hi"]])
    sizes = np.exp(srng.uniform(math.log(case["n_lo"]), math.log(case["n_hi"]),
                                case["clusters"])).astype(np.int64)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    rng = np.random.default_rng([seed, int(off[-1])])
    _, x, v = _cluster(rng, int(off[-1]), equal=True)
    m = np.repeat(1.0 / sizes, sizes)
    rs = np.concatenate([_radii(rng, x[a:b], np.arange(b - a), case["nnb"], 0.6 * case["lmax"])
                         for a, b in zip(off[:-1], off[1:])])
    dtr = np.exp(rng.uniform(math.log(2.0 ** -8), math.log(2.0 ** -4), len(m)))
    return off, m, x, v, rs * rs, dtr


def _irr_cluster(case):
    """The cluster whose irregular blocks are asked for: it belongs to the case, the seeds
    choose the blocks."""
    n = case["n"]
    rng = np.random.default_rng([n, case["lmax"]])
    m, x, v = _cluster(rng, n)
    rs = _radii(rng, x, np.arange(n), case["nnb"], 0.6 * case["lmax"])
    a = 3.0 * math.pi / 16.0
    d2 = (x * x).sum(1) + a * a
    acc = -x / d2[:, None] ** 1.5
    jrk = -v / d2[:, None] ** 1.5 + 3.0 * x * ((x * v).sum(1) / d2 ** 2.5)[:, None]
    t0 = np.floor(rng.uniform(0.0, 8.0, n)) / 256.0
    return m, x, v, rs * rs, acc / 2.0, jrk / 6.0, t0


def _irr_block(case, seed):
    rng = np.random.default_rng([seed, case["n"], case["ni"]])
    addr = np.sort(rng.choice(case["n"], size=case["ni"], replace=False)).astype(np.int32) + 1
    return 8.0 / 256.0 + rng.integers(0, 64) / 65536.0, addr


def _samples(case, seed):
    rng = np.random.default_rng([seed, case["samples"]])
    f = rng.normal(size=(8, case["samples"])).astype(np.float32)
    t = 0.1 * f[0] - 0.05 * f[1] * f[2] + 0.1 * np.tanh(f[5]) + 0.02 * rng.normal(size=f.shape[1])
    return f, t.astype(np.float32)


# ---------------------------------------------------------------------- the library
_open = {"gpunb": None, "ens": False, "irr": None}


def _check(rc=0):
    if rc:
        lib.check_error()
        raise RuntimeError(f"the call returned {rc}")


def _gpunb():
    if _open["gpunb"] is None:
        _open["gpunb"] = lib.Gpunb(N_MAX)
    return lib.load()


def _irr_store(case):
    """The irregular-force library holding the case's cluster: predictor records and the
    neighbour lists of one regular step of all particles."""
    key = (case["n"], case["lmax"], case["nnb"])
    L = _gpunb()
    if _open["irr"] and _open["irr"][0] == key:
        return L
    if _open["irr"]:
        for o in _open["irr"][1:]:
            o.close()
    n, lmax = case["n"], case["lmax"]
    m, x, v, h2, f, fd, t0 = _irr_cluster(case)
    irr, jp = lib.IrrSimd(n, lmax), lib.JPred(n)
    addr = np.arange(1, n + 1, dtype=np.int32)
    jp.set(addr, x, v, f, fd, m, t0)
    L.nb6_irr_sync_jp_(ctypes.byref(ctypes.c_int(n)))
    j = _gpu(_soa(x, v, m))
    i = _gpu(_soa(x, v, h2, np.full(n, 2.0 ** -7)))
    out = torch.zeros((7, n), dtype=torch.float64, device="cuda")
    rows = torch.zeros((n, lmax), dtype=torch.int32, device="cuda")
    da = _gpu(addr)
    torch.cuda.synchronize()
    _check(L.nb6_send_device(n, n, j.data_ptr(), None))
    _check(L.nb6_regf_device(n, n, i.data_ptr(), lmax, lmax - 1, 0, out.data_ptr(),
                             rows.data_ptr(), None))
    torch.cuda.synchronize()
    _check(L.nb6_irr_set_lists_device(n, da.data_ptr(), rows.data_ptr(), lmax, 1, None))
    torch.cuda.synchronize()
    _open["irr"] = (key, irr, jp)
    return L


def _force_out(ni, lmax):
    out = torch.zeros((7, ni), dtype=torch.float64, device="cuda")
    rows = torch.zeros((ni, lmax), dtype=torch.int32, device="cuda")
    return out, rows, {"acc": out[0:3], "jrk": out[3:6], "pot": out[6], "list": rows}


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind in ("host", "device"):
        L = _gpunb()
        m, x, v, idx, h2, dtr = _block(case, seed)
        n, ni, lmax = case["n"], case["ni"], case["lmax"]
        nnbmax = lmax - 50
        if kind == "device":
            j = _gpu(_soa(x, v, m))
            i = _gpu(_soa(x[idx], v[idx], h2, dtr))
            out, rows, s["out"] = _force_out(ni, lmax)
            s["keep"] = (j, i, out, rows)
            s["send"] = (n, n, j.data_ptr(), None)
            s["regf"] = (ni, ni, i.data_ptr(), lmax, nnbmax, case["m_flag"], out.data_ptr(),
                         rows.data_ptr(), None)
        else:
            xi, vi = x[idx].copy(), v[idx].copy()
            acc, jrk, pot = np.zeros((ni, 3)), np.zeros((ni, 3)), np.zeros(ni)
            rows = np.zeros((ni, lmax), np.int32)
            s["keep"] = (m, x, v, h2, dtr, xi, vi)
            s["send"] = (lib._ri(n), lib._d(m), lib._d(x), lib._d(v))
            s["regf"] = (lib._ri(ni), lib._d(h2), lib._d(dtr), lib._d(xi), lib._d(vi),
                         lib._d(acc), lib._d(jrk), lib._d(pot), lib._ri(lmax), lib._ri(nnbmax),
                         lib._i(rows), lib._ri(case["m_flag"]))
            s["out"] = {"acc": acc, "jrk": jrk, "pot": pot, "list": rows}
    elif kind == "ensemble":
        L = lib.load()
        if not _open["ens"]:
            _check(L.nb6_ens_open(ENS_CLUSTERS, ENS_PARTICLES))
            _open["ens"] = True
        off, m, x, v, h2, dtr = _ensemble(case, seed)
        n, lmax = len(m), case["lmax"]
        j, i = _gpu(_soa(x, v, m)), _gpu(_soa(x, v, h2, dtr))
        out, rows, s["out"] = _force_out(n, lmax)
        s["keep"] = (off, j, i, out, rows)
        s["send"] = (case["clusters"], lib._i(off), j.data_ptr(), n, None)
        s["regf"] = (i.data_ptr(), n, lmax, lmax - 50, 0, out.data_ptr(), rows.data_ptr(), 0, None)
    elif kind == "pot_host":
        L = lib.load()
        s["m"], s["x"], _ = _cluster(np.random.default_rng([seed, case["n"]]), case["n"],
                                     case["binaries"])
    elif kind == "pot":
        L = lib.load()
        n = case["n"]
        m, x, _ = _cluster(np.random.default_rng([seed, n]), n, case["binaries"])
        d = _gpu(np.concatenate([x.T, m[None]]))
        s["out"] = torch.zeros(n, dtype=torch.float64, device="cuda")
        s["keep"] = d
        s["call"] = (n, n, d.data_ptr(), 0, n, s["out"].data_ptr(), None)
    elif kind in ("irr", "irr_host"):
        L = _irr_store(case)
        ti, addr = _irr_block(case, seed)
        ni = len(addr)
        if kind == "irr":
            d = _gpu(addr)
            out = torch.zeros((ni, 8), dtype=torch.float64, device="cuda")
            s["keep"] = (d, out)
            s["call"] = (ti, ni, d.data_ptr(), out.data_ptr(), None)
            s["out"] = {"acc": out[:, 0:3], "jrk": out[:, 3:6], "nearest": out[:, 6],
                        "count": out[:, 7]}
        else:
            acc, jrk = np.zeros((ni, 3)), np.zeros((ni, 3))
            near = np.zeros(ni, np.int32)
            s["keep"] = addr
            s["call"] = (lib._rd(ti), lib._ri(ni), lib._i(addr), lib._d(acc), lib._d(jrk),
                         lib._i(near))
            s["out"] = {"acc": acc, "jrk": jrk, "nearest": near}
    else:
        L = _gpunb()
        f, t = _samples(case, seed)
        s["keep"] = (_gpu(f), _gpu(t), np.zeros(8, np.float32), np.ones(8, np.float32))
        s["w"] = np.zeros(L.nb6_rsnet_nparam(), np.float32)
        s["loss"] = ctypes.c_float()
        s["norm"] = tuple(a.ctypes.data for a in s["keep"][2:])
        s["epoch"] = (case["samples"], s["keep"][0].data_ptr(), s["keep"][1].data_ptr(),
                      case["batch"], 2e-3, 1 + seed, ctypes.addressof(s["loss"]), None)
    s["L"] = L
    return s


def run(state):
    s, L, kind = state, state["L"], state["kind"]
    if kind == "device":
        _check(L.nb6_send_device(*s["send"]))
        _check(L.nb6_regf_device(*s["regf"]))
    elif kind == "host":
        L.gpunb_send_(*s["send"])
        L.gpunb_regf_(*s["regf"])
        lib.check_error()
    elif kind == "ensemble":
        _check(L.nb6_ens_send_device(*s["send"]))
        _check(L.nb6_ens_regf_device(*s["regf"]))
    elif kind == "pot_host":
        return {"pot": lib.gpupot(s["m"], s["x"])}
    elif kind == "pot":
        _check(L.nb6_pot_device(*s["call"]))
    elif kind == "irr":
        _check(L.nb6_irr_firr_device(*s["call"]))
    elif kind == "irr_host":
        L.irr_simd_firr_vec_(*s["call"])
        lib.check_error()
    else:
        _check(L.nb6_rsnet_open(7))
        _check(L.nb6_rsnet_set_norm(*s["norm"]))
        _check(L.nb6_rsnet_train_epoch_device(*s["epoch"]))
        _check(L.nb6_rsnet_get_params(s["w"].ctypes.data))
        return {"weights": s["w"], "loss": np.float32(s["loss"].value)}
    return s["out"]


# ---------------------------------------------------------------------- work
def work(case):
    kind = case["kind"]
    if kind in ("host", "device"):
        n, ni = case["n"], case["ni"]
        return {"bytes": 56 * n + (64 + 56 + 4 * (case["nnb"] + 1)) * ni,
                "flops": PAIR_FLOPS * n * ni}
    if kind == "ensemble":
        srng = np.random.default_rng([case["clusters"], case["n_lo"], case["n_hi"]])
        sz = np.exp(srng.uniform(math.log(case["n_lo"]), math.log(case["n_hi"]),
                                 case["clusters"])).astype(np.int64)
        n = int(sz.sum())
        return {"bytes": (56 + 64 + 56 + 4 * (case["nnb"] + 1)) * n,
                "flops": PAIR_FLOPS * int((sz * sz).sum())}
    if kind in ("pot", "pot_host"):
        n = case["n"]
        return {"bytes": 40 * n, "flops": POT_FLOPS * n * n}
    if kind in ("irr", "irr_host"):
        # list entry, 64-byte record and time of every neighbour; own record, result
        ni, k = case["ni"], case["nnb"]
        return {"bytes": ni * (k * 76 + 72 + 64), "flops": PAIR_FLOPS * ni * k}
    n = case["samples"]
    # 4,672 weights, three products each (forward, weight gradient, back-propagated delta)
    return {"bytes": 36 * n, "flops": 6 * 4672 * n}


# ---------------------------------------------------------------------- 64-bit results
def _dev(a):
    t = torch.from_numpy(np.ascontiguousarray(a))
    return t.cuda() if torch.cuda.is_available() else t


def _pairs64(xj, vj, mj, xi, vi, h2, dtr, m_flag):
    """Regular force of i over the j that are not its neighbours, [7][ni]."""
    n, out = len(mj), []
    step = max(1, (1 << 26) // n)
    for a in range(0, len(h2), step):
        sl = slice(a, a + step)
        d = [xj[:, k][None] - xi[sl, k][:, None] for k in range(3)]
        w = [vj[:, k][None] - vi[sl, k][:, None] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        r2p = 0.0
        for k in range(3):
            e = d[k] + dtr[sl][:, None] * w[k]
            r2p = r2p + e * e
        thr = mj[None] * h2[sl][:, None] if m_flag else h2[sl][:, None]
        use = ~(torch.minimum(r2, r2p) < thr) & (r2 > 0)
        ri = torch.where(use, r2, torch.ones_like(r2)).rsqrt()
        mr = torch.where(use, mj[None].expand_as(ri), torch.zeros_like(ri)) * ri
        m3 = mr * ri * ri
        al = -3.0 * (d[0] * w[0] + d[1] * w[1] + d[2] * w[2]) * ri * ri
        out.append(torch.stack([(m3 * d[k]).sum(1) for k in range(3)]
                               + [(m3 * (w[k] + al * d[k])).sum(1) for k in range(3)]
                               + [mr.sum(1)]))
    return torch.cat(out, dim=1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("host", "device"):
        if case["n"] * case["ni"] > 3e10:
            return None
        m, x, v, idx, h2, dtr = _block(case, seed)
        f = _pairs64(_dev(x), _dev(v), _dev(m), _dev(x[idx]), _dev(v[idx]), _dev(h2), _dev(dtr),
                     case["m_flag"])
        o = {"acc": f[0:3], "jrk": f[3:6], "pot": f[6], "list": None}
        if kind == "host":
            o["acc"], o["jrk"] = o["acc"].T, o["jrk"].T
        return o
    if kind == "ensemble":
        off, m, x, v, h2, dtr = _ensemble(case, seed)
        f = torch.cat([_pairs64(*(_dev(a) for a in (x[s], v[s], m[s], x[s], v[s], h2[s], dtr[s])), 0)
                       for s in (slice(a, b) for a, b in zip(off[:-1], off[1:]))], dim=1)
        return {"acc": f[0:3], "jrk": f[3:6], "pot": f[6], "list": None}
    if kind in ("pot", "pot_host"):
        n = case["n"]
        m, x, _ = _cluster(np.random.default_rng([seed, n]), n, case["binaries"])
        m, x = _dev(m), _dev(x)
        out = []
        step = max(1, (1 << 27) // n)
        for a in range(0, n, step):
            r2 = 0.0
            for k in range(3):
                d = x[:, k][None] - x[a:a + step, k][:, None]
                r2 = r2 + d * d
            out.append(torch.where(r2 > 0, m[None] * r2.rsqrt(), torch.zeros_like(r2)).sum(1))
        p = torch.cat(out)
        return p if kind == "pot" else {"pot": p}
    if kind in ("irr", "irr_host"):
        m, x, v, h2, f, fd, t0 = (_dev(a) for a in _irr_cluster(case))
        ti, addr = _irr_block(case, seed)
        i = _dev(addr.astype(np.int64) - 1)
        s = (ti - t0)[:, None]
        xp = x + s * (v + s * (f + s * fd))
        vp = v + 2 * s * (f + 1.5 * s * fd)
        n, res = case["n"], []
        step = max(1, (1 << 26) // n)
        for a in range(0, len(i), step):
            k = i[a:a + step]
            r2 = r2p = 0.0
            for c in range(3):
                d = x[:, c][None] - x[k, c][:, None]
                e = d + 2.0 ** -7 * (v[:, c][None] - v[k, c][:, None])
                r2, r2p = r2 + d * d, r2p + e * e
            lst = torch.minimum(r2, r2p) < h2[k][:, None]
            lst &= (lst.sum(1) <= case["lmax"] - 1)[:, None]
            lst[torch.arange(len(k), device=lst.device), k] = False
            row, col = lst.nonzero(as_tuple=True)
            d, w = xp[col] - xp[k[row]], vp[col] - vp[k[row]]
            q2 = (d * d).sum(1)
            m3 = m[col] * q2 ** -1.5
            al = -3.0 * (d * w).sum(1) / q2
            o = torch.zeros((len(k), 6), dtype=torch.float64, device=x.device)
            o.index_add_(0, row, torch.cat([m3[:, None] * d, m3[:, None] * (w + al[:, None] * d)], 1))
            res.append(o)
        o = torch.cat(res)
        r = {"acc": o[:, 0:3], "jrk": o[:, 3:6], "nearest": None}
        return r if kind == "irr_host" else {**r, "count": None}
    return None      # training: the minibatch order is the library's own

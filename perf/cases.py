"""Workloads of the framework as its users run them, for timing and comparing builds.

Four kinds of case, each through public entry points:

* ``step``   -- step_ch() on a grid resident on the GPU (Harm3D), a number of steps between
  two reads of the state by the host program: shock tube, black-hole torus, binary disk;
* ``c2p``    -- batched con-to-prim of independent zones in the caller's device memory;
* ``train``  -- training of the guess network of the batched con-to-prim;
* ``metric`` -- records and connection of the binary-black-hole metric on a block.

Only grids and options that the repository's own tests, benchmark and problem set-ups use.
"""
import ctypes
import dataclasses
import functools
import math

import numpy as np
import torch

from coolharm3d_amd import _lib
from coolharm3d_amd.c2p import Con2PrimBatch
from coolharm3d_amd.harm import Harm3D
from coolharm3d_amd.pn import CENT, CORN, FACE1, FACE2, FACE3, PnMetric, bbh_block
from coolharm3d_amd.problems import (NG, balsara1, balsara1_grid, bbh_disk, bbh_gdet, bbh_grid, torus, torus_grid)

A_SPIN, GAM = 0.9, 5.0 / 3.0
DEV = "cuda"
MAX_ZONES = 192 * 192 * 128


# ---------------------------------------------------------------------------
# The cases

def _step(name, problem, n, steps, precision="fp64", graph=True, sync="state", coords="mks", recon="ppm"):
    return {"name": name, "kind": "step", "problem": problem, "n1": n[0], "n2": n[1], "n3": n[2], "steps": steps,
            "precision": precision, "graph": graph, "sync": sync, "coords": coords, "recon": recon}


def listed():
    return [
        # the smallest grid: a 1D shock tube, where launches are everything; the host reads the
        # state every 10 steps (the driver's energy diagnostics)
        _step("shock_1024", "shock", (1024, 1, 1), 10, coords="identity", recon="mc"),
        # a small block stepped from a C driver that keeps its own arrays: one eager step, then
        # everything the drop-in step_ch() copies back after each step
        _step("torus_24x24x16_driver", "torus", (24, 24, 16), 1, graph=False, sync="driver"),
        # ragged medium block, and the driver's own sync on a block of the size a rank gets
        _step("torus_67x45x33", "torus", (67, 45, 33), 10),
        _step("torus_96x96x64_driver", "torus", (96, 96, 64), 1, graph=False, sync="driver"),
        # mixed precision on the other theta map
        _step("torus_96x96x64_mixed", "torus", (96, 96, 64), 20, precision="mixed", coords="diag3"),
        # production torus, 100 steps between two reads of the state, both precisions
        _step("torus_192x192x128", "torus", (192, 192, 128), 100),
        _step("torus_192x192x128_mixed", "torus", (192, 192, 128), 100, precision="mixed"),
        # circumbinary disk on the time-dependent metric
        _step("disk_120x64x160_mixed", "disk", (120, 64, 160), 20, precision="mixed"),
        # batched con-to-prim: a large batch from the cold guess, an odd small one from the previous
        # primitives (the reference's guess), and one from the learned guess
        {"name": "c2p_cold_2e24", "kind": "c2p", "n": 1 << 24, "guess": "cold", "compact": True},
        {"name": "c2p_prim_100003", "kind": "c2p", "n": 100003, "guess": "prim", "compact": False},
        {"name": "c2p_learned_2e22", "kind": "c2p", "n": 1 << 22, "guess": "learned", "compact": True},
        # training the guess network, batches of 4096 as train_guess() draws them
        {"name": "train_4096x25", "kind": "train", "n": 1 << 18, "batch": 4096, "steps": 25},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["shock", "torus", "torus", "torus", "disk", "c2p", "c2p", "train", "metric"])
    if what == "shock":
        # even: an odd grid has a zone centred on the origin, where the floors' power of |x| diverges
        c = _step("", "shock", (2 * _log(rng, 32, 4096), 1, 1), rng.randint(1, 10), coords="identity", recon="mc",
                  graph=rng.random() < 0.7)
    elif what in ("torus", "disk"):
        while True:
            n = (_log(rng, 13, 220), _log(rng, 12, 200), _log(rng, 8, 200))
            if n[0] * n[1] * n[2] <= (MAX_ZONES if what == "torus" else MAX_ZONES // 3):
                break
        driver = rng.random() < 0.25
        c = _step("", what, n, 1 if driver else rng.randint(2, 20), precision=rng.choice(["fp64", "mixed"]),
                  graph=not driver, sync="driver" if driver else "state", coords=rng.choice(["mks", "diag3"]),
                  recon="ppm" if what == "disk" or rng.random() < 0.8 else "mc")
    elif what == "c2p":
        guess = rng.choice(["cold", "prim", "learned"])
        c = {"kind": "c2p", "n": _log(rng, 1000, 1 << 23), "guess": guess, "compact": rng.random() < 0.5}
    elif what == "train":
        c = {"kind": "train", "n": _log(rng, 1000, 1 << 18), "batch": _log(rng, 64, 8192), "steps": rng.randint(1, 25)}
    else:
        c = {"kind": "metric", "n1": _log(rng, 1, 40), "n2": _log(rng, 5, 160), "n3": _log(rng, 5, 200),
             "pos": rng.choice([FACE1, FACE2, FACE3, CENT, CORN]), "coords": rng.choice(["mks", "diag3"])}
    c.pop("name", None)
    return c


# ---------------------------------------------------------------------------
# Grids

def _ptr(a):
    return a.ctypes.data_as(_lib.c_double_p if a.dtype == np.float64 else _lib.c_int_p)


def _prepare_step(case, seed):
    n = (case["n1"], case["n2"], case["n3"])
    kw = {"precision": case["precision"]}
    if case["recon"] == "mc" and case["problem"] != "shock":
        kw.update(recon=2, ct_para=0, flux=0)       # MC slopes, Lax-Friedrichs, arithmetic EMFs
    if case["problem"] == "shock":
        grid = dataclasses.replace(balsara1_grid(n[0], dt0=1.0e-6), t_end=1.0e9)
        p = balsara1(grid)
        rng = np.random.default_rng(seed)
        p[..., :2] *= 1.0 + 0.02 * (rng.random((p.shape[0], 1, 1, 2)) - 0.5)
    elif case["problem"] == "torus":
        grid = torus_grid(*n, coords=case["coords"])
        p = torus(grid, seed=seed)
    else:
        grid = bbh_grid(*n, coords=case["coords"])
        p = bbh_disk(grid, bbh_gdet(grid, PnMetric), seed=seed)
    H = Harm3D(grid, **kw)
    H.set_prims(p)
    H.fixup_bounds()
    H.set_time(0.0, grid.dx[0])
    if case["graph"]:
        H.set_graph(True)
    st = {"case": case, "H": H}
    if case["sync"] == "driver":
        st["p"], st["gamma"] = np.zeros(H.shape + (8,)), np.zeros(H.shape)
        st["pflag"], st["nfail"] = np.zeros(H.shape, np.int32), np.zeros((15,) + H.shape, np.int32)
    return st


def _run_step(st):
    H, case = st["H"], st["case"]
    if case["steps"] < 100:
        # a restart from the state at hand, with the small first time step that restarts take (it grows
        # by at most 1.3 per step): thousands of passes then stay within the problem's life
        H.set_time(0.0, H.grid.dx[0])
    H.step_ch(case["steps"])
    if case["sync"] == "driver":
        lib, h = H.lib, H.h
        _lib.check(lib, lib.hgpu_download_prims(h, 0, _ptr(st["p"])), "hgpu_download_prims")
        _lib.check(lib, lib.hgpu_download_gamma(h, _ptr(st["gamma"])), "hgpu_download_gamma")
        _lib.check(lib, lib.hgpu_download_pflag(h, _ptr(st["pflag"])), "hgpu_download_pflag")
        _lib.check(lib, lib.hgpu_download_nfail(h, _ptr(st["nfail"])), "hgpu_download_nfail")
        t, dt, dt_old = H.time()
        return {"prims": st["p"], "gamma": st["gamma"], "pflag": st["pflag"], "nfail": st["nfail"],
                "nfailtot": H.nfailtot(), "m_tot": H.m_tot(), "dt": dt, "t": t}
    p = H.prims()
    t, dt, dt_old = H.time()
    return {"prims": p, "dt": dt, "t": t}


# ---------------------------------------------------------------------------
# Batched con-to-prim: zones on Kerr-Schild records.  The ranges are those of the library's
# own samples (hgpu_c2p_samples): r log-uniform in [1.3, 100], theta in [0.05, pi - 0.05], b^2/rho
# log-uniform in [1e-4, 1e2], u/rho in [1e-4, 10], Lorentz factors log-uniform from 1; to 10 here
# (beyond 15, a few zones in a million have no converged solution to compare).

def _zones(n, seed):
    """U[8][n], rth[2][n], primitives[8][n] in 64 bits, from the seed alone."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    u = torch.rand((14, n), generator=g, device=DEV, dtype=torch.float64)

    def logu(x, lo, hi):
        return torch.exp(math.log(lo) + x * (math.log(hi) - math.log(lo)))
    r, th = logu(u[0], 1.3, 100.0), 0.05 + u[1] * (math.pi - 0.1)
    gamma, sig, uor = logu(u[2], 1.0, 10.0), logu(u[3], 1e-4, 1e2), logu(u[4], 1e-4, 10.0)
    a = A_SPIN
    s2 = torch.sin(th) ** 2
    S = r * r + a * a * torch.cos(th) ** 2
    z = 2.0 * r / S
    g00, g01, g03 = z - 1.0, z, -z * a * s2
    g11, g13, g22 = 1.0 + z, -a * (1.0 + z) * s2, S
    g33 = s2 * (r * r + a * a * (1.0 + z * s2))
    gdet = S * torch.sin(th).abs()
    alpha = 1.0 / torch.sqrt(1.0 + z)
    beta1 = z / (1.0 + z)

    def direction(c, p):      # isotropic in the normal observer's frame
        c, p = 2.0 * c - 1.0, 2.0 * math.pi * p
        s = torch.sqrt(1.0 - c * c)
        e1, e2, e3 = s * torch.cos(p), s * torch.sin(p), c
        L00 = torch.sqrt(g11)
        L20 = g13 / L00
        x3 = e3 / torch.sqrt(g33 - L20 * L20)
        return (e1 - L20 * x3) / L00, e2 / torch.sqrt(g22), x3

    def lower(v):
        return (g00 * v[0] + g01 * v[1] + g03 * v[3], g01 * v[0] + g11 * v[1] + g13 * v[3], g22 * v[2],
                g03 * v[0] + g13 * v[1] + g33 * v[3])
    ut = torch.sqrt((gamma - 1.0) * (gamma + 1.0))
    v = [ut * x for x in direction(u[5], u[6])]
    B = list(direction(u[7], u[8]))
    ucon = (gamma / alpha, v[0] - gamma / alpha * beta1, v[1], v[2])
    ucov = lower(ucon)
    b0 = B[0] * ucov[1] + B[1] * ucov[2] + B[2] * ucov[3]
    bcon = [b0] + [(B[i] + b0 * ucon[i + 1]) / ucon[0] for i in range(3)]
    bcov = lower(bcon)
    scale = torch.sqrt(sig / sum(x * y for x, y in zip(bcon, bcov)))
    B, bcon, bcov = [x * scale for x in B], [x * scale for x in bcon], [x * scale for x in bcov]
    p = (GAM - 1.0) * uor
    eta, ptot = 1.0 + uor + p + sig, p + 0.5 * sig
    prim = torch.stack([torch.ones_like(r), uor] + v + B)
    T = [eta * ucon[0] * ucov[m] - bcon[0] * bcov[m] for m in range(4)]
    U = torch.stack([ucon[0], T[0] + ptot + ucon[0], T[1], T[2], T[3]] + B) * gdet
    guess = prim.clone()
    guess[:5] *= 1.0 + 0.1 * (2.0 * u[9:14] - 1.0)
    # scale-free invariants of the zone in the normal frame and the root's (W, gamma), for the network
    D = gamma
    Bsq = sum(x * y for x, y in zip([b * alpha for b in B], lower([0 * r] + [b * alpha for b in B])[1:]))
    W = (1.0 + GAM * uor) * gamma * gamma
    Bv = sum(alpha * b * x for b, x in zip(B, lower([0 * r] + v)[1:]))          # B.u~
    QdotB = -W / gamma * Bv
    vsq = 1.0 - 1.0 / gamma ** 2
    E = W - p + 0.5 * Bsq * (1.0 + vsq) - 0.5 * (QdotB / W) ** 2
    Qtsq = vsq * (W + Bsq) ** 2 - QdotB ** 2 * (Bsq + 2.0 * W) / W ** 2
    inv = {"D": D, "Bsq": Bsq, "QdotBsq": QdotB ** 2, "Qtsq": Qtsq, "E": E, "W": W, "gamma": gamma}
    return U, torch.stack([r, th]), prim, guess, inv


def _features(inv):
    """Inputs[n][8] and targets[n][2] of the guess network, as hgpu_mlp_features() defines them."""
    D, Bsq, QB, Q, E = (inv[k] for k in ("D", "Bsq", "QdotBsq", "Qtsq", "E"))
    Q = Q.clamp_min(0.0)
    f = [torch.log(Bsq / D + 1e-30), torch.log(Q / D ** 2 + 1e-30), torch.log(QB / D ** 3 + 1e-30), torch.log(E / D),
         torch.log((E - D - 0.5 * Bsq).abs() / D + 1e-12), torch.sqrt(Q) / E, Bsq / E, QB / (Bsq * Q + 1e-30)]
    return torch.stack(f, 1), torch.stack([torch.log(inv["W"] / D), torch.log(inv["gamma"])], 1)


def _unpack(w):
    """W1[8][64], b1, W2[64][64], b2, W3[64][2], b3 and the normalisations of a parameter blob."""
    o, out = 0, []
    for shape in ((8,), (8,), (8, 64), (64,), (64, 64), (64,), (64, 2), (2,), (2,), (2,)):
        m = int(np.prod(shape))
        out.append(w[o:o + m].reshape(shape))
        o += m
    return out


def _loss(w, x, y):
    mu, isd, W1, b1, W2, b2, W3, b3, ymu, ysd = _unpack(w)
    h = torch.nn.functional.gelu(((x - mu) * isd) @ W1 + b1, approximate="tanh")
    h = torch.nn.functional.gelu(h @ W2 + b2, approximate="tanh")
    return 0.5 * ((h @ W3 + b3 - (y - ymu) / ysd) ** 2).sum(1).mean()


def _blob(x, y, seed):
    """Initial parameters: normalisations from the data, Glorot-uniform weights."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    parts = [x.mean(0), 1.0 / x.std(0)]
    for shape in ((8, 64), (64,), (64, 64), (64,), (64, 2), (2,)):
        lim = math.sqrt(6.0 / sum(shape)) if len(shape) == 2 else 0.0
        parts.append(lim * (2.0 * torch.rand(shape, generator=g, device=DEV, dtype=torch.float64) - 1.0))
    return torch.cat([p.reshape(-1) for p in parts + [y.mean(0), y.std(0)]])


@functools.lru_cache(maxsize=1)
def _network():
    """The trained guess network that a user's program keeps (made here in 64 bits, then rounded)."""
    x, y = _features(_zones(1 << 16, 4242)[4])
    w = _blob(x, y, 1).requires_grad_(True)
    opt = torch.optim.Adam([w], lr=3e-3)
    fixed = torch.ones_like(w)
    fixed[:16] = 0.0
    fixed[-4:] = 0.0
    for k in range(300):
        at = slice((k % 16) * 4096, (k % 16) * 4096 + 4096)
        opt.param_groups[0]["lr"] = 3e-3 * 0.5 * (1.0 + math.cos(math.pi * k / 300))
        opt.zero_grad()
        _loss(w, x[at], y[at]).backward()
        w.grad *= fixed
        opt.step()
    return w.detach().float().contiguous()


def _prepare_c2p(case, seed):
    n = case["n"]
    U, rth, prim, guess, _ = _zones(n, seed)
    B = Con2PrimBatch()
    nbytes = int(B.lib.hgpu_c2p_workspace_bytes(n, 1 if case["compact"] else 0))
    return {"case": case, "lib": B.lib, "U": U, "rth": rth, "guess": guess if case["guess"] == "prim" else None,
            "mlp": _network() if case["guess"] == "learned" else None,
            "work": torch.empty(max(nbytes, 8), device=DEV, dtype=torch.uint8), "nbytes": nbytes,
            "prim": torch.zeros_like(prim), "code": torch.zeros(n, device=DEV, dtype=torch.int32),
            "iters": torch.zeros(n, device=DEV, dtype=torch.int32)}


def _run_c2p(st):
    case, lib = st["case"], st["lib"]
    if st["guess"] is not None:
        st["prim"].copy_(st["guess"])
    _lib.check(lib, lib.hgpu_c2p_solve(
        torch.cuda.current_stream().cuda_stream, case["n"], A_SPIN, GAM, st["U"].data_ptr(), st["rth"].data_ptr(),
        st["mlp"].data_ptr() if st["mlp"] is not None else None, 0 if case["guess"] == "prim" else 1,
        1 if case["compact"] else 0, 0, 0, st["work"].data_ptr() if case["compact"] else None, st["nbytes"],
        st["prim"].data_ptr(), st["code"].data_ptr(), st["iters"].data_ptr()), "hgpu_c2p_solve")
    p = st["prim"]
    return {"rho": p[0], "u": p[1], "v": p[2:5], "B": p[5:8], "code": st["code"], "iters": st["iters"]}


# ---------------------------------------------------------------------------
# Training: hgpu_mlp_train() from given weights on given features

def _prepare_train(case, seed):
    x, y = _features(_zones(case["n"], seed)[4])
    w0 = _blob(x, y, seed + 1)
    B = Con2PrimBatch()
    nbytes = int(B.lib.hgpu_mlp_workspace_bytes(case["batch"]))
    return {"case": case, "lib": B.lib, "seed": seed, "feat": x.t().float().contiguous(),
            "target": y.t().float().contiguous(), "w0": w0.float(), "w": w0.float(), "nbytes": nbytes,
            "work": torch.empty(nbytes, device=DEV, dtype=torch.uint8),
            "hist": torch.zeros(case["steps"], device=DEV, dtype=torch.float32)}


def _run_train(st):
    case, lib = st["case"], st["lib"]
    st["w"].copy_(st["w0"])
    _lib.check(lib, lib.hgpu_mlp_train(
        torch.cuda.current_stream().cuda_stream, case["n"], st["feat"].data_ptr(), st["target"].data_ptr(),
        st["seed"], case["steps"], case["batch"], 3e-3, st["work"].data_ptr(), st["nbytes"], st["w"].data_ptr(),
        st["hist"].data_ptr()), "hgpu_mlp_train")
    return {"w": st["w"], "loss": st["hist"]}


def _philox(key, ctr):
    """Philox4x32-10 (Salmon et al., SC11) on int64 tensors holding 32-bit words."""
    M = 0xFFFFFFFF

    def mul(m, c):                      # 32 x 32 -> (high, low) words, in 16-bit parts
        lo, hi = c & 0xFFFF, c >> 16
        t0, t1 = m * lo, m * hi         # below 2^48
        s = t0 + ((t1 & 0xFFFF) << 16)
        return ((t1 >> 16) + (s >> 32)) & M, s & M
    c, k = list(ctr), list(key)
    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c[0])
        h1, l1 = mul(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k[0], l1, h0 ^ c[3] ^ k[1], l0]
        k = [(k[0] + 0x9E3779B9) & M, (k[1] + 0xBB67AE85) & M]
    return c


def _exact_train(case, seed):
    """The same Adam steps (Kingma & Ba 2015, cosine-decayed rate) in 64 bits, on the batches that the
    library's documented counter-based draws give."""
    st = _prepare_train(case, seed)
    n, batch, steps = case["n"], case["batch"], case["steps"]
    x, y = st["feat"].t().double(), st["target"].t().double()
    w = st["w0"].double()
    m, v = torch.zeros_like(w), torch.zeros_like(w)
    fixed = torch.ones_like(w)
    fixed[:16] = 0.0
    fixed[-4:] = 0.0
    hist = []
    for t in range(1, steps + 1):
        d = t * batch + torch.arange(batch, device=DEV, dtype=torch.int64)
        z = torch.zeros_like(d)
        r = _philox((seed & 0xFFFFFFFF, seed >> 32), (d & 0xFFFFFFFF, d >> 32, z + 3, z))
        u = ((((r[0] << 21) ^ (r[1] >> 11)) & ((1 << 53) - 1)).double() + 0.5) / 9007199254740992.0
        k = (u * n).long().clamp_max(n - 1)
        w = w.detach().requires_grad_(True)
        loss = _loss(w, x[k], y[k])
        g, = torch.autograd.grad(loss, w)
        hist.append(loss.detach())
        with torch.no_grad():
            g = g * fixed
            m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
            lr = 3e-3 * 0.5 * (1.0 + math.cos(math.pi * (t - 1) / steps))
            w = w - lr * fixed * (m / (1 - 0.9 ** t)) / (torch.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
    return {"w": w.detach(), "loss": torch.stack(hist)}


# ---------------------------------------------------------------------------
# Binary metric on a block

def _prepare_metric(case, seed):
    rng = np.random.default_rng(seed)
    h = 0.3 if case["coords"] == "mks" else 0.0729419909586
    cfg = bbh_block(case["n1"], case["n2"], case["n3"], ghosts=0, h_slope=h, phi0=float(rng.uniform(0, 2 * math.pi)),
                    coords=case["coords"])
    M = PnMetric(cfg)
    n = case["n1"] * case["n2"] * case["n3"]
    return {"case": case, "M": M, "cfg": cfg, "t": float(rng.uniform(0.0, 500.0)),
            "geom": torch.zeros((n, 42), device=DEV, dtype=torch.float64),
            "conn": torch.zeros((n, 64), device=DEV, dtype=torch.float64)}


def _run_metric(st):
    lib, s = st["M"].lib, torch.cuda.current_stream().cuda_stream
    _lib.check(lib, lib.hgpu_pn_geometry(s, ctypes.byref(st["cfg"]), st["t"], st["case"]["pos"],
                                         st["geom"].data_ptr()), "hgpu_pn_geometry")
    _lib.check(lib, lib.hgpu_pn_connection(s, ctypes.byref(st["cfg"]), st["t"], st["conn"].data_ptr()),
               "hgpu_pn_connection")
    return {"geom": st["geom"], "conn": st["conn"]}


# ---------------------------------------------------------------------------

_PREPARE = {"step": _prepare_step, "c2p": _prepare_c2p, "train": _prepare_train, "metric": _prepare_metric}
_RUN = {"step": _run_step, "c2p": _run_c2p, "train": _run_train, "metric": _run_metric}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["case"]["kind"]](state)


def work(case):
    """Step: 320 B of state per zone and step (p read three times, written twice) and the state handed
    over once; about 6000 operations per zone and step (reconstruction, two face states, HLL, source
    terms, Newton).  Con-to-prim: U, position, solution, code and iterations of a zone, about 70
    operations per iteration.  Network: 9.5 kFLOP forward, twice that backward."""
    if case["kind"] == "step":
        n = (case["n1"], case["n2"], case["n3"])
        z, nt = n[0] * n[1] * n[2], (n[0] + 2 * NG) * (n[1] + 2 * NG) * (n[2] + 2 * NG)
        return {"bytes": 320.0 * z * case["steps"] + (64.0 if case["sync"] == "state" else 136.0) * nt,
                "flops": 6000.0 * z * case["steps"]}
    if case["kind"] == "c2p":
        n = case["n"]
        return {"bytes": (152.0 + (64.0 if case["guess"] == "prim" else 0.0)) * n,
                "flops": (900.0 + (9500.0 if case["guess"] == "learned" else 0.0)) * n}
    if case["kind"] == "train":
        return {"bytes": 40.0 * case["batch"] * case["steps"], "flops": 3 * 9500.0 * case["batch"] * case["steps"]}
    n = case["n1"] * case["n2"] * case["n3"]
    return {"bytes": 8.0 * (42 + 64) * n, "flops": 2000.0 * n}


def tolerance(case):
    """Step: states perturbed by one unit in the last place drift apart to 8e-14 in FP64; in mixed
    precision the FP32 faces' rounding grows to 5e-6 within two passes (against the FP64 step).
    Con-to-prim: 4e-12 from the true primitives (conditioning); an iteration more or less where the
    convergence test ties.  Training: 1.5e-6 from the steps in 64 bits."""
    if case["kind"] == "step":
        return {"rel": 2e-5, "differ": 1e-4} if case["precision"] == "mixed" else {"rel": 1e-11, "differ": 1e-5}
    if case["kind"] == "c2p":
        return {"rel": 2e-11, "differ": 1e-3}
    if case["kind"] == "train":
        return {"rel": 1e-5}
    return {"rel": 1e-12}


def exact(case, seed):
    """c2p: the primitives that the conserved variables were formed from; train: the steps in 64 bits.
    The step is in 64 bits itself (or mixes 32 and 64 by design) and has no closed form."""
    if case["kind"] == "c2p":
        p = _zones(case["n"], seed)[2]
        return {"rho": p[0], "u": p[1], "v": p[2:5], "B": p[5:8], "code": None, "iters": None}
    if case["kind"] == "train":
        return _exact_train(case, seed)
    return None

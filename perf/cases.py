"""The workloads this library is timed on: what a program that uses it has it
do, through the entry points such a program calls, over the range of sizes.

  flow      one case stepped by rk3: the miniapp's stage on the Taylor-Green
            vortex (three-dimensional) and on the isentropic vortex
            (two-dimensional), and the main solver's stage on the
            Taylor-Green vortex with its convective schemes.  `tuned` cases
            call autotune after the upload, as a long run does; the others
            keep the default launch selection, as the Fortran programs and
            the serving loop do;
  batch     many small independent cases advanced together;
  chem      chemical source terms of a list of cells, resident in HBM;
  ignition  0-D reactors set, run to t_end and read back, as the serving
            loop does for its ignition requests.

`exact` restates each path in plain torch (dense line operators, float64).
"""
import ctypes as C
import math
import xml.etree.ElementTree as ET

import numpy as np
import torch

import astr_amd as A
from astr_amd import chem as AC

MECHANISM = "tests/golden/Jachimowski88_H2-9-19.xml"
DEV = "cuda"
F8 = torch.float64


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _flow(name, path, im, jm, km, steps, tuned, conschm="643c", recon=0, chardec=False):
    return {"name": name, "family": "flow", "path": path, "im": im, "jm": jm, "km": km, "steps": steps,
            "tuned": tuned, "conschm": conschm, "recon": recon, "chardec": chardec}


def listed():
    return [
        # the smallest three-dimensional run the Fortran host is used for: one
        # step of the miniapp, statistics printed every step
        _flow("tgv_32", "tgv", 32, 32, 32, 1, False),
        # a box whose sides differ and divide nothing
        _flow("tgv_97x61x45", "tgv", 97, 61, 45, 1, True),
        # the reference example's own grid
        _flow("tgv_128", "tgv", 128, 128, 128, 1, True),
        # the headline workload
        _flow("tgv_256", "tgv", 256, 256, 256, 1, True),
        # a two-dimensional case of the served and batched mixes, ten steps
        # between two looks at it
        _flow("vortex_300x181", "vortex", 300, 181, 0, 10, False),
        # what `astr run` computes on its default scheme, untuned, on a box
        # with unequal sides
        _flow("main_96x80x63", "main", 96, 80, 63, 1, False),
        # the same stage on the reference example's grid, tuned
        _flow("main_128", "main", 128, 128, 128, 1, True),
        # shock-capturing convection, explicit (MP7)
        _flow("main_753e_mp7_96", "main", 96, 96, 96, 1, True, "753e", 3, False),
        # shock-capturing convection, compact, on characteristic variables
        _flow("main_543c_char_72", "main", 72, 72, 72, 1, True, "543c", 0, True),
        # the chemistry of a million cells
        {"name": "chem_1m", "family": "chem", "cells": 1 << 20},
        # a mixed batch, five steps
        {"name": "batch_12", "family": "batch", "cases": 12, "mix": 2026, "steps": 5},
        # ignition requests of one serving tick
        {"name": "ignition_40", "family": "ignition", "reactors": 40},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tgv", "tgv", "tgv", "vortex", "main", "main", "upwind", "chem", "batch", "ignition"])
    tuned = rng.random() < 0.6
    if kind == "tgv":
        n = _log_int(rng, 20, 210)
        im, jm, km = (max(12, int(round(n * rng.uniform(0.7, 1.2)))) for _ in range(3))
        c = _flow("", "tgv", im, jm, km, rng.choice([1, 1, 2]) if n < 120 else 1, tuned)
    elif kind == "vortex":
        im, jm = _log_int(rng, 64, 512), _log_int(rng, 64, 512)
        c = _flow("", "vortex", im, jm, 0, rng.choice([5, 10]), tuned)
    elif kind == "main":
        n = _log_int(rng, 20, 170)
        im, jm, km = (max(12, int(round(n * rng.uniform(0.7, 1.2)))) for _ in range(3))
        c = _flow("", "main", im, jm, km, 1, tuned)
    elif kind == "upwind":
        n = _log_int(rng, 24, 100)
        im, jm, km = (max(12, int(round(n * rng.uniform(0.8, 1.2)))) for _ in range(3))
        conschm = rng.choice(["753e", "753e", "543c"])
        c = _flow("", "main", im, jm, km, 1, tuned, conschm, rng.choice([1, 3]) if conschm == "753e" else 0,
                  rng.random() < 0.5)
    elif kind == "chem":
        return {"family": "chem", "cells": _log_int(rng, 1000, 1 << 20)}
    elif kind == "batch":
        return {"family": "batch", "cases": rng.randint(4, 16), "mix": rng.randrange(1 << 20), "steps": rng.choice([2, 5])}
    else:
        return {"family": "ignition", "reactors": _log_int(rng, 4, 64)}
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
REYNOLDS = 1600.0


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _config(c):
    if c["path"] == "vortex":
        return A.vortex_config(c["im"], c["jm"])
    make = A.main_config if c["path"] == "main" else A.tgv_config
    return make(c["im"], c["jm"], c["km"], deltat=0.128 / max(c["im"], c["jm"], c["km"]), reynolds=REYNOLDS)


def _close(f, n):
    """f on i, j, k < n with the duplicate planes i = im, j = jm, k = km."""
    for d in range(3):
        if n[d] > 0:
            f = torch.cat([f, f.narrow(2 - d, 0, 1)], dim=2 - d)
    return f


def _tgv(cfg, seed):
    """The Taylor-Green vortex with 1e-3 Gaussian velocity noise."""
    n = (cfg.im, cfg.jm, cfg.km)
    x, y, z = (torch.arange(m, device=DEV, dtype=F8) * (2 * math.pi / m) for m in n)
    x, y, z = x[None, None, :], y[None, :, None], z[:, None, None]
    g = _gen(seed)
    noise = [1e-3 * torch.randn(n[2], n[1], n[0], generator=g, device=DEV, dtype=F8) for _ in range(3)]
    u = torch.sin(x) * torch.cos(y) * torch.cos(z) + noise[0]
    v = -torch.cos(x) * torch.sin(y) * torch.cos(z) + noise[1]
    w = noise[2]
    p = 1.0 / (cfg.gamma * cfg.mach ** 2) + (torch.cos(2 * x) + torch.cos(2 * y)) * (torch.cos(2 * z) + 2.0) / 16.0
    e = p / (cfg.gamma - 1.0) + 0.5 * (u * u + v * v + w * w)
    return torch.stack([_close(f, n) for f in (torch.ones_like(u), u, v, w, e)])


def _vortex(cfg, seed):
    """An isentropic vortex of seeded strength and centre in a free stream."""
    g = _gen(seed)
    r = torch.rand(3, generator=g, device=DEV, dtype=F8)
    beta, xc, yc = 4.0 + 2.0 * r[0], cfg.lx * (0.4 + 0.2 * r[1]), cfg.ly * (0.4 + 0.2 * r[2])
    x = (torch.arange(cfg.im, device=DEV, dtype=F8) * (cfg.lx / cfg.im))[None, None, :] - xc
    y = (torch.arange(cfg.jm, device=DEV, dtype=F8) * (cfg.ly / cfg.jm))[None, :, None] - yc
    gm1, ma2 = cfg.gamma - 1.0, cfg.mach ** 2
    e = torch.exp(0.5 * (1.0 - (x * x + y * y)))
    u = 1.0 - beta / (2 * math.pi) * y * e
    v = beta / (2 * math.pi) * x * e
    t = 1.0 - gm1 * ma2 * beta ** 2 / (8 * math.pi ** 2) * e * e
    rho = t ** (1.0 / gm1)
    p = rho * t / (cfg.gamma * ma2)
    f = (rho, rho * u, rho * v, torch.zeros_like(rho), p / gm1 + 0.5 * rho * (u * u + v * v))
    return torch.stack([_close(s, (cfg.im, cfg.jm, 0)) for s in f])


def _initial(path, cfg, seed):
    return _vortex(cfg, seed) if path == "vortex" else _tgv(cfg, seed)


class _Resident:
    """A context's resident q as an array on the device, without a copy.  A
    tensor made of it holds it, and it holds the context, whose memory q is."""

    def __init__(self, flow):
        self.flow = flow
        lay = A.Layout()
        if A.lib().astr_hip_field_info(flow.h, C.byref(lay)) != 0:
            raise RuntimeError("astr_hip_field_info failed")
        self.__cuda_array_interface__ = {
            "shape": (5,) + flow.shape, "typestr": "<f8", "version": 3, "data": (lay.q, False),
            "strides": (8 * lay.field_stride, 8 * lay.plane, 8 * lay.pitch, 8)}


def _resident_q(flow):
    return torch.as_tensor(_Resident(flow), device=DEV)


def _batch_specs(c):
    """(path, config, seed offset) of a mixed batch's cases: vortices of side
    64..256 and Taylor-Green vortices of side 32..96, in turn."""
    rng = np.random.default_rng(c["mix"])
    out = []
    for k in range(c["cases"]):
        if k % 2 == 0:
            n = int(rng.integers(64, 257))
            out.append(("vortex", A.vortex_config(n), k))
        else:
            n = int(rng.integers(32, 97))
            out.append(("tgv", A.tgv_config(n, deltat=0.128 / n, reynolds=float(rng.uniform(100.0, 3000.0))), k))
    return out


def _cells(W, ix, n, seed):
    """T, p and Y (species, cells) of H2-air cells between the unburnt mixture
    and its combustion products with a radical pool."""
    g = _gen(seed)
    r = torch.rand(4, n, generator=g, device=DEV, dtype=F8)
    T = 900.0 + 1600.0 * r[0]
    p = 101325.0 * torch.exp(math.log(0.5) + math.log(10.0) * r[1])
    phi, c = 0.3 + 2.7 * r[2], r[3]
    Xu, Xb = torch.zeros(2, len(W), n, device=DEV, dtype=F8)
    Xu[ix["H2"]], Xu[ix["O2"]], Xu[ix["N2"]] = 2.0 * phi, 1.0, 0.79 / 0.21
    Xb[ix["H2O"]] = 2.0 * phi.clamp(max=1.0)
    Xb[ix["O2"]], Xb[ix["H2"]] = (1.0 - phi).clamp(min=0.0), 2.0 * (phi - 1.0).clamp(min=0.0)
    Xb[ix["N2"]] = 0.79 / 0.21
    Xb = Xb / Xb.sum(0)
    for s, v in (("OH", 1e-3), ("H", 1e-3), ("O", 1e-3), ("HO2", 1e-5), ("H2O2", 1e-5)):
        Xb[ix[s]] += v
    W = torch.tensor(np.asarray(W), device=DEV, dtype=F8)[:, None]
    Yu, Yb = Xu * W, Xb * W
    Y = (1.0 - c) * (Yu / Yu.sum(0)) + c * (Yb / Yb.sum(0))
    return T, p, (Y / Y.sum(0)).contiguous()


# ---------------------------------------------------------------------------
# prepare, run
# ---------------------------------------------------------------------------
def _make_flow(path, cfg, seed):
    f = A.Flow(cfg)
    f.upload(_initial(path, cfg, seed).cpu().numpy())
    return f


def prepare(case, seed):
    c = case
    if c["family"] == "flow":
        f = _make_flow(c["path"], _config(c), seed)
        if c["conschm"] != "643c":
            f.set_conschm(c["conschm"], c["recon"], c["chardec"])
        if c["tuned"]:
            f.autotune(3)
        return {"case": c, "flow": f, "q": _resident_q(f)}
    if c["family"] == "batch":
        flows = [_make_flow(path, cfg, seed * 64 + k) for path, cfg, k in _batch_specs(c)]
        b = A.Batch(flows)
        b.autotune(2)
        return {"case": c, "batch": b, "flows": flows, "q": [_resident_q(f) for f in flows]}
    mech = AC.Mechanism(MECHANISM)
    ix = {s: k for k, s in enumerate(mech.names)}
    if c["family"] == "chem":
        n = c["cells"]
        T, p, Y = _cells(mech.W, ix, n, seed)
        out = {"wdot": torch.empty(mech.ns, n, device=DEV, dtype=F8), "h": torch.empty(n, device=DEV, dtype=F8),
               "cp": torch.empty(n, device=DEV, dtype=F8)}
        return {"case": c, "mech": mech, "T": T, "p": p, "Y": Y, "out": out}
    rng = np.random.default_rng(seed)
    reqs = []
    for _ in range(c["reactors"]):
        phi = rng.uniform(0.5, 2.0)
        X = np.zeros(mech.ns)
        X[ix["H2"]], X[ix["O2"]], X[ix["N2"]] = 2.0 * phi, 1.0, 3.76
        Y = X * mech.W
        reqs.append((rng.uniform(950.0, 1400.0), rng.uniform(1.0, 10.0) * 101325.0, Y / Y.sum()))
    pool = AC.ReactorPool(mech, 64, rtol=1e-5, atol=1e-10)
    return {"case": c, "mech": mech, "pool": pool, "requests": reqs}


def run(state):
    c = state["case"]
    if c["family"] == "flow":
        f = state["flow"]
        if c["path"] == "vortex":
            f.rk3(c["steps"], stats=False)
            return {"q": state["q"]}
        if c["path"] == "main":
            ke, en, di = f.rk3(c["steps"], dissipation=True)
            return {"q": state["q"], "ke": ke, "en": en, "di": di}
        ke, en = f.rk3(c["steps"])
        return {"q": state["q"], "ke": ke, "en": en}
    if c["family"] == "batch":
        ke, en = state["batch"].rk3(c["steps"])
        return {"q": state["q"], "ke": ke, "en": en}
    if c["family"] == "chem":
        o, mech = state["out"], state["mech"]
        rc = A.lib().astr_hip_chem_rates_device(
            mech.h, c["cells"], state["T"].data_ptr(), state["p"].data_ptr(), 1, state["Y"].data_ptr(),
            o["wdot"].data_ptr(), o["h"].data_ptr(), o["cp"].data_ptr(), None, None)
        if rc != 0:
            raise RuntimeError(A.lib().astr_hip_chem_last_error().decode())
        return o
    pool = state["pool"]
    for s, (T, p, Y) in enumerate(state["requests"]):
        pool.set(s, T, p, Y, 1e-3)
    pool.run(100)
    got = [pool.get(s) for s in range(c["reactors"])]
    for s in range(c["reactors"]):
        pool.release(s)
    return {"T": np.array([g[1] for g in got]), "Y": np.array([g[2] for g in got])}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _flow_work(cfg, steps, upwind=0):
    # the state in and out once; per point and stage the operators' arithmetic:
    # nine line derivatives and five filtered lines per direction, the
    # pointwise fluxes, stresses and update
    pts = (cfg.im + 1) * (cfg.jm + 1) * (cfg.km + 1)
    nd = 3 if cfg.km > 0 else 2
    per = nd * (9 * 9 + 5 * 22 + upwind) + 130
    return {"bytes": 80.0 * pts, "flops": 3.0 * per * pts * steps}


def work(case):
    c = case
    if c["family"] == "flow":
        return _flow_work(_config(c), c["steps"], 0 if c["conschm"] == "643c" else (900 if c["chardec"] else 350))
    if c["family"] == "batch":
        w = [_flow_work(cfg, c["steps"]) for _, cfg, _ in _batch_specs(c)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    if c["family"] == "chem":
        return {"bytes": 176.0 * c["cells"], "flops": 1600.0 * c["cells"]}
    # about 170 integration steps, each six right-hand sides, ten Jacobian
    # columns and one 10 x 10 factorisation with six solves
    return {"bytes": 200.0 * c["reactors"], "flops": 170.0 * (16 * 1500.0 + 2000.0) * c["reactors"]}


# ---------------------------------------------------------------------------
# the paths in plain torch
# ---------------------------------------------------------------------------
def _operators(n, alfa, bh):
    """Derivative and filter of a line with periodic halo f(-5:n+5), as dense
    matrices on the n + 11 values (derivative.F90:63-306, filter.F90:31-285)."""
    def solve(off, a_in, a_end, rows):
        m = n + 1 + 2 * off
        M = np.eye(m)
        for u in range(m):
            a = a_end if u in (0, m - 1) else a_in
            if u > 0:
                M[u, u - 1] = a
            if u < m - 1:
                M[u, u + 1] = a
        B = np.zeros((m, n + 11))
        for u in range(m):
            for s, v in rows(u - off):
                B[u, u - off + s + 5] += v
        return np.linalg.solve(M, B)[off:off + n + 1]

    def d_rows(r):
        co = (0.75, -0.15, 1.0 / 60.0) if r in (-1, n + 1) else (7.0 / 9.0, 1.0 / 36.0)
        return [(s * (k + 1), s * v) for k, v in enumerate(co) for s in (1, -1)]

    c10 = ((193.0 + 126.0 * alfa) / 512.0, (105.0 + 302.0 * alfa) / 512.0, (-15.0 + 30.0 * alfa) / 128.0,
           (45.0 - 90.0 * alfa) / 1024.0, (-5.0 + 10.0 * alfa) / 512.0, (1.0 - 2.0 * alfa) / 1024.0)
    e, t = 1.0 - bh, 1.0 - 2.0 * alfa
    ch = np.array([
        [-e / 1024, 5 * e / 512, (979 + 45 * bh) / 1024, (15 + 113 * bh) / 128, -105 * e / 512, 63 * e / 256,
         -105 * e / 512, 15 * e / 128, -45 * e / 1024, 5 * e / 512, -e / 1024],
        [t / 1024, -5 * t / 512, (45 + 934 * alfa) / 1024, (113 + 30 * alfa) / 128, (105 + 302 * alfa) / 512,
         -63 * t / 256, 105 * t / 512, -15 * t / 128, 45 * t / 1024, -5 * t / 512, t / 1024],
        [-t / 1024, 5 * t / 512, (-45 + 90 * alfa) / 1024, (15 + 98 * alfa) / 128, (407 + 210 * alfa) / 512,
         (63 + 130 * alfa) / 256, -105 * t / 512, 15 * t / 128, -45 * t / 1024, 5 * t / 512, -t / 1024]])

    def f_rows(r):
        if r < 0:
            return [(j - 5 - r, ch[r + 3, j]) for j in range(11)]
        if r > n:
            return [(n + 5 - j - r, ch[n + 3 - r, j]) for j in range(11)]
        return [(s * k, v) for k, v in enumerate(c10) for s in (1, -1)]

    return solve(1, 1.0 / 3.0, 0.0, d_rows), solve(3, alfa, bh, f_rows)


def _fold(H, n):
    """The halo columns of H as columns of the line's own points."""
    out = np.zeros((n + 1, n + 1))
    for h in range(1, 6):
        out[:, n - h] += H[:, 5 - h]
        out[:, h] += H[:, n + 5 + h]
    return out


def _along(M, f, d):
    """M applied to f (..., k, j, i) along direction d (0: i, 1: j, 2: k)."""
    if d == 0:
        return f @ M.T
    if d == 1:
        return (f.transpose(-1, -2) @ M.T).transpose(-1, -2).contiguous()
    return (M @ f.reshape(f.shape[0], -1)).reshape(f.shape)


class _Exact:
    def __init__(self, cfg, main=False, recon=None):
        self.cfg, self.main, self.recon = cfg, main, recon
        self.n = (cfg.im, cfg.jm, cfg.km)
        self.nd = 3 if cfg.km > 0 else 2
        self.Di, self.Dh, self.F = [], [], []
        for d in range(self.nd):
            n = self.n[d]
            D, F = _operators(n, cfg.alfa_filter, cfg.beta_halo)
            t = lambda a: torch.tensor(a, device=DEV, dtype=F8)  # noqa: E731
            self.Di.append(t(D[:, 5:n + 6]))
            self.Dh.append(t(_fold(D, n)))
            self.F.append(t(F[:, 5:n + 6] + _fold(F, n)))
        self.inv = [self.n[d] / (cfg.lx, cfg.ly, cfg.lz)[d] for d in range(self.nd)]
        self.c2 = cfg.gamma * cfg.mach ** 2
        self.c6 = 1.0 / (cfg.gamma - 1.0)

    def prims(self, q):
        u, v, w = q[1] / q[0], q[2] / q[0], q[3] / q[0]
        p = (q[4] - 0.5 * q[0] * (u * u + v * v + w * w)) / self.c6
        return [q[0], u, v, w, p, p / q[0] * self.c2]

    def ddx(self, f, fh, d):
        """d/dx_d of lines whose points hold f and whose halo copies hold fh."""
        return (_along(self.Di[d], f, d) + _along(self.Dh[d], fh, d)) * self.inv[d]

    def filt(self, q):
        for d in range(self.nd):
            q = torch.stack([_along(self.F[d], q[m], d) for m in range(5)])
        return q

    def rhs(self, q, pr, stats, qh=None):
        """qrhs of q with the primitives pr at the points and, in the halo of
        direction d, qh[d] and its primitives (without qh: as at the points),
        and the step's statistics."""
        cfg = self.cfg
        qh = qh or [q] * self.nd
        ph = [self.prims(x) for x in qh] if self.main else [pr] * self.nd
        zero = torch.zeros_like(q[0])
        g = [[self.ddx(pr[1 + m], ph[d][1 + m], d) if d < self.nd else zero for d in range(3)] for m in range(3)]
        gt = [self.ddx(pr[5], ph[d][5], d) if d < self.nd else zero for d in range(3)]
        s = cfg.sutherland / cfg.ref_tem
        mu = pr[5] * torch.sqrt(pr[5]) * (1.0 + s) / (pr[5] + s) / cfg.reynolds
        st = None
        if stats:
            st = self.stats(pr, g, mu)
        div = (g[0][0] + g[1][1] + g[2][2]) / 3.0
        sg = [[mu * (g[a][b] + g[b][a]) - (2.0 * mu * div if a == b else 0.0) for b in range(3)] for a in range(3)]
        hcc = mu / cfg.prandtl / ((cfg.gamma - 1.0) * cfg.mach ** 2)
        qf = [hcc * gt[a] + sg[a][0] * pr[1] + sg[a][1] * pr[2] + sg[a][2] * pr[3] for a in range(3)]
        del g, gt
        out = [zero.clone() for _ in range(5)]
        for d in range(self.nd):
            if self.recon is None:
                for m in range(5):
                    out[m] -= self.ddx(self.flux(q, pr, m, d), self.flux(qh[d], ph[d], m, d), d)
            else:
                self.upwind(((q, pr), (qh[d], ph[d])), d, out)
            for a in range(3):
                out[1 + a] += self.ddx(sg[d][a], sg[d][a], d)
            out[4] += self.ddx(qf[d], qf[d], d)
        return torch.stack(out), st

    @staticmethod
    def flux(q, x, m, d):
        if m == 4:
            return (q[4] + x[4]) * x[1 + d]
        return q[m] * x[1 + d] + (x[4] if m == d + 1 else 0.0)

    def stats(self, pr, g, mu):
        inner = (slice(1, None) if self.nd == 3 else slice(None), slice(1, None), slice(1, None))
        n = self.n[0] * self.n[1] * max(self.n[2], 1)
        ke = (pr[0] * (pr[1] ** 2 + pr[2] ** 2 + pr[3] ** 2))[inner].sum() / (2.0 * n)
        w = ((g[2][1] - g[1][2]) ** 2 + (g[0][2] - g[2][0]) ** 2 + (g[1][0] - g[0][1]) ** 2)
        en = (pr[0] * w)[inner].sum() / (2.0 * n)
        ss = sum((0.5 * (g[a][b] + g[b][a])) ** 2 for a in range(3) for b in range(3))
        di = (2.0 * mu * (ss - (g[0][0] + g[1][1] + g[2][2]) ** 2 / 3.0))[inner].sum() / n
        return float(ke), float(en), float(di)

    def upwind(self, points_halo, d, out):
        """Steger-Warming split, MP7 or WENO7 interface values, difference."""
        n, ax = self.n[d], 2 - d
        sides = [self.split(q, x, d) for q, x in points_halo]
        # the schemes' thresholds are for fluxes that carry the metrics
        scale = self.inv[d] * math.prod(1.0 / v for v in self.inv)
        for m in range(5):
            rows = []
            for s in (0, 1):
                f, h = sides[0][s][m], sides[1][s][m]
                rows.append(scale * torch.cat([h.narrow(ax, n - 4, 4), f, h.narrow(ax, 1, 4)], dim=ax))
            # interfaces -1..n; row r of the line at r + 4
            wp = [rows[0].narrow(ax, k, n + 2) for k in range(7)]
            wm = [rows[1].narrow(ax, 7 - k, n + 2) for k in range(7)]
            rec = _mp7 if self.recon == 3 else _weno7
            fh = rec(wp) + rec(wm)
            out[m] -= (fh.narrow(ax, 1, n + 1) - fh.narrow(ax, 0, n + 1)) * (self.inv[d] / scale)

    def split(self, q, x, d):
        gam = self.cfg.gamma
        rho, vel = x[0], x[1:4]
        c = torch.sqrt(x[5]) / self.cfg.mach
        u = vel[d]
        full = [self.flux(q, x, m, d) for m in range(5)]
        lam = (u, u + c, u - c)
        pos = [0.5 * (v + torch.sqrt(v * v + (0.04 / self.inv[d]) ** 2)) for v in lam]
        k2 = 0.5 * (gam - 1.0) * (vel[0] ** 2 + vel[1] ** 2 + vel[2] ** 2)
        res = []
        for s in (0, 1):
            e0, e3, e4 = pos if s == 0 else [lam[i] - pos[i] for i in range(3)]
            v2, v3 = e3 - e4, 2.0 * e0 - e3 - e4
            v4 = e0 - v3 * 0.5 / gam
            f = [rho * v4] + [rho * (v4 * vel[a] + (v2 * c * 0.5 / gam if a == d else 0.0)) for a in range(3)]
            f.append(e0 * q[4] + rho * (v2 * u * c * 0.5 / gam - v3 * (k2 + c * c) * 0.5 / gam / (gam - 1.0)))
            up = u >= c if s == 0 else u <= -c
            dn = u <= -c if s == 0 else u >= c
            res.append([torch.where(up, full[m], torch.where(dn, torch.zeros_like(c), f[m])) for m in range(5)])
        return res

    def qswap(self, q, pr):
        """Per direction the halo copy, then the mean of the duplicate planes,
        which take the primitives of the result."""
        qh = []
        for d in range(self.nd):
            qh.append(q)
            ax, q = 3 - d, q.clone()
            mean = 0.5 * (q.select(ax, 0) + q.select(ax, -1))
            for i in (0, -1):
                q.select(ax, i).copy_(mean)
        pr = [x.clone() for x in pr]
        for x, new in zip(pr, self.prims(q)):
            for d in range(self.nd):
                for i in (0, -1):
                    x.select(2 - d, i).copy_(new.select(2 - d, i))
        return q, pr, qh

    def steps(self, q, steps):
        cfg, rk = self.cfg, ((1.0, 0.0, 1.0), (0.75, 0.25, 0.25), (1.0 / 3.0, 2.0 / 3.0, 2.0 / 3.0))
        hist, pr = [], self.prims(q)
        for _ in range(steps):
            for s, (a, b, c) in enumerate(rk):
                qh = None
                if self.main:
                    q, pr, qh = self.qswap(self.filt(q), pr)
                else:
                    pr = self.prims(q)
                r, st = self.rhs(q, pr, s == 0, qh)
                if s == 0:
                    q0 = q
                    hist.append(st)
                q = a * q0 + b * q + c * r * cfg.deltat
                if self.main:
                    pr = self.prims(q)
                else:
                    q = self.filt(q)
        ke, en, di = (np.array(h) for h in zip(*hist))
        return {"q": q, "ke": ke, "en": en, "di": di}


def _minmod(*v):
    lo, hi = v[0], v[0]
    for x in v[1:]:
        lo, hi = torch.minimum(lo, x), torch.maximum(hi, x)
    return lo.clamp(min=0.0) + hi.clamp(max=0.0)


def _mp7(u):
    ul = (-3.0 * u[0] + 25.0 * u[1] - 101.0 * u[2] + 319.0 * u[3] + 214.0 * u[4] - 38.0 * u[5] + 4.0 * u[6]) / 420.0
    ump = u[3] + _minmod(u[4] - u[3], 4.0 * (u[3] - u[2]))
    dm, d0, d1 = (u[k] - 2.0 * u[k + 1] + u[k + 2] for k in (1, 2, 3))
    hm = _minmod(4.0 * dm - d0, 4.0 * d0 - dm, dm, d0)
    h0 = _minmod(4.0 * d0 - d1, 4.0 * d1 - d0, d0, d1)
    uul = u[3] + 4.0 * (u[3] - u[2])
    umd = 0.5 * (u[3] + u[4]) - 0.5 * h0
    ulc = u[3] + 0.5 * (u[3] - u[2]) + hm * (4.0 / 3.0)
    mn, mx = torch.minimum, torch.maximum
    lo = mx(mn(mn(u[3], u[4]), umd), mn(mn(u[3], uul), ulc))
    hi = mn(mx(mx(u[3], u[4]), umd), mx(mx(u[3], uul), ulc))
    return torch.where((ul - u[3]) * (ul - ump) >= 1.0e-10, ul + _minmod(lo - ul, hi - ul), ul)


def _weno7(u):
    cand = [(-3, 13, -23, 25), (1, -5, 13, 3), (-1, 7, 7, -1), (3, 13, -5, 1)]
    first = [(-2, 9, -18, 11), (1, -6, 3, 2), (-2, -3, 6, -1), (-11, 18, -9, 2)]
    second = [(-1, 4, -5, 2), (0, 1, -2, 1), (1, -2, 1, 0), (2, -5, 4, -1)]
    third = (-1, 3, -3, 1)
    lin = (1.0 / 35.0, 12.0 / 35.0, 18.0 / 35.0, 4.0 / 35.0)
    num = den = 0.0
    for k in range(4):
        dot = lambda co: sum(a * u[k + j] for j, a in enumerate(co) if a)  # noqa: E731
        b = dot(first[k]) ** 2 / 36.0 + dot(second[k]) ** 2 * (13.0 / 12.0) + dot(third) ** 2 * (781.0 / 720.0)
        w = lin[k] / (b + 1.0e-6) ** 2
        num, den = num + w * dot(cand[k]) / 12.0, den + w
    return num / den


class _Kinetics:
    """Ideal-gas thermodynamics and mass-action rates of a CTML mechanism."""

    R, R_ENTHALPY = 8314.46261815324, 8314.2
    ATOMS = {"H": 1.008, "O": 15.999, "N": 14.007}

    def __init__(self, path):
        root = ET.parse(path).getroot()
        pairs = lambda t: [(a, float(b)) for a, b in (x.split(":") for x in (t or "").split())]  # noqa: E731
        names = next(p for p in root.iter("phase") if p.get("id") == "gas").find("speciesArray").text.split()
        self.ix = {s: k for k, s in enumerate(names)}
        self.W, self.nasa = np.zeros(len(names)), [None] * len(names)
        for sp in root.iter("species"):
            if sp.get("name") in self.ix:
                k = self.ix[sp.get("name")]
                self.W[k] = sum(n * self.ATOMS[e] for e, n in pairs(sp.find("atomArray").text))
                lo, hi = sorted(sp.iter("NASA"), key=lambda b: float(b.get("Tmin")))
                co = [[float(v) for v in b.find("floatArray").text.replace(",", " ").split()] for b in (lo, hi)]
                self.nasa[k] = (float(lo.get("Tmax")), co[0], co[1], float(lo.get("P0") or 101325.0))
        self.reactions = []
        for r in root.iter("reaction"):
            arr, ef = r.find("rateCoeff/Arrhenius"), r.find("rateCoeff/efficiencies")
            unit = {"cal/mol": 4184.0, "kcal/mol": 4.184e6, "J/mol": 1000.0, "kJ/mol": 1e6, "K": self.R}
            eff = None
            if r.get("type") == "threeBody":
                eff = np.full(len(names), float(ef.get("default", "1.0")) if ef is not None else 1.0)
                for s, v in pairs(ef.text if ef is not None else ""):
                    if s in self.ix:
                        eff[self.ix[s]] = v
            self.reactions.append((
                float(arr.find("A").text), float(arr.find("b").text),
                float(arr.find("E").text) * unit[arr.find("E").get("units", "cal/mol")] / self.R,
                r.get("reversible", "yes") != "no", eff,
                [(self.ix[s], v) for s, v in pairs(r.find("reactants").text)],
                [(self.ix[s], v) for s, v in pairs(r.find("products").text)]))

    def rates(self, T, p, Y):
        ns = len(self.W)
        rho = p / (self.R * T * sum(Y[k] / self.W[k] for k in range(ns)))
        c = [rho * Y[k] / self.W[k] for k in range(ns)]
        cp, h, g = 0.0, 0.0, []
        for k in range(ns):
            tm, lo, hi, p0 = self.nasa[k]
            a = [torch.where(T <= tm, *(torch.tensor(v[j], device=DEV, dtype=F8) for v in (lo, hi))) for j in range(7)]
            hrt = a[0] + T * (a[1] / 2 + T * (a[2] / 3 + T * (a[3] / 4 + T * a[4] / 5))) + a[5] / T
            sr = a[0] * torch.log(T) + T * (a[1] + T * (a[2] / 2 + T * (a[3] / 3 + T * a[4] / 4))) + a[6]
            cp = cp + Y[k] / self.W[k] * (a[0] + T * (a[1] + T * (a[2] + T * (a[3] + T * a[4]))))
            h = h + Y[k] * hrt * (self.R_ENTHALPY / self.W[k]) * T
            g.append(hrt - sr)
        w = [torch.zeros_like(T) for _ in range(ns)]
        lc0 = torch.log(self.nasa[0][3] / (self.R * T))
        for A_, b, ta, rev, eff, reac, prod in self.reactions:
            lk = math.log(A_) + b * torch.log(T) - ta / T
            fwd = torch.exp(lk)
            for k, v in reac:
                fwd = fwd * c[k] ** v
            if rev:
                dg = sum(v * g[k] for k, v in prod) - sum(v * g[k] for k, v in reac)
                dn = sum(v for _, v in prod) - sum(v for _, v in reac)
                bwd = torch.exp(lk + dg - dn * lc0)
                for k, v in prod:
                    bwd = bwd * c[k] ** v
                fwd = fwd - bwd
            if eff is not None:
                fwd = fwd * sum(float(eff[k]) * c[k] for k in range(ns))
            for k, v in reac:
                w[k] = w[k] - v * fwd
            for k, v in prod:
                w[k] = w[k] + v * fwd
        return {"wdot": torch.stack([w[k] * self.W[k] for k in range(ns)]), "h": h, "cp": cp * self.R}


def exact(case, seed):
    c = case
    if c["family"] == "flow":
        if c["chardec"] or c["conschm"] == "543c":
            return None  # the projected and the compact interface fluxes have no short restatement
        cfg = _config(c)
        E = _Exact(cfg, c["path"] == "main", c["recon"] if c["conschm"] == "753e" else None)
        o = E.steps(_initial(c["path"], cfg, seed), c["steps"])
        keep = {"vortex": ("q",), "tgv": ("q", "ke", "en"), "main": ("q", "ke", "en", "di")}[c["path"]]
        return {k: o[k] for k in keep}
    if c["family"] == "batch":
        res = [_Exact(cfg).steps(_initial(path, cfg, seed * 64 + k), c["steps"]) for path, cfg, k in _batch_specs(c)]
        return {"q": [r["q"] for r in res], "ke": np.array([r["ke"] for r in res]), "en": np.array([r["en"] for r in res])}
    if c["family"] == "chem":
        K = _Kinetics(MECHANISM)
        return K.rates(*_cells(K.W, K.ix, c["cells"], seed))
    return None  # an integration to a tolerance, not to rounding

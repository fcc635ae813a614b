"""The work that programs built on this package have it do, as timed cases.

A case is one piece of a run: a scenario resident on the GPU (or a batch of
them) advanced by a number of time steps through `Model.step` /
`Batch.step`, and its fields brought to the host, as a program does between
two outputs.  The listed cases span the package's forms and sizes: one-row
flumes and small channels, where the launches of a step count, the shipped
examples' sizes, the 1024 x 1024 x 10 run, the mixed form at 2048 x 2048 x
8, and batches of small and of mid-size scenarios.

`exact` holds its own statement of the time step for wet, walled, inviscid
scenarios in plain 64-bit torch (the equations of NHWAVE's fluxes,
eval_duvw, poisson_solver and get_Omega), with a direct solve of the
pressure system.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from nhwave_amd import capi
from nhwave_amd import scenario as S
from nhwave_amd.batch import Batch
from nhwave_amd.model import Model

# fields of a run that a program keeps: the surface, the velocities, the
# dynamic pressure of a non-hydrostatic run and the wet-dry mask
FIELDS = ("Eta", "U", "V", "W", "Mask")


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # the shipped submerged-bar flume's size and options: one row, a linear
        # wave train from the west over a bar, an east sponge
        _c("flume_300x1x3", "flume", 300, 1, 3, 20, wave="LEF_LIN", tol=1e-12),
        # the shipped cnoidal breaker flume's size: one row, 20 levels (the line
        # solver's range), the k-epsilon closure
        _c("breaker_ke_880x1x20", "flume", 880, 1, 20, 4, wave="LEF_CON", turb=10, line=True, tol=1e-12),
        # solitary wave in a flat channel, the package's parity configuration
        _c("channel_512x8x3", "channel", 512, 8, 3, 20, tol=1e-12),
        # run-up on a plane beach, hydrostatic, wet-dry, ragged sides
        _c("runup_hydro_257x33x5", "runup", 257, 33, 5, 40, nh=False),
        # hydrostatic basin, third-order time stepping, odd sides
        _c("basin_rk3_333x217x7", "basin", 333, 217, 7, 20, nh=False, order=3),
        # the shipped Monai Valley run's size: internal irregular wavemaker,
        # k-epsilon, non-hydrostatic, run-up
        _c("irregular_ke_492x243x4", "irregular", 492, 243, 4, 8, turb=10),
        # the shipped steady-flow run's size: discharge boundary, friction side
        # walls, log-law bottom, k-epsilon
        _c("steady_ke_656x100x15", "steady", 656, 100, 15, 6, turb=10, tol=1e-12),
        # constant viscosities over bumps with a drying beach
        _c("viscous_301x420x9", "bumps", 301, 420, 9, 12, turb=1),
        # the benchmark's 1024 x 1024 x 10 run
        _c("bumps_1024x1024x10", "bumps", 1024, 1024, 10, 24),
        # the mixed form at its configured size
        _c("mixed_2048x2048x8", "bumps", 2048, 2048, 8, 20, mixed=True, tol=1e-8),
        # a mixed-precision ensemble in one batch
        _c("ensemble12_mixed", "batch", 128, 384, 10, 6, members=12, mixed=True, tol=1e-8),
        # many small double-precision scenarios in one batch
        _c("ensemble24_small", "batch", 32, 96, 6, 6, members=24, tol=1e-12),
    ]


def _c(name, kind, m, n, k, steps, nh=True, order=2, wave="NONE", turb=0, line=False, mixed=False, members=1,
       tol=1e-10) -> dict:
    """m x n x k cells; for a batch, grids of m .. n cells a side and 3 .. k
    levels, in even ratios.  turb: 0 inviscid, 1 constant viscosities, 10 k-epsilon."""
    return {"name": name, "kind": kind, "m": m, "n": n, "k": k, "steps": steps, "nh": nh, "order": order,
            "wave": wave, "turb": turb, "line": line, "mixed": mixed, "members": members, "tol": tol}


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["flume", "breaker", "channel", "runup", "basin", "irregular", "steady", "bumps", "bumps",
                       "mixed", "batch", "batch"])
    t = 1e-12
    if kind == "flume":
        wave = rng.choice(["LEF_LIN", "LEF_STK", "LEF_SOL", "LEF_CON"])
        c = _c("", "flume", _log(rng, 120, 2000), rng.choice([1, 1, 3]), rng.randint(2, 12), 20, wave=wave,
               turb=rng.choice([0, 0, 1, 10]), tol=t)
        if c["k"] < 3 and c["turb"] == 10:
            c["turb"] = 1
    elif kind == "breaker":
        c = _c("", "flume", _log(rng, 300, 1200), 1, rng.randint(17, 24), 4, wave="LEF_CON", turb=10, line=True, tol=t)
    elif kind == "channel":
        c = _c("", "channel", _log(rng, 100, 900), rng.randint(4, 12), rng.randint(2, 5), 20, tol=t)
    elif kind == "runup":
        c = _c("", "runup", _log(rng, 64, 512), rng.randint(4, 64), rng.randint(2, 8), 40,
               nh=rng.random() < 0.3, tol=t)
    elif kind == "basin":
        c = _c("", "basin", _log(rng, 64, 600), _log(rng, 64, 400), rng.randint(3, 10), 20, nh=False,
               order=rng.choice([1, 2, 3]))
    elif kind == "irregular":
        c = _c("", "irregular", _log(rng, 200, 640), _log(rng, 64, 300), rng.randint(3, 6), 8, turb=10, tol=t)
    elif kind == "steady":
        c = _c("", "steady", _log(rng, 400, 900), _log(rng, 16, 128), rng.randint(4, 15), 6,
               turb=rng.choice([0, 10]), tol=t)
    elif kind == "bumps":
        c = _c("", "bumps", _log(rng, 96, 1024), _log(rng, 96, 1024), rng.randint(3, 16), 12,
               nh=rng.random() < 0.85, turb=rng.choice([0, 0, 0, 1]), tol=1e-11)
        if c["k"] > 10 and c["m"] * c["n"] > 600 * 600:
            c["k"] = 10
    elif kind == "mixed":
        c = _c("", "bumps", _log(rng, 256, 1536), _log(rng, 256, 1536), rng.randint(3, 10), 8, mixed=True, tol=1e-8)
    else:
        lo = rng.randint(24, 96)
        c = _c("", "batch", lo, lo * rng.randint(2, 3), rng.randint(4, 10), 6, members=rng.randint(5, 16),
               mixed=rng.random() < 0.5, tol=1e-8)
        if not c["mixed"]:
            c["tol"] = t
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# scenarios
# ---------------------------------------------------------------------------

def _viscous(s, turb, visc=1.0e-6, cvs=0.001, chs=0.001):
    if not turb:
        return s
    return s.with_(viscous=True, turb=turb, visc=visc, cvs=cvs, chs=chs)


def _scenario(case: dict, seed: int):
    rng = np.random.default_rng(seed)
    m, n, k, kind = case["m"], case["n"], case["k"], case["kind"]
    kw = dict(tol=case["tol"], non_hydro=case["nh"])
    if kind == "flume":
        dx, depth = 0.02, 0.4
        per = float(rng.uniform(1.6, 2.4))
        sponge = (0.0, 0.15 * m * dx, 0.0, 0.0) if case["wave"] != "LEF_SOL" else None
        s = S.wave_flume(mglob=m, nglob=n, kglob=k, dx=dx, depth=depth, wavemaker=case["wave"],
                         amp=float(rng.uniform(0.01, 0.025)) if case["wave"] != "LEF_CON" else
                         float(rng.uniform(0.06, 0.1)),
                         per=per, bottom="beach" if case["turb"] == 10 else "bar", sponge=sponge, **kw)
    elif kind == "channel":
        s = S.solitary_channel(mglob=m, nglob=n, kglob=k, amp_ratio=float(rng.uniform(0.12, 0.24)),
                               x0=float(rng.uniform(0.2, 0.5)) * m * 0.05, **kw)
    elif kind == "runup":
        s = S.beach_runup(mglob=m, nglob=n, kglob=k, dx=0.1, amp=float(rng.uniform(0.03, 0.06)),
                          x0=float(rng.uniform(0.1, 0.2)) * m * 0.1, **kw)
    elif kind == "basin":
        s = _wet_basin(m, n, k, rng, **kw)
    elif kind == "irregular":
        dx = 0.011
        s = S.internal_wave_basin(mglob=m, nglob=n, kglob=k, dx=dx, dy=0.014, depth=0.135, nfreq=32,
                                  dirs=(-10.0, 0.0, 10.0), hs=0.01, box=(0.3, 0.5, 0.0, n * 0.014),
                                  seed=int(rng.integers(1 << 30)), **kw)
    elif kind == "steady":
        s = S.steady_flume(mglob=m, nglob=n, kglob=k, dx=0.015, depth=0.3, obstacle=float(rng.uniform(0.07, 0.12)),
                           width=0.2, tramp=float(rng.uniform(2.0, 5.0)), zob=1.5e-5,
                           bc_y=5 if case["turb"] else 1, **kw)
    else:
        s = S.bumps_beach(n=n, m=m, kglob=k, dx=10.0, seed=int(rng.integers(1 << 30)), nbumps=16,
                          beach_width=min(1200.0, 2.5 * m), amp=float(rng.uniform(1.0, 3.0)),
                          center=(0.4 * m * 10.0, 0.5 * n * 10.0), radius=min(500.0, 2.0 * min(m, n)), **kw)
    if n > 1 and kind in ("flume", "channel", "steady"):
        # uneven across the tank, as a real bottom is, so that the transverse
        # velocity is a result and not the round-off of a symmetric run
        y = 1.0 + 0.05 * np.cos(np.pi * (np.arange(n) + 0.5) / n)
        s = s.with_(hcg=s.hcg * y[:, None])
    s = s.with_(time_order=case["order"])
    if kind == "bumps":
        return _viscous(s, case["turb"], 1.0e-6, 0.01, 1.0)
    return _viscous(s, case["turb"])


def _wet_basin(m, n, k, rng, dx=5.0, dy=6.0, **kw):
    """A closed basin that stays wet: four bumps on a 20 m bottom, a surface
    hump at rest."""
    x, y = np.meshgrid((np.arange(m) + 0.5) * dx, (np.arange(n) + 0.5) * dy)
    lx, ly = m * dx, n * dy
    h = np.full((n, m), 20.0)
    for _ in range(4):
        cx, cy, r = rng.uniform(0, lx), rng.uniform(0, ly), rng.uniform(0.1, 0.3) * max(lx, ly)
        h += rng.uniform(-6.0, 6.0) * np.exp(-((x - cx) ** 2 + (y - cy) ** 2) / r ** 2)
    h = np.clip(h, 5.0, 40.0)
    cx, cy, r = rng.uniform(0.3, 0.7) * lx, rng.uniform(0.3, 0.7) * ly, 0.15 * min(lx, ly)
    eta = rng.uniform(0.5, 1.5) * np.exp(-((x - cx) ** 2 + (y - cy) ** 2) / r ** 2)
    return S.Scenario(name=f"basin_{m}x{n}x{k}", mglob=m, nglob=n, kglob=k, dx=dx, dy=dy, hcg=h, etag=eta,
                      dt_ini=0.05, dt_max=60.0, **kw)


def _members(case: dict, seed: int) -> list:
    rng = np.random.default_rng(seed)
    out = []
    for q in range(case["members"]):
        side = int(round(case["m"] * (case["n"] / case["m"]) ** (q / (case["members"] - 1))))
        out.append(S.bumps_beach(n=side, kglob=3 + q % (case["k"] - 2), dx=10.0, seed=int(rng.integers(1 << 30)),
                                 nbumps=8, beach_width=min(1200.0, 2.5 * side), amp=float(rng.uniform(0.5, 3.0)),
                                 radius=min(500.0, 2.0 * side), tol=case["tol"]))
    return out


# ---------------------------------------------------------------------------
# the timed path
# ---------------------------------------------------------------------------

def prepare(case: dict, seed: int):
    """The run resident on the GPU: its bathymetry and initial state uploaded,
    `initial` done.  The first steps of the run are in the timed part."""
    precision = capi.NHW_MIXED if case["mixed"] else capi.NHW_FP64
    if case["kind"] == "batch":
        return case, Batch(_members(case, seed), precision=precision, autotune=False)
    solver = capi.NHW_SOLVER_LINE if case["line"] else capi.NHW_SOLVER_MG
    return case, Model(_scenario(case, seed), precision=precision, solver=solver)


def _results(case: dict, m: Model) -> dict:
    got = m.download(*FIELDS, *(("P",) if case["nh"] and not case["mixed"] else ()))
    # the cells of the grid: the ghost cells around them are boundary scratch
    # (those above the surface hold clipped extrapolations), no results
    got = {f: _cells(v) for f, v in got.items()}
    if case["mixed"]:
        # the mixed form's results have single precision and are kept in it
        got = {f: v if v.dtype == np.int32 else v.astype(np.float32) for f, v in got.items()}
    return got


def _cells(v):
    g = S.NGHOST
    return v[(slice(g, -g),) * v.ndim]


def run(state):
    case, m = state
    m.step(case["steps"])
    if case["kind"] == "batch":
        # up to 64 arrays: the surface and mask of every member, the velocities
        # of the first few
        out = []
        for q, b in enumerate(m.members):
            r = _results(case, b)
            out.append({f: r[f] for f in (FIELDS if q < 4 else ("Eta", "Mask"))})
        return out
    return _results(case, m)


def work(case: dict) -> dict:
    """Bytes and operations of one pass that no form of the time step avoids:
    per RK stage and cell the momenta, velocities, Omega and P read and
    written once and the stage copies of the momenta read once, per column
    the depth, surface, bottom slopes and masks; the fields of the result
    once.  Operations: about 500 a cell and stage (slopes, HLL, update), and
    300 more for a pressure solve (15-point rows of a few iterations)."""
    if case["kind"] == "batch":
        # the members' sides are spaced evenly in their logarithm: the mean of side^2
        lo, hi = case["m"], case["n"]
        side2 = (hi * hi - lo * lo) / (2.0 * math.log(hi / lo)) if hi > lo else lo * lo
        cols, k = case["members"] * side2, 0.5 * (3 + case["k"])
    else:
        cols, k = float(case["m"] * case["n"]), case["k"]
    cells, s3 = cols * k, 4.0 if case["mixed"] else 8.0
    stage = cells * (s3 * (7 * 2 + 3) + (16.0 if case["nh"] else 0.0)) + cols * 8.0 * 24
    passes = case["steps"] * case["order"]
    return {"bytes": passes * stage + cells * 8.0 * 4, "flops": passes * cells * (800.0 if case["nh"] else 500.0)}


# ---------------------------------------------------------------------------
# the same steps in plain 64-bit torch
# ---------------------------------------------------------------------------

def exact(case: dict, seed: int):
    """Wet, walled, inviscid runs.  None for the others: wet-dry fronts,
    wavemakers and closures have no short independent statement, and a
    direct solve of a pressure system with wide rows takes minutes."""
    if case["kind"] not in ("channel", "basin") or case["mixed"] or (case["nh"] and case["n"] * case["k"] > 64):
        return None
    w = _Wet(_scenario(case, seed))
    for _ in range(case["steps"]):
        w.step()
    out = {"Eta": w.Eta, "U": w.U, "V": w.V, "W": w.W, "Mask": torch.ones_like(w.Eta, dtype=torch.int32)}
    if case["nh"]:
        out["P"] = w.P
    return {f: _cells(v.cpu()) for f, v in out.items()}


class _Wet:
    """NHWAVE's time step where every cell is wet: arrays [k, j, i] with two
    ghost cells a side."""

    def __init__(self, s):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)  # noqa: E731
        self.s, self.dev = s, dev
        f = S.bathymetry_fields(s)
        i0 = S.initial_fields(s)
        dsig, sig, sigc = S.vertical_grid(s.kglob, s.ivgrd, s.grd_r)
        self.dsig, self.sig, self.sigc = t(dsig), t(sig), t(sigc)
        self.dsig_h, self.sig_h = dsig, sig
        self.Hc, self.DelxH, self.DelyH = t(f["Hc"]), t(f["DelxH"]), t(f["DelyH"])
        self.Hfx, self.Hfy = t(f["Hfx"]), t(f["Hfy"])
        self.g = float(np.float32(9.81))
        self.dt, self.M, self.N, self.K = s.dt_ini, s.mglob, s.nglob, s.kglob
        self.Eta = t(i0["Eta"])
        self._mirror(self.Eta)
        self.D = self.Hc + self.Eta
        self.U, self.V, self.W = t(i0["U"]), t(i0["V"]), t(i0["W"])
        self.DU, self.DV, self.DW = (torch.zeros_like(self.U) for _ in range(3))
        self.P = torch.zeros((s.kloc + 1, s.nloc, s.mloc), dtype=torch.float64, device=dev)
        self.Om = torch.zeros_like(self.P)
        self.DelxEta, self.DelyEta = torch.zeros_like(self.Eta), torch.zeros_like(self.Eta)
        self.Eta0 = self.Eta.clone()
        self.EtaxL, self.EtaxR = torch.zeros_like(self.Hfx), torch.zeros_like(self.Hfx)
        self.EtayL, self.EtayR = torch.zeros_like(self.Hfy), torch.zeros_like(self.Hfy)
        self._vel_bc()
        self.DU, self.DV, self.DW = self.D * self.U, self.D * self.V, self.D * self.W

    # -- ghosts and slopes --------------------------------------------------
    @staticmethod
    def _mirror(a):
        a[2:-2, 0], a[2:-2, 1] = a[2:-2, 3], a[2:-2, 2]
        a[2:-2, -1], a[2:-2, -2] = a[2:-2, -4], a[2:-2, -3]
        a[0], a[1], a[-1], a[-2] = a[3].clone(), a[2].clone(), a[-4].clone(), a[-3].clone()

    @staticmethod
    def _lim(a, b):
        s = a.abs() + b.abs()
        v = (a * b.abs() + a.abs() * b) / torch.where(s < 1e-16, torch.ones_like(s), s)
        return torch.where(s < float(np.float32(1e-16)), torch.zeros_like(v), v)

    def _slope(self, a, dim, h):
        d = torch.diff(a, dim=dim) / h
        n = d.shape[dim]
        mid = self._lim(d.narrow(dim, 1, n - 1), d.narrow(dim, 0, n - 1))
        return torch.cat([d.narrow(dim, 0, 1), mid, d.narrow(dim, n - 1, 1)], dim)

    def _delx(self, a):
        return self._slope(a, a.dim() - 1, self.s.dx)

    def _dely(self, a):
        return self._slope(a, a.dim() - 2, self.s.dy)

    def _delz(self, a):
        h = torch.diff(self.sigc)
        h[0], h[-1] = 0.5 * (self.dsig[0] + self.dsig[1]), 0.5 * (self.dsig[-2] + self.dsig[-1])
        d = torch.diff(a, dim=0)
        mid_h = torch.diff(self.sigc)[:, None, None]
        t = d / mid_h
        mid = self._lim(t[1:], t[:-1])
        return torch.cat([(d[0] / h[0])[None], mid, (d[-1] / h[-1])[None]], 0)

    def _zfaces(self, a):
        """left and right states at the sigma faces Kbeg .. Kend1, interior columns"""
        d, g, K = self._delz(a)[:, 2:-2, 2:-2], a[:, 2:-2, 2:-2], self.K
        ds = self.dsig[:, None, None]
        left = (g + 0.5 * ds * d)[1:K + 2]
        right = (g - 0.5 * ds * d)[2:K + 3]
        return left, right

    def _uvw_z(self):
        (uL, uR), (vL, vR), (wL, wR) = (self._zfaces(a) for a in (self.U, self.V, self.W))
        q = lambda a: a[2:-2, 2:-2]  # noqa: E731
        wL[-1] = (q(self.Eta) - q(self.Eta0)) / self.dt + q(self.DelxEta) * uL[-1] + q(self.DelyEta) * vL[-1]
        wR[0] = -q(self.DelxH) * uR[0] - q(self.DelyH) * vR[0]
        return uL, uR, vL, vR, wL, wR

    def _vel_bc(self):
        K = self.K
        k = slice(2, K + 2)
        for a, sx, sy in ((self.U, -1, 1), (self.V, 1, -1), (self.W, 1, 1), (self.DU, -1, 1), (self.DV, 1, -1),
                          (self.DW, 1, 1)):
            for e in (0, 1):
                a[k, 2:-2, 1 - e] = sx * a[k, 2:-2, 2 + e]
                a[k, 2:-2, -2 + e] = sx * a[k, 2:-2, -3 - e]
                a[k, 1 - e, 2:-2] = sy * a[k, 2 + e, 2:-2]
                a[k, -2 + e, 2:-2] = sy * a[k, -3 - e, 2:-2]
        uL, _, vL, _, wL, wR = self._uvw_z()
        pad = lambda a: torch.nn.functional.pad(a, (2, 2, 2, 2))  # noqa: E731
        q = lambda a: a[2:-2, 2:-2]  # noqa: E731
        ut, vt, wt = pad(uL[-1]), pad(vL[-1]), pad(wL[-1])
        dxu, dxv, dxw = (q(self._delx(a)) for a in (ut, vt, wt))
        dyu, dyv, dyw = (q(self._dely(a)) for a in (ut, vt, wt))
        ex, ey, D = q(self.DelxEta), q(self.DelyEta), q(self.D)
        A2 = 1.0 + ex * ex + ey * ey
        wl, wr = wL[-1], wR[0]
        I = (slice(2, -2), slice(2, -2))
        for e in (1, 2):
            gb, sb, gt, st = 2 - e, 1 + e, K + 1 + e, K + 2 - e
            self.DW[(gb, *I)] = 2.0 * D * wr - self.DW[(sb, *I)]
            self.DU[(gb, *I)], self.DV[(gb, *I)] = self.DU[(sb, *I)].clone(), self.DV[(sb, *I)].clone()
            h = self.sigc[gt] - self.sigc[st]
            dws = self.DW[(st, *I)]
            self.DW[(gt, *I)] = 2.0 * D * wl - dws
            for a, sl, tz, c, t3 in (
                    (self.DU, ex, uL[-1], ex, 2.0 * ex * dxu - (1.0 - ex * ex) * dxw + ey * (dyu + dxv + ex * dyw)),
                    (self.DV, ey, vL[-1], ey, 2.0 * ey * dyv - (1.0 - ey * ey) * dyw + ex * (dxv + dyu + ey * dxw))):
                t2 = sl * (D * wl - dws) / (h / 2.0)
                src = a[(st, *I)]
                v = src + h * (-t2 + D * D / A2 * t3)
                old = 2.0 * D * tz - src
                hi, lo = torch.minimum(3.0 * old, torch.maximum(-old, v)), torch.maximum(3.0 * old, torch.minimum(-old, v))
                a[(gt, *I)] = torch.where(old > 0, hi, torch.where(old < 0, lo, v))
            for a, b in ((self.U, self.DU), (self.V, self.DV), (self.W, self.DW)):
                a[(gb, *I)], a[(gt, *I)] = b[(gb, *I)] / D, b[(gt, *I)] / D

    def _get_uvw(self):
        I = (slice(2, self.K + 2), slice(2, -2), slice(2, -2))
        D = self.D[2:-2, 2:-2]
        for a, b in ((self.U, self.DU), (self.V, self.DV), (self.W, self.DW)):
            a[I] = b[I] / D
        self._vel_bc()

    # -- face states and fluxes ----------------------------------------------
    def _faces(self, a, axis):
        """states left and right of the faces Ibeg .. Iend1 (axis 0: x) or
        Jbeg .. Jend1 (1: y) of the interior rows"""
        d = self._delx(a) if axis == 0 else self._dely(a)
        h = self.s.dx if axis == 0 else self.s.dy
        lo, hi = a + 0.5 * h * d, a - 0.5 * h * d
        if axis == 0:
            L, R = lo[..., 2:-2, 1:-2], hi[..., 2:-2, 2:-1]
        else:
            L, R = lo[..., 1:-2, 2:-2], hi[..., 2:-1, 2:-2]
        return (L[2:-2], R[2:-2]) if a.dim() == 3 else (L, R)

    def _side(self, axis):
        """surface and depth states, wave speeds and the HLL closure of one axis"""
        eL, eR = self._faces(self.Eta, axis)
        h = self.Hfx[2:-2, 2:-2] if axis == 0 else self.Hfy[2:-2, 2:-2]
        if axis == 0:
            self.EtaxL[2:-2, 2:-2], self.EtaxR[2:-2, 2:-2] = eL, eR
        else:
            self.EtayL[2:-2, 2:-2], self.EtayR[2:-2, 2:-2] = eL, eR
        dL, dR = torch.clamp(eL + h, min=self.s.min_dep), torch.clamp(eR + h, min=self.s.min_dep)
        nL, nR = self._faces(self.U if axis == 0 else self.V, axis)
        pL, pR = torch.sqrt(self.g * dL.abs()), torch.sqrt(self.g * dR.abs())
        ps = 0.5 * (pL + pR) + 0.25 * (nL - nR)
        us = 0.5 * (nL + nR) + pL - pR
        sl, sr = torch.minimum(nL - pL, us - ps), torch.maximum(nR + pR, us + ps)

        def hll(fl, fr, ul, ur):
            f = (sr * fl - sl * fr + sl * sr * (ur - ul)) / (sr - sl)
            return torch.where(sl >= 0, fl, torch.where(sr <= 0, fr, f))
        return eL, eR, h, dL, dR, nL, nR, hll

    def _walls(self, f, axis, first=0.0, last=0.0):
        if axis == 0:
            f[..., 0], f[..., -1] = first, last
        else:
            f[..., 0, :], f[..., -1, :] = first, last
        return f

    def _fluxes(self):
        self.DelxEta, self.DelyEta = self._delx(self.Eta), self._dely(self.Eta)
        out = []
        for ax in (0, 1):
            eL, eR, h, dL, dR, nL, nR, hll = self._side(ax)
            mom = [self._faces(a, ax) for a in (self.DU, self.DV, self.DW)]
            vel = [self._faces(a, ax) for a in (self.U, self.V, self.W)]
            prL, prR = 0.5 * self.g * (eL * eL + 2.0 * eL * h), 0.5 * self.g * (eR * eR + 2.0 * eR * h)
            mL, mR = mom[ax]
            fl = [self._walls(hll(mL, mR, dL.expand_as(mL), dR.expand_as(mR)), ax)]
            for q in range(3):
                if q == ax:
                    f = hll(mL * nL + prL, mR * nR + prR, *mom[q])
                    a, b = (prR[..., 0], prL[..., -1]) if ax == 0 else (prR[..., 0, :], prL[..., -1, :])
                    f = self._walls(f, ax, a, b)
                else:
                    (vL, vR) = vel[q]
                    f = self._walls(hll(dL * nL * vL, dR * nR * vR, *mom[q]), ax)
                fl.append(f)
            out.append(fl)
        uL, uR, vL, vR, wL, wR = self._uvw_z()
        om = self.Om[2:self.K + 3, 2:-2, 2:-2]
        z = []
        for L, R in ((uL, uR), (vL, vR), (wL, wR)):
            f = 0.5 * (om * (L + R) - om.abs() * (R - L))
            f[0], f[-1] = 0.0, 0.0
            z.append(f)
        return out[0], out[1], z

    # -- the step ---------------------------------------------------------------
    def step(self):
        s, K = self.s, self.K
        q = lambda a: a[..., 2:-2, 2:-2]  # noqa: E731
        I = (slice(2, K + 2), slice(2, -2), slice(2, -2))
        c = torch.sqrt(self.g * q(self.D))
        ds = self.dsig[2:K + 2, None, None]
        lim = min(float((s.dx / (self.U[I].abs() + c)).min()), float((s.dy / (self.V[I].abs() + c)).min()),
                  float((ds * q(self.D) / self.W[I].abs().clamp(min=float(np.float32(1e-16)))).min()), 1e7)
        self.dt = min(float(np.float32(1.05)) * self.dt, s.cfl * lim, s.dt_max)
        D0, M0 = self.D.clone(), [a.clone() for a in (self.DU, self.DV, self.DW)]
        self.Eta0 = self.Eta.clone()
        third, two3 = float(np.float32(1.0) / np.float32(3.0)), float(np.float32(2.0) / np.float32(3.0))
        for A, B in {1: [(0.0, 1.0)], 2: [(0.0, 1.0), (0.5, 0.5)],
                     3: [(0.0, 1.0), (0.75, 0.25), (third, two3)]}[s.time_order]:
            self._stage(A, B, D0, M0)

    def _stage(self, A, B, D0, M0):
        s, K, dt = self.s, self.K, self.dt
        q = lambda a: a[..., 2:-2, 2:-2]  # noqa: E731
        I = (slice(2, K + 2), slice(2, -2), slice(2, -2))
        dx, dy, ds = s.dx, s.dy, self.dsig[2:K + 2, None, None]
        hx, hy = q(self.Hfx), q(self.Hfy)
        ex, ey = q(self.EtaxL)[:, 1:] + q(self.EtaxR)[:, :-1], q(self.EtayL)[1:] + q(self.EtayR)[:-1]
        srcx = self.g * 0.5 * ex * (hx[:, 1:] - hx[:, :-1]) / dx
        srcy = self.g * 0.5 * ey * (hy[1:] - hy[:-1]) / dy
        X, Y, Z = self._fluxes()
        dX, dY = [torch.diff(f, dim=2) / dx for f in X], [torch.diff(f, dim=1) / dy for f in Y]
        dZ = [torch.diff(f, dim=0) / ds for f in Z]
        R1 = -((dX[0] + dY[0]) * ds).sum(0)
        q(self.D).copy_(A * q(D0) + B * (q(self.D) + dt * R1))
        self._mirror(self.D)
        self.Eta = self.D - self.Hc
        self.DelxEta, self.DelyEta = self._delx(self.Eta), self._dely(self.Eta)
        f = s.fcor
        du = -dX[1] - dY[1] - dZ[0] + f * self.DV[I] + srcx
        dv = -dX[2] - dY[2] - dZ[1] - f * self.DU[I] + srcy
        dw = -dX[3] - dY[3] - dZ[2]
        for a, r in ((self.DU, du), (self.DV, dv), (self.DW, dw)):
            a[I] += dt * r
        if s.non_hydro:
            self._get_uvw()
            self._pressure()
            P = self.P
            z, z1 = slice(2, K + 2), slice(3, K + 3)
            px = 0.5 * ((P[z, 2:-2, 3:-1] - P[z, 2:-2, 1:-3]) + (P[z1, 2:-2, 3:-1] - P[z1, 2:-2, 1:-3])) / (2. * dx)
            py = 0.5 * ((P[z, 3:-1, 2:-2] - P[z, 1:-3, 2:-2]) + (P[z1, 3:-1, 2:-2] - P[z1, 1:-3, 2:-2])) / (2. * dy)
            pz = (P[z1, 2:-2, 2:-2] - P[z, 2:-2, 2:-2]) / ds
            D, sc = q(self.D), self.sigc[2:K + 2, None, None]
            sx = ((1.0 - sc) * q(self.DelxH) - sc * q(self.DelxEta)) / D
            sy = ((1.0 - sc) * q(self.DelyH) - sc * q(self.DelyEta)) / D
            self.DU[I] -= D * dt / 1000.0 * (px + pz * sx)
            self.DV[I] -= D * dt / 1000.0 * (py + pz * sy)
            self.DW[I] -= dt / 1000.0 * pz
        for a, a0 in zip((self.DU, self.DV, self.DW), M0):
            a[I] = A * a0[I] + B * a[I]
        self._get_uvw()
        # Omega from the mass fluxes of the new state
        self.DelxEta, self.DelyEta = self._delx(self.Eta), self._dely(self.Eta)
        E = []
        for ax, mom in ((0, self.DU), (1, self.DV)):
            _, _, _, dL, dR, _, _, hll = self._side(ax)
            mL, mR = self._faces(mom, ax)
            E.append(self._walls(hll(mL, mR, dL.expand_as(mL), dR.expand_as(mR)), ax))
        div = R1 + torch.diff(E[0], dim=2) / dx + torch.diff(E[1], dim=1) / dy
        self.Om.zero_()
        self.Om[3:K + 3, 2:-2, 2:-2] = -torch.cumsum(ds * div, 0)

    # -- pressure -----------------------------------------------------------------
    def _pressure(self):
        """The 15-point sigma-coordinate pressure system, solved directly by
        block elimination along x (blocks of the N K unknowns of one column
        of cells)."""
        s, M, N, K, dx, dy = self.s, self.M, self.N, self.K, self.s.dx, self.s.dy
        n = lambda a: a.cpu().numpy()  # noqa: E731
        q = lambda a: n(a)[2:-2, 2:-2]  # noqa: E731
        ds, sig = self.dsig_h, self.sig_h[2:K + 2, None, None]
        D = q(self.D)
        sx = ((1. - sig) * q(self.DelxH) - sig * q(self.DelxEta)) / D
        sy = ((1. - sig) * q(self.DelyH) - sig * q(self.DelyEta)) / D
        A1 = sx * sx + sy * sy + (1. / D) ** 2
        up, dn = ds[2:K + 2, None, None], ds[1:K + 1, None, None]
        sm = up + dn
        U, V, W = n(self.U), n(self.V), n(self.W)
        f = up / sm
        uf = (1.0 - f) * U[2:K + 2] + f * U[1:K + 1]
        vf = (1.0 - f) * V[2:K + 2] + f * V[1:K + 1]
        dz = lambda a: (a[2:K + 2, 2:-2, 2:-2] - a[1:K + 1, 2:-2, 2:-2]) / (0.5 * sm)  # noqa: E731
        rhs = -((uf[:, 2:-2, 3:-1] - uf[:, 2:-2, 1:-3]) / (2. * dx) + dz(U) * sx +
                (vf[:, 3:-1, 2:-2] - vf[:, 1:-3, 2:-2]) / (2. * dy) + dz(V) * sy + dz(W) / D) * 1000.0 / self.dt
        # couplings of cell (k, j, i) to (k + c, j + b, i + a); a neighbour across
        # a side wall or the bottom mirrors onto its image, one above the top is zero
        z = lambda a, p: np.pad(a, p)  # noqa: E731
        xm, xp = z(sx, ((0, 0), (0, 0), (1, 0)))[..., :-1], z(sx, ((0, 0), (0, 0), (0, 1)))[..., 1:]
        ym, yp = z(sy, ((0, 0), (1, 0), (0, 0)))[:, :-1], z(sy, ((0, 0), (0, 1), (0, 0)))[:, 1:]
        one = np.ones_like(sx)
        r6, r13 = A1 / (0.5 * sm * up), A1 / (0.5 * sm * dn)
        cx, cy = 1. / (2. * dx * sm), 1. / (2. * dy * sm)
        st = {(0, 0, 0): 2. / dx ** 2 + 2. / dy ** 2 + r6 + r13, (1, 0, 0): -one / dx ** 2, (-1, 0, 0): -one / dx ** 2,
              (0, 1, 0): -one / dy ** 2, (0, -1, 0): -one / dy ** 2, (0, 0, 1): -r6, (0, 0, -1): -r13,
              (0, -1, 1): (ym + sy) * cy, (-1, 0, 1): (xm + sx) * cx, (1, 0, 1): -(xp + sx) * cx,
              (0, 1, 1): -(yp + sy) * cy, (0, 1, -1): (yp + sy) * cy, (1, 0, -1): (xp + sx) * cx,
              (-1, 0, -1): -(xm + sx) * cx, (0, -1, -1): -(ym + sy) * cy}
        nb = N * K
        B = {a: np.zeros((M, nb, nb)) for a in (-1, 0, 1)}
        kk, jj, ii = np.meshgrid(np.arange(K), np.arange(N), np.arange(M), indexing="ij")
        for (a, b, c), v in st.items():
            i2, j2, k2 = ii + a, jj + b, kk + c
            i2 = np.clip(i2, 0, M - 1)
            j2 = np.clip(j2, 0, N - 1)
            k2 = np.where(k2 < 0, 1, k2)
            ok = k2 < K
            for d in (-1, 0, 1):
                w = ok & (i2 - ii == d)
                np.add.at(B[d], (ii[w], (kk * N + jj)[w], (k2 * N + j2)[w]), v[w])
        r = np.ascontiguousarray(rhs.transpose(2, 0, 1)).reshape(M, nb)
        G, y = np.zeros((M, nb, nb)), np.zeros((M, nb))
        for i in range(M):
            a, v = B[0][i], r[i]
            if i:
                a, v = a - B[-1][i] @ G[i - 1], v - B[-1][i] @ y[i - 1]
            sol = np.linalg.solve(a, np.concatenate([B[1][i], v[:, None]], 1))
            G[i], y[i] = sol[:, :-1], sol[:, -1]
        for i in range(M - 2, -1, -1):
            y[i] -= G[i] @ y[i + 1]
        p = torch.as_tensor(np.ascontiguousarray(y.reshape(M, K, N).transpose(1, 2, 0)), device=self.dev)
        k = slice(2, K + 2)
        self.P[k, 2:-2, 2:-2] = p
        for e in (0, 1):
            self.P[k, 2:-2, 1 - e], self.P[k, 2:-2, -2 + e] = p[..., e], p[..., -1 - e]
            self.P[k, 1 - e, 2:-2], self.P[k, -2 + e, 2:-2] = p[:, min(e, self.N - 1)], p[:, max(self.N - 1 - e, 0)]

"""The calls that programs make of this framework, as cases to be timed and checked.

Every case goes through the public binding (`st_amd`).  Sizes are those of the
repository's tests, benchmark and serving workloads and generic ones between
them; line lengths are the supported ones (16 to 512 points: a power of two, or
3, 5 or 7 times one).

Kinds of case:
  march      one run: Compute_CFL, Compute_Tstep and the RK stages of `steps`
             steps on the resident state (periodic, or with a non-periodic x,
             planar shock and sponge; artificial transport on or off)
  log        what the driver does per step: march, Compute_Grad, diagnostics
  batch      an ensemble of equal grids advanced together
  group      ensembles of four grid sizes advanced together
  serve      a resumed run is admitted to a slot from host memory, advanced and
             stored back
  operators  the operators and right-hand sides that a host program calls one by
             one on its own arrays
Device arrays are (5, nx, nz, ny) here: the state Q(ny, nz, nx, 5) in Fortran
order.  `exact` restates the scheme with every line operator as a dense matrix.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "shock-turbulence_amd", "python"))
import st_amd  # noqa: E402

GAMMA, PR, VIS, CFL = 1.4, 0.7, 0.76, 0.5
MACH, SPONGE = 1.5, (5.0, 2.0, 0.4)
GROUP_SLOTS = {48: 4, 64: 4, 96: 3, 128: 1}      # the ensemble's mix, a quarter of it
LENGTHS = (16, 32, 40, 48, 56, 64, 80, 96, 112, 128, 160, 192, 224, 256, 320, 384, 448, 512)
MOST = 256 ** 3                                   # points of a drawn case


def _grid(kind, name, nx, ny, nz, **kw):
    c = {"name": name, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "hyper": 1, "rk": 0, "shock": False, "steps": 1,
         "slots": 1}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest runs: start-up checks and small decaying boxes, where launches count
        _grid("march", "march_32", 32, 32, 32, steps=2),
        # one small production box by itself (the smallest size of the ensemble)
        _grid("march", "march_48", 48, 48, 48, steps=2),
        # a box with sides of 7, 5 and 7 times a power of two
        _grid("march", "march_112x80x56", 112, 80, 56),
        # direct simulation without artificial transport, the five-stage scheme alone
        _grid("march", "march_128_plain", 128, 128, 128, hyper=0, rk=2),
        # the benchmark's decaying turbulence
        _grid("march", "march_256", 256, 256, 256),
        # a small shock tube with turbulence and sponge layers (non-periodic x)
        _grid("march", "shock_96x32x48", 96, 32, 48, shock=True),
        # the shock-turbulence workload at its full size
        _grid("march", "shock_512x192x192", 512, 192, 192, shock=True),
        # the driver's loop with its log line per step
        _grid("log", "log_96", 96, 96, 96),
        # the ensemble's largest group of equal grids
        _grid("batch", "batch_48x16", 48, 48, 48, slots=16),
        # a mixed ensemble in one launch sequence
        _grid("group", "group_48_to_128", 48, 48, 48),
        # a serving run resumed from host memory, advanced and handed back
        _grid("serve", "serve_64", 64, 64, 64),
        # a host program that calls the operators itself
        _grid("operators", "operators_96x64x80", 96, 64, 80),
    ]


def draw(rng):
    kind = rng.choice(("march", "march", "march", "shock", "log", "batch", "serve", "operators"))
    if kind in ("batch", "serve"):
        most = 96 ** 3
    elif kind == "operators":
        most = 128 ** 3
    else:
        most = MOST
    # points spread over the logarithm, then sides near the cube root, each a supported length
    side = math.exp(rng.uniform(math.log(24.0), math.log(most ** (1.0 / 3.0))))
    n = []
    for stretch in (2.0 if kind == "shock" else 1.0, 1.0, 1.0):
        want = side * stretch * math.exp(rng.uniform(-0.35, 0.35))
        n.append(min(LENGTHS, key=lambda v: abs(math.log(v / want))))
    while n[0] * n[1] * n[2] > most:
        k = n.index(max(n))
        n[k] = LENGTHS[LENGTHS.index(n[k]) - 1]
    pts = n[0] * n[1] * n[2]
    c = _grid("march" if kind == "shock" else kind, None, *n, shock=kind == "shock")
    del c["name"]
    if kind == "march":
        c["hyper"] = rng.choice((1, 1, 0))
        c["rk"] = rng.choice((0, 0, 1, 2))
    if kind in ("march", "shock"):
        c["steps"] = 2 if pts < 64 ** 3 else 1
    if kind == "batch":
        c["slots"] = rng.randint(2, max(2, min(24, 4_000_000 // pts)))
    return c


# ---- inputs ---------------------------------------------------------------

def _params(case):
    """(constructor arguments, k0, Mach number) of a case's flow."""
    if case["shock"]:
        h = 2.0 * np.pi / case["ny"]
        return dict(period=(h * (case["nx"] - 1), 2.0 * np.pi, 2.0 * np.pi), Re=500.0, Pr=PR, hyper_param=1, cfl_cal=CFL,
                    nonperiodic_x=1), 4.0, 1.0
    k0, mt = (8.0, 0.5) if min(case["nx"], case["ny"], case["nz"]) >= 128 else (4.0, 0.3)
    re = st_amd.re_for_taylor(40.0, k0, 1.0, mt, GAMMA, VIS)
    return dict(Re=re, Pr=PR, hyper_param=case["hyper"], cfl_cal=CFL, rk_scheme=case["rk"]), k0, mt


def _turbulence(n, k0, seed):
    """Solenoidal velocity (3, nx, nz, ny), rms 1, spectrum k^4 exp(-2 (k/k0)^2)."""
    nx, ny, nz = n
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    f = torch.randn((3, nx, nz, ny), generator=gen, device="cuda", dtype=torch.float64)
    F = torch.fft.rfftn(f, dim=(1, 2, 3))
    kx = torch.fft.fftfreq(nx, 1.0 / nx, device="cuda", dtype=torch.float64).reshape(-1, 1, 1)
    kz = torch.fft.fftfreq(nz, 1.0 / nz, device="cuda", dtype=torch.float64).reshape(1, -1, 1)
    ky = torch.fft.rfftfreq(ny, 1.0 / ny, device="cuda", dtype=torch.float64).reshape(1, 1, -1)
    k2 = kx * kx + ky * ky + kz * kz
    keep = (2 * kx.abs() < nx) & (2 * kz.abs() < nz) & (2 * ky < ny) & (k2 > 0) & (k2 < (0.5 * min(n)) ** 2)
    amp = torch.where(keep, k2.sqrt() * torch.exp(-k2 / (k0 * k0)), torch.zeros_like(k2))
    F *= amp
    dot = (F[0] * kx + F[1] * ky + F[2] * kz) / torch.where(k2 > 0, k2, torch.ones_like(k2))
    F[0] -= dot * kx
    F[1] -= dot * ky
    F[2] -= dot * kz
    u = torch.fft.irfftn(F, s=(nx, nz, ny), dim=(1, 2, 3))
    return u / u.square().mean().sqrt()


def _shock_states():
    m2, g = MACH * MACH, GAMMA
    r2 = (g + 1.0) * m2 / ((g - 1.0) * m2 + 2.0)
    p2 = (1.0 + 2.0 * g / (g + 1.0) * (m2 - 1.0)) / g
    out = []
    for rho, u, p in ((1.0, MACH, 1.0 / g), (r2, MACH / r2, p2)):
        out.append(np.array([rho * u, 0.0, 0.0, rho, p / (g - 1.0) + 0.5 * rho * u * u]))
    return out


def _state(case, seed, n=None):
    """Conserved state (5, nx, nz, ny) on the GPU."""
    n = n or (case["nx"], case["ny"], case["nz"])
    kw, k0, mt = _params(case)
    u = _turbulence(n, k0, seed)
    if not case["shock"]:
        rho = torch.ones_like(u[0])
        p = torch.full_like(rho, 1.0 / (GAMMA * mt * mt))
    else:
        s1, s2 = _shock_states()
        x = torch.linspace(0.0, 1.0, n[0], device="cuda", dtype=torch.float64).reshape(-1, 1, 1)
        phi = (0.5 * (1.0 + torch.tanh((x - 0.25) * (n[0] - 1) / 2.0))).expand_as(u[0])
        rho = s1[3] + (s2[3] - s1[3]) * phi
        p1, p2 = ((GAMMA - 1.0) * (s[4] - 0.5 * s[0] * s[0] / s[3]) for s in (s1, s2))
        p = p1 + (p2 - p1) * phi
        u = 0.1 * u * (1.0 - phi)
        u[0] += s1[0] / s1[3] + (s2[0] / s2[3] - s1[0] / s1[3]) * phi
    return torch.stack((rho * u[0], rho * u[1], rho * u[2], rho,
                        p / (GAMMA - 1.0) + 0.5 * rho * u.square().sum(0)))


class _Device:
    """A device address of the library as a tensor."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner                              # lives as long as its views
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f8", "version": 3}


def _resident(s):
    """The resident state of a solver or batch, (5, slots, nx, nz, ny)."""
    p = ctypes.POINTER(ctypes.c_double)()
    s._chk(st_amd.lib().st_state_dev(s.h, ctypes.byref(p)), "st_state_dev")
    ny, nz, nx = s.shape
    return torch.as_tensor(_Device(s, ctypes.cast(p, ctypes.c_void_p).value, (5, s.nslots, nx, nz, ny)), device="cuda")


def _host(q):
    """A device array (fields, nx, nz, ny) as the Fortran-ordered host array (ny, nz, nx, fields)."""
    return q.cpu().numpy().T


def prepare(case, seed):
    kw, _, _ = _params(case)
    dims = (case["nx"], case["ny"], case["nz"])
    st = {"case": case}
    if case["kind"] in ("march", "log"):
        s = st_amd.Solver(*dims, **kw)
        if case["shock"]:
            s.sponge(*SPONGE, *_shock_states())
        view = _resident(s)
        view[:, 0] = _state(case, seed)
        torch.cuda.synchronize()
        st.update(s=s, view=view, time=0.0, step=0)
    elif case["kind"] == "batch":
        b = st_amd.Batch(*dims, case["slots"], **kw)
        for k in range(case["slots"]):
            b.load(k, _host(_state(case, 1000 * seed + k)), kw["Re"], 10 ** 9)
        st.update(s=b, view=_resident(b))
    elif case["kind"] == "group":
        bs = []
        for n, ns in GROUP_SLOTS.items():
            b = st_amd.Batch(n, n, n, ns, **kw)
            for k in range(ns):
                b.load(k, _host(_state(case, 1000 * seed + 100 * len(bs) + k, (n, n, n))), kw["Re"], 10 ** 9)
            bs.append(b)
        st.update(s=st_amd.Group(bs), view=[_resident(b) for b in bs])
    elif case["kind"] == "serve":
        st.update(s=st_amd.Batch(*dims, 2, **kw), Q=_host(_state(case, seed)), Re=kw["Re"])
    else:
        q = _state(case, seed)
        u = _turbulence(dims, 4.0, seed + 77)
        st.update(s=st_amd.Solver(*dims, **kw), Q=_host(q), F=_host(u)[..., 0].copy(order="F"), F3=_host(u))
    return st


# ---- one pass -------------------------------------------------------------

def run(st):
    case, s = st["case"], st["s"]
    kind = case["kind"]
    if kind == "march":
        st["time"], st["step"], dts = s.march(case["steps"], st["time"], st["step"])
        return {"Q": st["view"], "dt": dts}
    if kind == "log":
        st["time"], st["step"], dts = s.march(1, st["time"], st["step"])
        maxdil, enst = s.compute_grad()
        return {"Q": st["view"], "dt": dts, "maxdil": float(maxdil), "enstrophy": float(enst), "diag": s.diagnostics()}
    if kind in ("batch", "group"):
        s.march(1)
        return st["view"]
    if kind == "serve":
        s.load(0, st["Q"], st["Re"], 1, time=1.0, step=2)
        s.march(1)
        Q = s.store(0)
        s.release(0)
        return Q
    F, Q = st["F"], st["Q"]
    d1 = [s.dfd(d, F) for d in range(3)]
    d1.append(s.dfd(0, F, dF=d1[1], iadd=1, cadd=-1.0))
    d2 = [s.d2fd2(d, F) for d in range(2)] + list(s.d2fd2(2, F, iadd=1))
    r = s.rhs(Q)
    h = s.hyper_rhs(r)
    return {"d1": d1, "d2": d2, "filter": s.compact_filter(st["F3"]), "gauss": s.gaussian_filter(F), "rhs": r, "full": h,
            "fixed": s.fix_pressure(Q)}


# ---- what a pass cannot do without -----------------------------------------

def _stages(case):
    return {0: 11, 1: 11, 2: 5}[case["rk"]]


def work(case):
    """Bytes: a stage reads and writes the state and the register of the
    low-storage scheme (20 fields); host operators read and write their arrays
    once.  Operations: about 2000 a point and stage with the artificial
    transport, 1200 without (the scheme's own count)."""
    pts = case["nx"] * case["ny"] * case["nz"]
    kind = case["kind"]
    if kind == "operators":
        # 5 + 5 line derivatives and filters of one or three fields, two right-hand sides and a fix of five
        return {"bytes": 8.0 * pts * (4 * 2 + 1 + 4 + 2 + 6 + 2 + 10 + 10 + 10), "flops": 2200.0 * pts}
    if kind == "group":
        pts = sum(n ** 3 * s for n, s in GROUP_SLOTS.items())
    elif kind == "batch":
        pts *= case["slots"]
    stages = _stages(case) * (case["steps"] if kind == "march" else 1)
    extra = 10.0 * pts if kind in ("log", "serve") else 0.0
    return {"bytes": 8.0 * (20.0 * pts * stages + extra), "flops": (2000.0 if case["hyper"] else 1200.0) * pts * stages}


# ---- the scheme in 64 bits with dense operators ----------------------------

CC5 = ((0.0, -4.801594388477952e-01, -1.404247195200064e+00, -2.016477077503357e+00, -1.056444269767207e+00),
       (1.028639988104959e-01, 7.408540575766301e-01, 7.426530946683799e-01, 4.694937902357905e-01, 1.881733382887932e-01))
LD6 = ((0.0, -4.4127377153877382565e-1, -1.073982008079781868e0, -1.7063570791256758809e0, -2.7979293162682443056e0,
        -4.0913537120919160454e0),
       (1.1584888181285561688e-1, 3.7287699051652864918e-1, 7.3795368921435295698e-1, 5.7981109366311039538e-1,
        1.031284991300145194e0, 1.5e-1))
LD5 = ((0.0, -6.0512264332862261228e-1, -2.04375640234761394333e0, -0.74069990637544192841e0, -4.42317651302968168941e0),
       (2.6874543888713438496e-1, 8.014706973220802933e-1, 5.0515704269422722538e-1, 5.6235680379000296407e-1,
        5.900655127758823335e-2))
AL, BE = 0.66624, 0.16688


def _matrix(op, n, h, closed):
    """Dense n x n matrix of a line operator; closed: with boundary rows."""
    A, B = np.zeros((n, n)), np.zeros((n, n))
    i = np.arange(n)

    def band(M, off, v):
        M[i, (i + off) % n] += v

    if op == "d1":
        left, right = (1.0 / 3.0,), {1: 14.0 / 18.0, 2: 1.0 / 36.0}
        for m, v in right.items():
            band(B, m, v / h)
            band(B, -m, -v / h)
    elif op == "d2":
        left, right = (2.0 / 11.0,), {1: 12.0 / 11.0, 2: 3.0 / 44.0}
        for m, v in right.items():
            band(B, m, v / h ** 2)
            band(B, -m, v / h ** 2)
            band(B, 0, -2.0 * v / h ** 2)
    elif op == "filter":
        left = (AL, BE)
        for m, v in enumerate((0.99965, 0.66652, 0.16674, 4.0e-5, -5.0e-6)):
            for o in {m, -m}:
                band(B, o, v)
    else:
        left = ()
        for m, v in enumerate((3565.0 / 10368.0, 3091.0 / 12960.0, 1997.0 / 25920.0, 149.0 / 12960.0, 107.0 / 103680.0)):
            for o in {m, -m}:
                if closed:                              # mirrored at the ends
                    j = np.abs(i + o)
                    np.add.at(B, (i, np.where(j > n - 1, 2 * (n - 1) - j, j)), v)
                else:
                    band(B, o, v)
        return B
    band(A, 0, 1.0)
    for m, v in enumerate(left):
        band(A, m + 1, v)
        band(A, -m - 1, v)
    if closed:
        ab = 0.45
        rows = {
            "d1": [({0: 1, 1: 2}, [-2.5, 2.0, 0.5]), ({0: 1 / 6, 1: 1, 2: 0.5}, [-5 / 9, -0.5, 1.0, 1 / 18])],
            "d2": [({0: 1, 1: 11}, [13.0, -27.0, 15.0, -1.0]),
                   ({0: 0.1, 1: 1, 2: -0.35}, [1.2375, -3.0, 2.325, -0.6, 0.0375])],
            "filter": [({0: 1}, [15 / 16, 1 / 4, -3 / 8, 1 / 4, -1 / 16]),
                       ({0: ab, 1: 1, 2: ab}, [1 / 16 + 7 / 8 * ab, 3 / 4 + ab / 2, 3 / 8 + ab / 4, -1 / 4 + ab / 2,
                                               1 / 16 - ab / 8]),
                       ({1: ab, 2: 1, 3: ab}, [(-1 / 8 + ab / 4) / 2, (1 / 2 + ab) / 2, 5 / 8 + 3 / 4 * ab,
                                               (1 / 2 + ab) / 2, (-1 / 8 + ab / 4) / 2]),
                       ({1: BE, 2: AL, 3: 1, 4: AL, 5: BE},
                        [(1 / 32 - AL / 16 + BE / 16) / 2, (-3 / 16 + 3 / 8 * AL + 13 / 8 * BE) / 2,
                         (15 / 32 + 17 / 16 * AL + 15 / 16 * BE) / 2, 11 / 16 + 5 / 8 * AL - 5 / 8 * BE,
                         (15 / 32 + 17 / 16 * AL + 15 / 16 * BE) / 2, (-3 / 16 + 3 / 8 * AL + 13 / 8 * BE) / 2,
                         (1 / 32 - AL / 16 + BE / 16) / 2])],
        }[op]
        scale = {"d1": 1.0 / h, "d2": 1.0 / h ** 2, "filter": 1.0}[op]
        for r, (lhs, rhs) in enumerate(rows):
            for end in (False, True):
                at = (lambda k: n - 1 - k) if end else (lambda k: k)
                A[at(r)] = 0.0
                B[at(r)] = 0.0
                for k, v in lhs.items():
                    A[at(r), at(k)] = v
                for k, v in enumerate(rhs):
                    B[at(r), at(k)] = scale * (-v if end and op == "d1" else v)
    return np.linalg.solve(A, B)


class _Exact:
    """One periodic or closed-x grid; fields are (nx, nz, ny) in 64 bits."""

    def __init__(self, case, n, dev):
        kw, _, _ = _params(case)
        self.shock, self.hyper, self.rk = case["shock"], case["hyper"], case["rk"]
        per = kw.get("period", (2.0 * np.pi,) * 3)
        self.h = [per[d] / (n[d] - 1 if self.shock and d == 0 else n[d]) for d in range(3)]
        self.re = 1.0 / kw["Re"]
        self.M = {(op, d): torch.from_numpy(_matrix(op, n[d], self.h[d], self.shock and d == 0)).to(dev)
                  for op in ("d1", "d2", "filter", "gauss") for d in range(3)}
        self.sigma = None
        if self.shock:
            amp, power, frac = SPONGE
            left = math.ceil(frac * n[0] / 2.0)
            g = np.arange(1, n[0] + 1)
            one = np.float32(1.0) * (left - g + 1).astype(np.float32) / np.float32(left)
            two = (g - (n[0] - left)).astype(np.float32) / np.float32(left)
            sig = np.where(g <= left, one, np.where(g >= n[0] - left, two, 0)).astype(np.float64) ** power * amp
            ref = np.where(g[:, None] <= left, *_shock_states())
            self.sigma = torch.from_numpy(sig).to(dev).reshape(-1, 1, 1)
            self.ref = torch.from_numpy(ref.T.copy()).to(dev).reshape(5, -1, 1, 1)

    def on(self, op, d, f):
        M = self.M[op, d]
        if d == 0:
            return (M @ f.reshape(f.shape[0], -1)).reshape(f.shape)
        if d == 1:
            return (f.reshape(-1, f.shape[2]) @ M.T.contiguous()).reshape(f.shape)
        return torch.matmul(M, f)

    def d1(self, d, f):
        return self.on("d1", d, f)

    def lap(self, f):
        return sum(self.on("d2", d, f) for d in range(3))

    def smooth(self, op, f):
        for d in (1, 2, 0):
            f = self.on(op, d, f)
        return f

    def prim(self, Q):
        e = (Q[4] - 0.5 * (Q[0] ** 2 + Q[1] ** 2 + Q[2] ** 2) / Q[3]) / Q[3]
        return [Q[i] / Q[3] for i in range(3)], (GAMMA - 1.0) * Q[3] * e, GAMMA * e

    def rhs(self, Q):
        """The convective and viscous right-hand side and the gradients
        du[i][d], dT[d]."""
        rho = Q[3]
        u, p, T = self.prim(Q)
        mu = ((GAMMA - 1.0) * T) ** VIS * self.re
        mup = VIS * mu / T
        du = [[self.d1(d, u[i]) for d in range(3)] for i in range(3)]
        dT = [self.d1(d, T) for d in range(3)]
        dil = du[0][0] + du[1][1] + du[2][2]
        out = []
        energy = -sum(self.d1(d, (Q[4] + p) * u[d]) for d in range(3))
        energy += (mu * self.lap(T) + mup * sum(g * g for g in dT)) / PR
        for i in range(3):
            f = -self.d1(i, p)
            for d in range(3):
                f -= 0.5 * (self.d1(d, rho * u[i] * u[d]) + u[i] * self.d1(d, rho * u[d]) + rho * u[d] * du[i][d])
            visc = sum((4.0 / 3.0 if d == i else 1.0) * self.on("d2", d, u[i]) for d in range(3))
            visc = mu * (visc + sum(self.d1(i, du[j][j]) for j in range(3) if j != i) / 3.0)
            visc += mup * sum(dT[j] * (du[i][j] + du[j][i]) for j in range(3)) - 2.0 / 3.0 * mup * dT[i] * dil
            out.append(f + visc)
            energy += u[i] * visc
        strain = sum(2.0 * du[i][i] ** 2 for i in range(3)) - 2.0 / 3.0 * dil ** 2
        strain += (du[0][1] + du[1][0]) ** 2 + (du[0][2] + du[2][0]) ** 2 + (du[1][2] + du[2][1]) ** 2
        out.append(-sum(self.d1(d, rho * u[d]) for d in range(3)))
        out.append(energy + mu * strain)
        return torch.stack(out), du, dT

    def coefficients(self, Q, du, S=None):
        """beta*, mu*, kappa* (S: the strain magnitude, 0 without gradients)."""
        u, p, T = self.prim(Q)
        if self.shock:
            cb = 1.0
        else:
            dil = du[0][0] + du[1][1] + du[2][2]
            om2 = (du[2][1] - du[1][2]) ** 2 + (du[0][2] - du[2][0]) ** 2 + (du[1][0] - du[0][1]) ** 2
            cb = 0.5 * (1.0 - torch.tanh(2.5 + 10.0 * dil)) * dil ** 2 / (dil ** 2 + om2 + 1.0e-7) + 1.0e-20
        if S is None:
            S = sum(du[i][i] ** 2 for i in range(3))
            S = S + 0.5 * ((du[0][1] + du[1][0]) ** 2 + (du[0][2] + du[2][0]) ** 2 + (du[1][2] + du[2][1]) ** 2)
            S = torch.sqrt(0.5 * S)
        s4 = self.smooth("gauss", Q[3] * self.lap(self.lap(S)).abs())
        e4 = self.smooth("gauss", Q[3] / T * torch.sqrt(GAMMA * p / Q[3]) * self.lap(self.lap(T / GAMMA)).abs())
        return cb * s4 * self.h[0] ** 6, 2.0e-3 * s4 * self.h[0] ** 6, 1.0e-2 * e4 * self.h[0] ** 5

    def full(self, Q):
        r, du, dT = self.rhs(Q)
        H = None
        if self.hyper:
            H = self.coefficients(Q, du)
            r = r + self.transport(Q, du, dT, H)
        return r, H

    def transport(self, Q, du, dT, H):
        beta, mu, kap = H
        u = [Q[i] / Q[3] for i in range(3)]
        dil = du[0][0] + du[1][1] + du[2][2]
        out = [torch.zeros_like(dil) for _ in range(5)]
        for d in range(3):
            heat = kap * dT[d]
            for i in range(3):
                t = mu * (du[i][d] + du[d][i])
                if i == d:
                    t = t + (beta - 2.0 / 3.0 * mu) * dil
                out[i] = out[i] + self.d1(d, t)
                heat = heat + u[i] * t
            out[4] = out[4] + self.d1(d, heat)
        return torch.stack(out)

    def dt(self, Q, H):
        u, p, T = self.prim(Q)
        c = torch.sqrt(GAMMA * p / Q[3])
        dt = CFL / float(sum((c + u[d].abs()) * 2.199 / self.h[d] for d in range(3)).max())
        if H is not None:
            h2 = self.h[0] ** 2
            dt = min([dt] + [float(np.float32(0.2)) * float(v.min()) for v in
                             (Q[3] * h2 / H[1], Q[3] * h2 / H[0], Q[3] * h2 * c * c / (H[2] * T))])
        return dt

    def fix(self, Q):
        ke = 0.5 * (Q[0] ** 2 + Q[1] ** 2 + Q[2] ** 2) / Q[3]
        p = (GAMMA - 1.0) * (Q[4] - ke)
        Q = Q.clone()
        Q[4] = torch.where(p < 0.0, torch.full_like(p, 0.71463), p) / (GAMMA - 1.0) + ke
        return Q

    def step(self, Q, dt):
        H = None
        for table in {0: (CC5, LD6), 1: (LD5, LD6), 2: (CC5,)}[self.rk]:
            W = torch.zeros_like(Q)
            for a, b in zip(*table):
                r, H = self.full(Q)
                if self.sigma is not None:
                    r = r - self.sigma * (Q - self.ref)
                W = a * W + dt * r
                Q = Q + b * W
                Q = self.fix(torch.stack([self.smooth("filter", q) for q in Q]))
        return Q, H

    def march(self, Q, steps, step=0, H=None):
        """Steps from the driver's counter `step`; H limits dt from step 2 on
        (with a closed x, from the first step)."""
        dts = []
        for k in range(step, step + steps):
            dts.append(self.dt(Q, H if self.shock or k > 1 else None))
            Q, H = self.step(Q, dts[-1])
        return Q, dts


def exact(case, seed):
    dims = (case["nx"], case["ny"], case["nz"])
    kind = case["kind"]
    if kind in ("march", "log"):
        X, Q = _Exact(case, dims, "cuda"), _state(case, seed)
        Q, dts = X.march(Q, case["steps"])
        out = {"Q": Q[:, None], "dt": np.array(dts)}
        if kind == "log":
            u, p, _ = X.prim(Q)
            du = [[X.d1(d, u[i]) for d in range(3)] for i in range(3)]
            om2 = (du[2][1] - du[1][2]) ** 2 + (du[0][2] - du[2][0]) ** 2 + (du[1][0] - du[0][1]) ** 2
            ke = 0.5 * (Q[0] ** 2 + Q[1] ** 2 + Q[2] ** 2) / Q[3]
            ent = Q[3] * torch.log(p * Q[3] ** -GAMMA)
            out.update(maxdil=float((du[0][0] + du[1][1] + du[2][2]).abs().max()), enstrophy=0.5 * float(om2.mean()),
                       diag=torch.stack([f.mean() for f in (Q[0], Q[1], Q[2], ke, Q[3], Q[4], ent)]).cpu().numpy())
        return out
    if kind == "batch":
        X = _Exact(case, dims, "cuda")
        return torch.stack([X.march(_state(case, 1000 * seed + k), 1)[0] for k in range(case["slots"])], dim=1)
    if kind == "group":
        out = []
        for g, (n, ns) in enumerate(GROUP_SLOTS.items()):
            X = _Exact(case, (n, n, n), "cuda")
            out.append(torch.stack([X.march(_state(case, 1000 * seed + 100 * g + k, (n, n, n)), 1)[0] for k in range(ns)],
                                   dim=1))
        return out
    X, Q = _Exact(case, dims, "cuda"), _state(case, seed)
    if kind == "serve":
        u, _, _ = X.prim(Q)
        du = [[X.d1(d, u[i]) for d in range(3)] for i in range(3)]
        return _host(X.march(Q, 1, 2, X.coefficients(Q, du, torch.zeros_like(Q[3])))[0])
    F3 = _turbulence(dims, 4.0, seed + 77)
    F = F3[0]
    d1 = [X.d1(d, F) for d in range(3)]
    rhs, du, dT = X.rhs(Q)
    full = rhs + X.transport(Q, du, dT, X.coefficients(Q, du))
    return {"d1": [_host(f) for f in d1 + [d1[1] - d1[0]]],
            "d2": [_host(X.on("d2", d, F)) for d in range(2)] + [_host(d1[2]), _host(X.on("d2", 2, F))],
            "filter": _host(torch.stack([X.smooth("filter", f) for f in F3])), "gauss": _host(X.smooth("gauss", F)),
            "rhs": _host(rhs), "full": _host(full), "fixed": _host(X.fix(Q))}

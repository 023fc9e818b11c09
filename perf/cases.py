"""The work that users of this solver have it do, as measured cases.

Kinds of a case:

  run       a running box (its first step taken) advances `steps` RK3 steps and hands over the
            real-space state as the output files hold it (stage_output / staged_output). With
            `host_loop` it is driven as the Fortran host drives it: one step at a time, time and dt
            read after each. With `closure` the learned closure is on.
  ensemble  `boxes` independent boxes of each of three sizes advance `steps` steps; every box's state
            is read.
  train     `steps` Adam steps of the closure network on batches of (n, 28) / (n, 18) samples.
  filter    a fine run advances `steps` steps and hands over the box-filtered fields the closure is
            trained on.
  restart   a state is loaded from host memory and its CFL step, moments, budgets and spectrum are read.

Double-precision runs return double-precision fields. Runs whose transforms or network are in single
precision return single-precision fields: that is what their snapshots hold.

exact() restates the method in 64 bits, apart from the library. Its transforms, and those that make the
inputs, are products with the DFT matrix of each axis (lengths up to 512): plain, and as exact as an FFT.
"""
import math

import numpy as np
import torch

from laps_amd.closure import init_params
from laps_amd.params import LAPS_FP64, LAPS_MIXED, default_params
from laps_amd.runtime import Ensemble, Laps, mlp_train

GAMMA = 5.0 / 3.0
TWO_PI = 2.0 * math.pi
LENGTHS = (16, 32, 64, 96, 128, 256, 512)


def _run(name, n, precision, dealias, hall, steps, **kw):
    c = dict(kind="run", nx=n[0], ny=n[1], nz=n[2], precision=precision, dealias=dealias, hall=hall, aeb=False,
             closure=False, host_loop=False, steps=steps)
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest box, driven as the Fortran host drives it: launches and host reads count
        _run("box32_host_loop", (32, 32, 32), "fp64", 1, False, 10, host_loop=True),
        # a small non-cubic expanding box with a 96-point axis and phase-shift dealiasing
        _run("ebox96x32x64_shift", (96, 32, 64), "fp64", 3, True, 20, aeb=True),
        # the solver's default grid and compact filter, double precision
        _run("default128x128x64_filter", (128, 128, 64), "fp64", 2, False, 40),
        # the 256^3 Hall workload: double and mixed precision, phase shift, and the 2/3 rule
        _run("hall256_shift_fp64", (256, 256, 256), "fp64", 3, True, 10),
        _run("hall256_shift_mixed", (256, 256, 256), "mixed", 3, True, 16),
        _run("hall256_twothirds_fp64", (256, 256, 256), "fp64", 1, True, 20),
        # the corotating expanding box with 512-point axes, mixed precision: the largest
        _run("ebox512x512x128_mixed", (512, 512, 128), "mixed", 1, True, 12, aeb=True),
        # parameter scan: 8 boxes each of 32^3, 64^3 and 96^3 in one ensemble
        dict(name="ensemble24", kind="ensemble", n0=32, n1=64, n2=96, boxes=8, precision="mixed", steps=48),
        # the closure: a coarse run that uses it, its training, and its training data
        _run("closure64", (64, 64, 64), "fp64", 1, True, 20, closure=True),
        dict(name="train4096", kind="train", n=65536, batch=4096, steps=40),
        dict(name="filter128to32", kind="filter", nx=128, ny=128, nz=128, r=4, steps=4),
        # start of a run from a restart file, with its first diagnostics
        dict(name="restart128", kind="restart", nx=128, ny=128, nz=128),
    ]


def draw(rng):
    kind = rng.choice(("run",) * 7 + ("ensemble", "closure", "train", "train", "filter", "restart"))
    if kind == "train":
        n = int(2 ** rng.uniform(9, 16))
        return dict(kind="train", n=n, batch=max(64, int(n / 2 ** rng.uniform(0, 5))), steps=rng.randint(4, 40))
    if kind == "ensemble":
        n = rng.sample((16, 32, 64, 96), 3)
        return dict(kind="ensemble", n0=n[0], n1=n[1], n2=n[2], boxes=rng.randint(1, 6),
                    precision=rng.choice(("fp64", "mixed")), steps=rng.randint(2, 20))

    def grid(most):
        while True:
            g = [rng.choice(LENGTHS) for _ in range(3)]
            p = g[0] * g[1] * g[2]
            if 2 ** 12 <= p <= most and rng.random() < 0.25 + math.log2(p) / 32:
                return g, p

    if kind == "filter":
        (nx, ny, nz), _ = grid(2 ** 22)
        return dict(kind="filter", nx=nx, ny=ny, nz=nz, r=rng.choice((1, 2, 4, 8)), steps=rng.randint(1, 6))
    if kind == "restart":
        (nx, ny, nz), _ = grid(2 ** 22)
        return dict(kind="restart", nx=nx, ny=ny, nz=nz)
    closure = kind == "closure"
    n, pts = grid(2 ** 21 if closure else 2 ** 24)
    steps = max(2, min(40, int(2 ** 27 / pts * rng.uniform(0.3, 1.0))))
    dealias = rng.choice((1, 2, 3))
    return _run(None, n, "fp64" if closure else rng.choice(("fp64", "mixed")), dealias, rng.random() < 0.7, steps,
                aeb=not closure and rng.random() < 0.3, closure=closure,
                host_loop=pts <= 2 ** 17 and rng.random() < 0.5)


# ------------------------------------------------------------------ inputs

def _params(c, n=None, di=None):
    nx, ny, nz = n or (c["nx"], c["ny"], c["nz"])
    kw = dict(nx=nx, ny=ny, nz=nz, Lx=TWO_PI, Ly=TWO_PI, Lz=TWO_PI, adiabatic_index=GAMMA, cfl=0.2,
              dealias_option=c.get("dealias", 1), if_visc=1, viscosity=2e-3, if_resis=1, resistivity=2e-3,
              precision=LAPS_MIXED if c.get("precision") == "mixed" else LAPS_FP64)
    hall = c.get("hall", True) if di is None else di > 0
    if hall:
        kw.update(if_hall=1, ion_inertial_length=0.05 if di is None else di)
    if c.get("aeb"):
        kw.update(if_aeb=1, if_corotating=1, radius0=1.0, Ur0=0.5, corotating_angle=0.25)
    return default_params(**kw)


def _modes(n):
    m = torch.arange(n, dtype=torch.float64, device="cuda")
    return torch.where(m <= n // 2, m, m - n)


def _dft(n, sign):
    t = (torch.arange(n, device="cuda")[:, None] * torch.arange(n, device="cuda")[None, :]) % n
    a = t.double() * (TWO_PI / n)
    return torch.complex(torch.cos(a), sign * torch.sin(a))


def _fwd(f):
    """the half spectrum [z][y][kx] of one real field [z][y][x], divided by the number of points"""
    nz, ny, nx = f.shape
    w = _dft(nx, -1)[:, : nx // 2 + 1] / nx
    f = torch.complex(f @ w.real.contiguous(), f @ w.imag.contiguous())
    f = torch.tensordot(f, _dft(ny, -1) / ny, dims=([1], [0]))                  # [z][kx][ky]
    return torch.tensordot(f, _dft(nz, -1) / nz, dims=([0], [0])).permute(2, 1, 0).contiguous()


def _inv(f, nx):
    """the real field of a half spectrum (the imaginary parts of kx = 0 and nx/2 do not enter)"""
    nz, ny, nxh = f.shape
    f = torch.tensordot(f, _dft(nz, 1), dims=([0], [0]))                        # [ky][kx][z]
    f = torch.tensordot(f, _dft(ny, 1), dims=([0], [0])).permute(1, 2, 0)       # [z][y][kx]
    w = _dft(nx, 1)[:nxh] * 2.0
    w[0] *= 0.5
    w[-1] *= 0.5
    return f.real.contiguous() @ w.real.contiguous() - f.imag.contiguous() @ w.imag.contiguous()


def _state(nx, ny, nz, seed, amp=0.2):
    """Conserved (8) and primitive (4) fields [field][z][y][x] on the GPU: rho = p = 1, B0 = (1, 0, 0) and
    random modes in shells 1 to n/8 with amplitude |k|^(-5/3), rms |db| = rms |du| = amp, div b = 0."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    mx, my, mz = _modes(nx)[None, None, : nx // 2 + 1], _modes(ny)[None, :, None], _modes(nz)[:, None, None]
    k2 = mx * mx + my * my + mz * mz
    shell = torch.round(torch.sqrt(k2))
    kmax = max(2, min(nx, ny, nz) // 8)
    w = torch.where((shell >= 1) & (shell <= kmax), k2.clamp(min=1.0) ** (-5.0 / 6.0), torch.zeros_like(k2))

    def modes():
        r = torch.randn((3, nz, ny, nx), generator=g, dtype=torch.float64, device="cuda")
        return torch.stack([_fwd(a) * w for a in r])

    def field(f):
        v = torch.stack([_inv(a, nx) for a in f])
        return v * (amp / torch.sqrt((v * v).sum(0).mean()))

    u = field(modes())
    bh = modes()
    kb = (mx * bh[0] + my * bh[1] + mz * bh[2]) / k2.clamp(min=1.0)
    b = field(torch.stack((bh[0] - mx * kb, bh[1] - my * kb, bh[2] - mz * kb)))
    b[0] += 1.0
    one = torch.ones((nz, ny, nx), dtype=torch.float64, device="cuda")
    e = one / (GAMMA - 1.0) + 0.5 * ((u * u).sum(0) + (b * b).sum(0))
    return torch.cat((one[None], u, b, e[None])), torch.cat((u, one[None]))


def _host(t):
    """a GPU array [field][z][y][x] as the library's host layout (nx, ny, nz, field)"""
    return t.cpu().numpy().T


def _closure_vector(seed):
    """A closure network with outputs of the size of subgrid stresses, and the normalisation it was trained
    with."""
    p = init_params(seed)
    xstd = np.concatenate([np.full(7, 0.3), np.full(21, 1.0)])
    xmean = np.zeros(28)
    xmean[0] = xmean[4] = 1.0
    return np.concatenate([p, xmean, xstd, np.full(18, 2e-3)]).astype(np.float32)


def _samples(n, seed):
    """Normalised features and targets as the training has them: the targets a smooth function of the features
    with noise."""
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((n, 28), dtype=np.float32)
    A = rng.standard_normal((28, 18), dtype=np.float32) / 6.0
    T = np.tanh(X @ A) + 0.3 * rng.standard_normal((n, 18), dtype=np.float32)
    return X, T.astype(np.float32)


def _boxes(c):
    """(n, d_i, amplitude) of each box of an ensemble: d_i alternates, the amplitude varies"""
    return [(n, 0.05 if i % 2 else 0.0, 0.1 + 0.3 * i / c["boxes"])
            for n in (c["n0"], c["n1"], c["n2"]) for i in range(c["boxes"])]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        X, T = _samples(case["n"], seed)
        return dict(case=case, X=X, T=T, P=init_params(seed))
    if kind == "ensemble":
        e = Ensemble([_params(dict(case, dealias=1), (n, n, n), di) for n, di, _ in _boxes(case)])
        for i, (n, _, amp) in enumerate(_boxes(case)):
            uu, pr = _state(n, n, n, seed * 1000 + i, amp)
            e.box(i).set_state(_host(uu), _host(pr))
        e.step(1)
        e.sync()
        return dict(case=case, e=e)
    uu, pr = (_host(t) for t in _state(case["nx"], case["ny"], case["nz"], seed))
    g = Laps(_params(case))
    if kind == "restart":
        return dict(case=case, g=g, uu=uu, pr=pr)
    g.set_state(uu, pr)
    if case.get("closure"):
        g.closure_set(_closure_vector(seed))
    g.step(1)
    g.sync()
    return dict(case=case, g=g)


# ------------------------------------------------------------------ one pass

class _Payload(np.ndarray):
    """a view of a context's pinned output buffer, which lives as long as the context does"""
    context = None


def _single(a):
    """a double-precision array in the library's layout as single precision"""
    return torch.from_numpy(a.T).to(torch.float32)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "train":
        P, hist = mlp_train(state["X"], state["T"], state["P"], case["steps"], case["batch"], 2e-3)
        return P, hist
    if kind == "ensemble":
        e = state["e"]
        e.step(case["steps"])
        out = [b.state()[0].T for b in e.boxes]
        if case["precision"] == "mixed":
            out = [torch.from_numpy(a).to(torch.float32) for a in out]
            return [torch.stack(out[i * case["boxes"]:(i + 1) * case["boxes"]]) for i in range(3)]
        return [np.stack(out[i * case["boxes"]:(i + 1) * case["boxes"]]) for i in range(3)]
    g = state["g"]
    if kind == "filter":
        g.step(case["steps"])
        return g.closure_filter(case["r"]).T
    if kind == "restart":
        g.set_state(state["uu"], state["pr"])
        dtmin, _ = g.cfl()
        ave, var, ru2 = g.moments()
        bud = g.budgets()
        return dict(dt=dtmin, ave=ave, var=var[1:7], ru2=ru2, energy=[bud[k] for k in
                    ("e", "kinetic", "magnetic", "internal")], spectrum=g.spectral().T)
    if case["host_loop"]:
        for _ in range(case["steps"]):
            g.step(1)
            g.scalars()
    else:
        g.step(case["steps"])
    g.stage_output(primitive=False)
    w, t, dt, _ = g.staged_output(copy=False)
    if case["precision"] == "mixed" or case["closure"]:
        return dict(time=np.float32(t), dt=np.float32(dt), state=_single(w))
    w = w.T.view(_Payload)
    w.context = g
    return dict(time=t, dt=dt, state=w)


# ------------------------------------------------------------------ work

def _mask(dealias, n):
    """factor of every mode [z][y][x] that the dealiasing leaves"""
    nx, ny, nz = n
    ax, ay, az = _modes(nx)[: nx // 2 + 1] / nx, _modes(ny) / ny, _modes(nz) / nz
    r2 = (ax * ax)[None, None, :] + (ay * ay)[None, :, None] + (az * az)[:, None, None]
    if dealias == 1:
        return (torch.sqrt(r2) <= 1.0 / 3.0).double()
    if dealias == 3:
        mx, my, mz = ((_modes(k) ** 2).long() for k in n)
        x2, y2, z2 = nx * nx, ny * ny, nz * nz
        s = (mx[: nx // 2 + 1] * (y2 * z2))[None, None, :] + (my * (x2 * z2))[None, :, None] + \
            (mz * (x2 * y2))[:, None, None]
        return (9 * s < 2 * x2 * y2 * z2).double()
    af = 0.495
    a, b, c = (5 + 6 * af) / 8, (1 + 2 * af) / 2, -(1 - 2 * af) / 8

    def f(m):
        t = TWO_PI * m
        return (a + b * torch.cos(t) + c * torch.cos(2 * t)) / (1 + 2 * af * torch.cos(t))

    return f(ax)[None, None, :] * f(ay)[None, :, None] * f(az)[:, None, None]


def _step_work(n, dealias, hall, aeb, steps):
    """Of `steps` RK3 steps of one box: per substage the kept state read and written and the previous right-hand
    side read and written once; the flops of the transforms (8 fields and, with Hall, the current to real space,
    12 products back, 13 with the expanding box's source; twice on the shifted grid)."""
    pts = float(n[0] * n[1] * n[2])
    kept = {1: 4.0 / 3.0 * math.pi / 27.0, 3: 4.0 / 3.0 * math.pi * (math.sqrt(2.0) / 3.0) ** 3}.get(dealias, 1.0) * pts / 2
    nf = 8 + (3 if hall else 0) + 12 + (1 if aeb else 0)
    grids = 2 if dealias == 3 else 1
    return 3 * steps * kept * 16 * 8 * 4, 3 * steps * grids * pts * (nf * 2.5 * math.log2(pts) + 100)


def work(case):
    kind = case["kind"]
    if kind == "train":
        b = min(case["batch"], case["n"])
        return dict(bytes=4.0 * (min(case["n"], case["steps"] * b) * 46 + 2 * 7186),
                    flops=6.0 * case["steps"] * b * 7040)
    if kind == "ensemble":
        by = fl = 0.0
        for n, di, _ in _boxes(case):
            s = _step_work((n, n, n), 1, di > 0, False, case["steps"])
            by += s[0] + 64.0 * n ** 3
            fl += s[1]
        return dict(bytes=by, flops=fl)
    n = (case["nx"], case["ny"], case["nz"])
    pts = float(n[0] * n[1] * n[2])
    if kind == "restart":
        return dict(bytes=pts * (12 * 8 + 8 * 8), flops=pts * 8 * 2.5 * math.log2(pts))
    by, fl = _step_work(n, case.get("dealias", 1), case.get("hall", True), case.get("aeb", False), case["steps"])
    if kind == "filter":
        return dict(bytes=by + pts * 8 * 26 / case["r"] ** 3, flops=fl + pts * (11 * 2.5 * math.log2(pts) + 100))
    if case["closure"]:
        fl += case["steps"] * pts * (2.0 * 7040 + 20 * 2.5 * math.log2(pts))
    return dict(bytes=by + pts * 8 * 8, flops=fl)


# ------------------------------------------------------------------ the method in 64 bits

PAIRS = ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))
IDX = ((0, 1, 2), (1, 3, 4), (2, 4, 5))


class _Box:
    """The solver's step in plain torch: RK3 in spectral space, products in real space."""

    def __init__(self, p, uu, prim, net=None):
        self.p, self.n = p, (p.nx, p.ny, p.nz)
        nx, ny, nz = self.n
        self.w = (_modes(nx)[None, None, : nx // 2 + 1], _modes(ny)[None, :, None], _modes(nz)[:, None, None])
        self.mask = _mask(p.dealias_option, self.n)
        self.real, self.prim = uu, prim
        self.U = torch.stack([self.fwd(f) for f in uu])
        self.net = net
        self.fresh, self.time, self.dt, self.prev = True, 0.0, 0.0, 0.0
        self.phase = None
        if p.dealias_option == 3:
            def ph(m, n):
                return torch.exp(1j * math.pi * m / n)
            self.phase = ph(self.w[0], nx) * ph(self.w[1], ny) * ph(self.w[2], nz)

    def fwd(self, f):
        return _fwd(f)

    def inv(self, f):
        return torch.stack([_inv(a, self.n[0]) for a in f])

    def radius(self):
        return self.p.radius0 + (self.p.Ur0 if self.p.if_aeb else 0.0) * self.time

    def k(self):
        r = self.p.radius0 / self.radius()
        wx, wy, wz = self.w
        if self.p.if_aeb and self.p.if_corotating:
            c, s = math.cos(self.p.corotating_angle), math.sin(self.p.corotating_angle)
            return wx * c + wy * s, (-wx * s + wy * c) * r, wz * r
        return wx, wy * r, wz * r

    def curl(self, B):
        k = self.k()
        return [1j * (k[(a + 1) % 3] * B[(a + 2) % 3] - k[(a + 2) % 3] * B[(a + 1) % 3]) for a in range(3)]

    def primitives(self, f):
        u = f[1:4] / f[0]
        p = (GAMMA - 1) * (f[7] - 0.5 * (f[1:4] * u).sum(0) - 0.5 * (f[4:7] ** 2).sum(0))
        return torch.cat((u, p[None]))

    def cfl(self, f, q):
        p = self.p
        d = (p.Lx / p.nx, p.Ly / p.ny, p.Lz / p.nz)
        rr = self.radius() / p.radius0
        cs2 = p.adiabatic_index * q[3] / f[0]
        ca = [f[4 + a] / torch.sqrt(f[0]) for a in range(3)]
        cms2 = cs2 + ca[0] ** 2 + ca[1] ** 2 + ca[2] ** 2
        out = None
        for a in range(3):
            cf = torch.sqrt((cms2 + torch.sqrt((cms2 ** 2 - 4 * cs2 * ca[a] ** 2).clamp(min=0))) / 2)
            c = q[a].abs() + cf
            if p.if_hall:
                bm = torch.maximum(torch.maximum(f[4], f[5]), f[6])
                c = torch.maximum(c, p.ion_inertial_length / f[0] * bm / min(d))
            t = float((d[a] / c).min()) * (1.0 if a == 0 else rr)
            out = t if out is None else min(out, t)
        return out

    def fluxes(self, f, q, J):
        """spectra of the products: mass (3), momentum tensor (6), E (3), energy (3), expanding-box source"""
        rho, m, B, e = f[0], f[1:4], f[4:7], f[7]
        u, p = q[0:3], q[3]
        ptot = p + 0.5 * (B * B).sum(0)
        out = [self.fwd(m[a]) for a in range(3)]
        for a, b in PAIRS:
            out.append(self.fwd(m[b] * u[a] - B[a] * B[b] + (ptot if a == b else 0.0)))
        for a in range(3):
            b, c = (a + 1) % 3, (a + 2) % 3
            E = u[c] * B[b] - u[b] * B[c]
            if J is not None:
                E = E + self.p.ion_inertial_length / rho * (J[b] * B[c] - J[c] * B[b])
            out.append(self.fwd(E))
        ub = (u * B).sum(0)
        for a in range(3):
            out.append(self.fwd((e + ptot) * u[a] - ub * B[a]))
        if self.p.if_aeb:
            tau, g = self.radius() / self.p.Ur0, self.p.adiabatic_index
            out.append(self.fwd(-(2 * g / (g - 1) * p + 2 * B[0] ** 2 + B[1] ** 2 + B[2] ** 2 + m[0] * u[0] +
                                  2 * m[1] * u[1] + 2 * m[2] * u[2]) / tau))
        return torch.stack(out)

    def closure(self):
        """the closure's right-hand side of the momentum, B and the energy"""
        p = self.p
        f = self.real if self.fresh else self.inv(self.U)
        q = self.prim if self.fresh else self.primitives(f)
        g = torch.stack((f[0], q[0], q[1], q[2], f[4], f[5], f[6]))
        d = (p.Lx / p.nx, p.Ly / p.ny, p.Lz / p.nz)
        grad = [(torch.roll(g, -1, 3 - a) - torch.roll(g, 1, 3 - a)) / (2 * d[a]) for a in range(3)]
        X = torch.cat((g, torch.stack(grad, 1).reshape((21,) + g.shape[1:])))
        W1, b1, W2, b2, W3, b3, xm, xs, ys = self.net
        X = (X.reshape(28, -1).T - xm) / xs
        Y = ((torch.tanh(torch.tanh(X @ W1 + b1) @ W2 + b2) @ W3 + b3) * ys).T.reshape((18,) + g.shape[1:])
        trR, trM = Y[0] + Y[3] + Y[5], Y[6] + Y[9] + Y[11]
        s = -0.5 * (p.adiabatic_index - 1) * (trR + trM) + 0.5 * trM
        tau = [self.fwd(Y[c] - Y[6 + c] + (s if c in (0, 3, 5) else 0.0)) for c in range(6)]
        E, F = [self.fwd(Y[12 + a]) for a in range(3)], [self.fwd(Y[15 + a]) for a in range(3)]
        k = self.w
        R = [-1j * sum(k[b] * tau[IDX[a][b]] for b in range(3)) for a in range(3)]
        R += [-1j * (k[(a + 1) % 3] * E[(a + 2) % 3] - k[(a + 2) % 3] * E[(a + 1) % 3]) for a in range(3)]
        R.append(-1j * sum(k[b] * F[b] for b in range(3)))
        return R

    def substage(self, irk, R):
        p, hall = self.p, bool(self.p.if_hall)
        first = self.fresh and irk == 0
        f = self.real if first else self.inv(self.U)
        q = self.prim if first else self.primitives(f)
        if irk == 0:
            t = self.cfl(f, q) * p.cfl
            self.dt = self.prev if 0.98 * t <= self.prev <= 1.02 * t else t
            self.prev = self.dt
        J = torch.stack(self.curl(self.U[4:7])) if hall else None
        F = self.fluxes(f, q, self.inv(J) if hall else None)
        del f, q
        if self.phase is not None:
            fs = self.inv(self.U * self.phase)
            F = 0.5 * (F + self.phase.conj() * self.fluxes(fs, self.primitives(fs),
                                                           self.inv(J * self.phase) if hall else None))
            del fs
        k = self.k()
        dt = self.dt
        c = (8 / 15, 5 / 12, 3 / 4)[irk] * dt
        d = (0.0, -17 / 60, -5 / 12)[irk] * dt
        ts = (8 / 15, 2 / 15, 1 / 3)[irk] * dt
        r = p.radius0 / self.radius()
        wx, wy, wz = self.w
        cc, ss = (math.cos(p.corotating_angle), math.sin(p.corotating_angle)) if p.if_corotating else (1.0, 0.0)
        k2 = wx ** 2 * (cc ** 2 + (ss * r) ** 2) + wy ** 2 * (ss ** 2 + (cc * r) ** 2) + \
            2 * wx * wy * cc * ss * (1 - r * r) + (wz * r) ** 2
        if irk == 0:
            self.Fp = [None] * 8
        new = torch.empty_like(self.U)
        for v in range(8):
            if v == 0:
                fnl = -1j * sum(k[a] * F[a] for a in range(3))
            elif v < 4:
                fnl = -1j * sum(k[a] * F[3 + IDX[v - 1][a]] for a in range(3))
            elif v < 7:
                a, b = (v - 3) % 3, (v - 2) % 3
                fnl = -1j * (k[a] * F[9 + b] - k[b] * F[9 + a])
            else:
                fnl = -1j * sum(k[a] * F[12 + a] for a in range(3))
                if p.if_aeb:
                    fnl = fnl + F[15]
            if R is not None and v >= 1:
                fnl = fnl + R[v - 1]
            if p.if_aeb and v < 7:
                fnl = fnl - (2, 2, 3, 3, 2, 1, 1)[v] * self.U[v] * (p.Ur0 / self.radius())
            un = self.U[v] + c * fnl
            if irk:
                un = un + d * self.Fp[v]
            self.Fp[v] = fnl
            if v in (1, 2, 3):
                un = un / (1 + ts * p.viscosity * k2)
            elif v in (4, 5, 6):
                un = un / (1 + ts * p.resistivity * k2)
            new[v] = un * self.mask
        self.U = new

    def step(self):
        R = self.closure() if self.net else None
        for irk in range(3):
            self.substage(irk, R)
        self.fresh = False
        self.time += self.dt


def _net(vec):
    v = torch.from_numpy(vec).double().cuda()
    out, o = [], 0
    for shape in ((28, 64), (64,), (64, 64), (64,), (64, 18), (18,), (28,), (28,), (18,)):
        k = int(np.prod(shape))
        out.append(v[o:o + k].reshape(shape))
        o += k
    return out


def _train_exact(case, seed):
    X, T = _samples(case["n"], seed)
    X, T = torch.from_numpy(X).double().cuda(), torch.from_numpy(T).double().cuda()
    W = [w.clone() for w in _net(np.concatenate([init_params(seed), np.zeros(74, np.float32)]))[:6]]
    m, v = [torch.zeros_like(w) for w in W], [torch.zeros_like(w) for w in W]
    B = min(case["batch"], case["n"])
    hist = []
    for s in range(case["steps"]):
        o = (s % (case["n"] // B)) * B
        x, t = X[o:o + B], T[o:o + B]
        h1 = torch.tanh(x @ W[0] + W[1])
        h2 = torch.tanh(h1 @ W[2] + W[3])
        r = h2 @ W[4] + W[5] - t
        hist.append(float((r * r).mean()))
        dy = 2 * r / r.numel()
        d2 = (dy @ W[4].T) * (1 - h2 * h2)
        d1 = (d2 @ W[2].T) * (1 - h1 * h1)
        G = [x.T @ d1, d1.sum(0), h1.T @ d2, d2.sum(0), h2.T @ dy, dy.sum(0)]
        for i in range(6):
            m[i] = 0.9 * m[i] + 0.1 * G[i]
            v[i] = 0.999 * v[i] + 0.001 * G[i] ** 2
            W[i] = W[i] - 2e-3 * (m[i] / (1 - 0.9 ** (s + 1))) / (torch.sqrt(v[i] / (1 - 0.999 ** (s + 1))) + 1e-8)
    return torch.cat([w.reshape(-1) for w in W]).cpu(), torch.tensor(hist, dtype=torch.float64)


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _train_exact(case, seed)
    if kind == "ensemble":
        out = []
        for i, (n, di, amp) in enumerate(_boxes(case)):
            b = _Box(_params(dict(case, dealias=1), (n, n, n), di), *_state(n, n, n, seed * 1000 + i, amp))
            for _ in range(case["steps"] + 1):
                b.step()
            out.append(b.inv(b.U).cpu())
        return [torch.stack(out[i * case["boxes"]:(i + 1) * case["boxes"]]) for i in range(3)]
    p = _params(case)
    uu, pr = _state(case["nx"], case["ny"], case["nz"], seed)
    if kind == "restart":
        b = _Box(p, uu, pr)
        f = torch.stack((uu[0], pr[0], pr[1], pr[2], uu[4], uu[5], uu[6], pr[3]))
        ave = f.mean((1, 2, 3))
        var = ((f - ave[:, None, None, None]) ** 2).mean((1, 2, 3))
        ru2 = (uu[0] * (pr[:3] - ave[1:4, None, None, None]) ** 2).mean((1, 2, 3))
        en = [float(uu[7].mean()), float(0.5 * (uu[1:4] * pr[:3]).sum(0).mean()),
              float(0.5 * (uu[4:7] ** 2).sum(0).mean()), float(pr[3].mean()) / (p.adiabatic_index - 1)]
        return dict(dt=b.cfl(uu, pr), ave=ave.cpu(), var=var[1:7].cpu(), ru2=ru2.cpu(), energy=en,
                    spectrum=torch.view_as_real(b.U).reshape(-1).cpu())
    b = _Box(p, uu, pr, _net(_closure_vector(seed)) if case.get("closure") else None)
    del uu, pr
    for _ in range(case["steps"] + 1):
        b.step()
    f = b.inv(b.U)
    if kind == "filter":
        q, J, r = b.primitives(f), b.inv(torch.stack(b.curl(b.U[4:7]))), case["r"]
        rho, m, B, u = f[0], f[1:4], f[4:7], q[:3]
        out = list(f) + [m[i] * u[j] for i, j in PAIRS] + [B[i] * B[j] for i, j in PAIRS]
        for a in range(3):
            s, t = (a + 1) % 3, (a + 2) % 3
            out.append(u[t] * B[s] - u[s] * B[t] + p.ion_inertial_length / rho * (J[s] * B[t] - J[t] * B[s]))
        ub, h = (u * B).sum(0), f[7] + q[3] + 0.5 * (B * B).sum(0)
        out += [h * u[a] - ub * B[a] for a in range(3)]
        out = torch.stack(out)
        s = out.shape
        return out.reshape(26, s[1] // r, r, s[2] // r, r, s[3] // r, r).mean((2, 4, 6)).cpu()
    return dict(time=b.time, dt=b.dt, state=f.cpu())

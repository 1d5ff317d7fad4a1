"""The work this package is used for, as timed calls.

A case is one pass of a user's program through the public entry points: a
solve that advances and hands its field back (`Solver`), many solves of uneven
size (`Batch`), or the operators of class `Calc` on device tensors.  Sizes,
schemes, penalties and time steps are those of the reference's ini files
(32^3, 64^3 and 128^3 boxes, dt = 1e-7 and 5e-7, M1 = M2 = 1e4), of the tests
and of bench.py.
"""
import math

import numpy as np
import torch

import cudabubble_amd as vb

KAPPA, D = 2.0, 1.5
AREA = 3.0 / (2.0 * math.sqrt(2.0))


def listed():
    return [
        # the smallest box of the ini files, the default precision and driver: a
        # step is a few dozen short launches, so their latency is what counts
        dict(name="drift 32", kind="solve", n=32, nz=32, fp32=False, scheme=4, dt=1e-7, drift=True, steps=16),
        # the 65 x 65 x 64 boxes of the ini files (trimmed to 64^3), mixed precision
        dict(name="drift 64 mixed", kind="solve", n=64, nz=64, fp32=True, scheme=4, dt=1e-7, drift=True, steps=32),
        # the drop-in run: adaptive dt with the energy test after each attempt
        dict(name="adaptive 128", kind="solve", n=128, nz=128, fp32=False, scheme=4, dt=0.0, drift=False, steps=16),
        # a flat box that no power of two fits, the two-stage scheme, no penalties
        dict(name="etdrk2 96x48 mixed", kind="solve", n=96, nz=48, fp32=True, scheme=2, dt=5e-7, drift=False, steps=32),
        # the Forward-Euler driver with its residual and energies after each chunk
        dict(name="euler 64", kind="solve", n=64, nz=64, fp32=False, scheme=1, dt=1e-7, drift=False, steps=16),
        # the benchmark's grid in both precisions, a field kept every few dozen steps
        dict(name="drift 256 mixed", kind="solve", n=256, nz=256, fp32=True, scheme=4, dt=5e-7, drift=True, steps=48),
        dict(name="drift 256", kind="solve", n=256, nz=256, fp32=False, scheme=4, dt=5e-7, drift=True, steps=32),
        # the largest solve here: 57 million points
        dict(name="drift 384 mixed", kind="solve", n=384, nz=384, fp32=True, scheme=4, dt=5e-7, drift=True, steps=24),
        # vesicles of uneven size side by side on one GPU
        dict(name="batch mixed sizes", kind="batch", n32=8, n64=6, n96=2, n128=3, drift=True, steps=8),
        # one forward and one inverse transform: a call whose launches dominate,
        # and one that streams
        dict(name="transform 32", kind="transform", n=32, nz=32, fp32=False),
        dict(name="transform 384 fp32", kind="transform", n=384, nz=384, fp32=True),
        # a program written against class Calc: the integrals, the nonlinear
        # term and the first combines of an ETDRK4 step, operator by operator
        dict(name="stage 128", kind="stage", n=128, nz=128, dt=5e-7),
    ]


SIZES = (16, 32, 48, 64, 96, 128, 192, 256, 384)


def draw(rng):
    kind = rng.choice(("solve", "solve", "solve", "solve", "batch", "transform", "transform", "stage"))
    if kind == "batch":
        return dict(kind="batch", n32=rng.randint(1, 10), n64=rng.randint(1, 8), n96=rng.randint(0, 3),
                    n128=rng.randint(0, 4), drift=rng.random() < 0.8, steps=rng.choice((4, 6, 8, 9)))
    n = rng.choice(SIZES)
    nz = n if rng.random() < 0.6 else rng.choice([m for m in SIZES if n <= 2 * m <= 4 * n])
    if kind == "transform":
        if n == 384 and rng.random() < 0.5:
            nz = min(nz, 256)
        return dict(kind=kind, n=n, nz=nz, fp32=rng.random() < 0.5 if n * n * nz < 256 ** 3 else True)
    if n * n * nz > 256 ** 3:
        n, nz = 256, min(nz, 256)
    if kind == "stage":
        return dict(kind=kind, n=n, nz=nz, dt=rng.choice((1e-7, 2e-7, 5e-7)))
    scheme = rng.choice((4, 4, 4, 2, 1))
    if scheme == 1:     # dt = 1e-7 is past the explicit scheme's limit on finer grids
        n, nz = min(n, 96), min(n, nz, 96)
    fp32 = rng.random() < 0.5
    adaptive = scheme != 1 and not fp32 and n >= 48 and rng.random() < 0.3
    steps = rng.randint(4, 32) if n * n * nz > 96 ** 3 else rng.randint(8, 48)
    return dict(kind="solve", n=n, nz=nz, fp32=fp32, scheme=scheme,
                dt=0.0 if adaptive else 1e-7 if scheme == 1 else rng.choice((1e-7, 2e-7)) if n < 96 else 5e-7,
                drift=scheme == 4 and not adaptive and rng.random() < 0.7, steps=steps)


# ---- inputs -----------------------------------------------------------------
def _field(n, nz, seed):
    """A seeded vesicle (ellipsoid, torus or biconcave disk) as a tanh profile."""
    eps = 2.0 * 2 * math.pi / n
    kind = (vb.SHAPE_ELLIPSOID, vb.SHAPE_TORUS, vb.SHAPE_DISK)[seed % 3]
    phi, _ = vb.shape(kind, seed, n, nz, 1.0, eps)
    return eps, phi


def _params(n, nz, eps, fp32, scheme, dt, drift):
    # penalties except in the two-stage scheme's plain relaxation; targets from
    # the initial field
    m = 0.0 if scheme == 2 else 1e4
    return vb.params_default(nx=n, nz=nz, eps=eps, scheme=scheme, precision=vb.FP32_MIXED if fp32 else vb.FP64,
                             phi_lut_mode=vb.LUT_ACCURATE, M1=m, M2=m, alpha=0.0, beta=0.0, penalty_drift=int(drift),
                             time_step=dt or 1e-7, fixed_time_step=dt)


def _members(case, seed):
    """(n, dt, seed) of every solve of a batch."""
    out = []
    for n in (32, 64, 96, 128):
        for k in range(case["n%d" % n]):
            out.append((n, 1e-7, seed * 100 + len(out)))
    return out


def _calc_field(n, nz, seed):
    eps, phi = _field(n, nz, seed)
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    d = torch.from_numpy(phi).cuda()
    return eps, d + 1e-3 * torch.randn(d.shape, generator=g, device="cuda", dtype=torch.float64)


def prepare(case, seed):
    if case["kind"] == "solve":
        eps, phi = _field(case["n"], case["nz"], seed)
        p = _params(case["n"], case["nz"], eps, case["fp32"], case["scheme"], case["dt"], case["drift"])
        return dict(case=case, phi=phi, s=vb.Solver(p, phi))
    if case["kind"] == "batch":
        ps, phis = [], []
        for n, dt, sd in _members(case, seed):
            eps, phi = _field(n, n, sd)
            ps.append(_params(n, n, eps, True, vb.ETDRK4, dt, case["drift"]))
            phis.append(phi)
        return dict(case=case, b=vb.Batch(ps, phis), count=len(ps))
    n, nz = case["n"], case["nz"]
    eps, d = _calc_field(n, nz, seed)
    real = lambda dt=torch.float64: torch.empty((nz, n, n), dtype=dt, device="cuda")
    spec = lambda dt=torch.complex128: torch.empty((nz, n, n // 2 + 1), dtype=dt, device="cuda")
    if case["kind"] == "transform":
        if case["fp32"]:
            return dict(case=case, c=vb.Calc(n, nz, precision=vb.FP32_MIXED), d=d.float(), fd=spec(torch.complex64),
                        back=real(torch.float32))
        return dict(case=case, c=vb.Calc(n, nz), d=d, fd=spec(), back=real())
    names = ("lap", "f", "tmp1", "nld", "nl", "dx", "dy", "dz", "st", "ff", "d1")
    return dict(case=case, c=vb.Calc(n, nz), eps=eps, d=d, fd=spec(), fn=spec(), b=spec(), **{k: real() for k in names})


# ---- the pass ---------------------------------------------------------------
def run(state):
    case = state["case"]
    if case["kind"] == "solve":
        return _run_solve(state, case)
    if case["kind"] == "batch":
        b = state["b"]
        reps = b.step(case["steps"])
        return dict(steps=[r["evaluations"] for r in reps][:1],
                    phi=[b.get_phi(i).astype(np.float32) for i in range(state["count"])])
    c = state["c"]
    if case["kind"] == "transform":
        c.r2c(state["d"], state["fd"])
        c.c2r(state["fd"], state["back"])
        return state["fd"], state["back"]
    return _run_stage(state, c)


def _run_solve(state, case):
    s = state["s"]
    if not case["dt"]:
        s.set_phi(state["phi"])     # each adaptive run starts from its initial field
    out = {}
    if case["scheme"] == vb.EULER:
        out["residual"] = s.residual()
    r = s.step(case["steps"])
    out.update(steps=r["steps"], evaluations=r["evaluations"], rejections=r["rejections"], status=r["status"])
    out.update(s.state())
    if not case["fp32"]:
        out["E"], out["V"], out["A"], out["Eb"] = s.query()
    # a mixed-precision run keeps its fields in single precision
    phi = s.get_phi()
    out["phi"] = phi.astype(np.float32) if case["fp32"] else phi
    return out


def _run_stage(t, c):
    eps, dt = t["eps"], t["case"]["dt"]
    c.r2c(t["d"], t["fd"])
    # volume, surface and bending energy of the field (phasefield.cpp:283-325)
    c.fftgradient(t["fd"], t["dx"], t["dy"], t["dz"])
    c.s_term(t["st"], t["d"], t["dx"], t["dy"], t["dz"], eps)
    vol = c.intf(t["d"], 1.0, 0.5)
    area = c.intf(t["st"], 0.0, AREA)
    c.lap_spec(t["fd"], t["lap"])
    c.f(t["f"], t["lap"], t["d"], eps)
    c.multi(t["f"], t["f"], t["ff"])
    bend = c.intf(t["ff"], 0.0, 1.0 / (2.0 * eps))
    # the nonlinear term with fixed multipliers (belastic.cpp:473-488)
    c.nld(t["nld"], t["d"], t["f"], t["tmp1"], eps)
    c.nld2(t["nl"], t["f"], t["nld"], 2.5, -1.5, 1.0)
    c.r2c(t["nl"], t["fn"])
    # the first combines (belastic.cpp:519-535)
    c.etd41(t["d1"], t["fd"], t["fn"], eps, dt)
    c.etd42(t["b"], t["fd"], t["fn"], eps, dt)
    return dict(V=vol, A=area, Eb=bend, **{k: t[k] for k in ("fd", "dx", "dy", "dz", "st", "lap", "f", "ff", "tmp1",
                                                             "nld", "nl", "fn", "d1", "b")})


# ---- what a pass cannot do without --------------------------------------------
def _evaluations(case):
    per = 2 if case["drift"] else 1
    return case["steps"] * per


def _solve_work(n, nz, fp32, scheme, evals):
    # an evaluation reads the FP64 state spectrum and writes the new one; each of
    # its stages takes the stage field's spectrum in and gives the nonlinear
    # term's out in the work precision, with four real transforms and some
    # thirty operations a point between
    pts, modes = n * n * nz, (n // 2 + 1) * n * nz
    cs, stages = (8 if fp32 else 16), max(1, scheme)
    bytes_ = evals * (2 * 16 * modes + stages * 2 * cs * modes) + 8 * pts
    flops = evals * stages * (4 * 2.5 * pts * math.log2(pts) + 30 * pts)
    return bytes_, flops


def work(case):
    if case["kind"] == "solve":
        b, f = _solve_work(case["n"], case["nz"], case["fp32"], case["scheme"], _evaluations(case))
        return {"bytes": b, "flops": f}
    if case["kind"] == "batch":
        w = [_solve_work(n, n, True, 4, _evaluations(case)) for n, _, _ in _members(case, 0)]
        return {"bytes": sum(x[0] for x in w), "flops": sum(x[1] for x in w)}
    n, nz = case["n"], case["nz"]
    pts, modes = n * n * nz, (n // 2 + 1) * n * nz
    one = 2.5 * pts * math.log2(pts)
    if case["kind"] == "transform":
        r, c = (4, 8) if case["fp32"] else (8, 16)
        return {"bytes": 2 * (r * pts + c * modes), "flops": 2 * one}
    # operator by operator: each reads its inputs and writes its output once
    transforms = 2 + 3 + 1 + 2 + 1
    bytes_ = 8 * pts * (2 + 3 + 1 + 2 + 1 + 5 + 1 + 1 + 3 + 2 + 1 + 2 + 5 + 3) + 16 * modes * (2 + 1 + 1 + 2 + 3)
    return {"bytes": bytes_, "flops": transforms * one + 60 * pts}


# ---- the same in 64 bits, with torch's transforms ------------------------------
def _grid(n, nz):
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    fold = torch.minimum(k, n - k)
    z = torch.arange(nz, device="cuda", dtype=torch.float64)
    fz = torch.minimum(z, nz - z)
    kx = torch.arange(n // 2 + 1, device="cuda", dtype=torch.float64)
    k2 = fz[:, None, None] ** 2 + fold[None, :, None] ** 2 + kx[None, None, :] ** 2
    # signed wave numbers with each component's Nyquist plane zeroed
    sg = torch.where(k < n - k, k, k - n)
    sg[n // 2] = 0
    sz = torch.where(z < nz - z, z, z - nz)
    sz[nz // 2] = 0
    sx = kx.clone()
    sx[n // 2] = 0
    return k2, (sx[None, None, :], sg[None, :, None], sz[:, None, None])


def _fwd(u):
    return torch.fft.rfftn(u) / u.numel()


def _inv(s, shape):
    return torch.fft.irfftn(s, s=shape) * (shape[0] * shape[1] * shape[2])


def _phi_functions(z):
    """(e^z - 1 - z) / z^2 and the three ETDRK4 brackets over z^3, in 64 bits."""
    z = z.cpu().numpy().astype(np.longdouble)
    small = np.abs(z) < 1
    zs = np.where(small, z, 0.5)
    t, u = np.full(z.shape, np.longdouble(1) / 6), np.full(z.shape, np.longdouble(0.5))
    s = [np.zeros(z.shape, np.longdouble) for _ in range(4)]
    for k in range(2, 40):
        s[3] += u
        u = u * zs / (k + 1)
        if k >= 3:
            s[0] += (k - 2) ** 2 * t
            s[1] += (k - 2) * t
            s[2] += (4 - k) * t
            t = t * zs / (k + 1)
    zl = np.where(small, 1.0, z)
    e = np.exp(zl)
    c = [(-4 - zl + e * (4 - 3 * zl + zl * zl)) / zl ** 3, (2 + zl + e * (zl - 2)) / zl ** 3,
         (-4 - 3 * zl - zl * zl + e * (4 - zl)) / zl ** 3, (e - 1 - zl) / (zl * zl)]
    return [torch.from_numpy(np.where(small, a, b).astype(np.float64)).cuda() for a, b in zip(s, c)]


class _Model:
    """The solver's equations on full fields."""

    def __init__(self, n, nz, eps, scheme, m):
        self.shape, self.eps, self.scheme, self.m = (nz, n, n), eps, scheme, m
        self.k2, (sx, sy, sz) = _grid(n, nz)
        w = torch.full((n // 2 + 1,), 2.0, device="cuda", dtype=torch.float64)
        w[0] = w[-1] = 1.0
        self.gw = w * (sx ** 2 + sy ** 2 + sz ** 2)
        self.H = -eps * self.k2 ** 2 - KAPPA * self.k2 / eps + D * (-self.k2 - KAPPA / eps ** 2) / eps
        self.L3 = (2 * math.pi) ** 3
        self.tabs = {}

    def table(self, h):
        if h not in self.tabs:
            # coefficients depend on |k|^2 alone
            m, back = torch.unique(self.k2, return_inverse=True)
            H = -self.eps * m ** 2 - KAPPA * m / self.eps + D * (-m - KAPPA / self.eps ** 2) / self.eps
            f1, f2, f3, p2 = _phi_functions(h * H)
            hh = h if self.scheme == 2 else h / 2
            self.tabs = {h: [x[back] for x in (torch.exp(hh * H), torch.expm1(hh * H) / H, torch.exp(h * H), h * f1,
                                               2 * h * f2, h * f3, h * p2)]}
        return self.tabs[h]

    def integrals(self, vh):
        v = _inv(vh, self.shape)
        lap = _inv(-self.k2 * vh, self.shape)
        w = v * v - 1
        f = -self.eps * lap + w * v / self.eps
        V = ((vh[0, 0, 0].real + 1) * 0.5 * self.L3).item()
        g2 = (self.gw * vh.abs() ** 2).sum().item()
        A = (0.5 * self.eps * g2 + 0.25 / self.eps * (w * w).mean().item()) * AREA * self.L3
        Eb = (f * f).mean().item() / (2 * self.eps) * self.L3
        return v, f, V, A, Eb

    def energy(self, V, A, Eb, tg):
        return Eb + 0.5 * self.m * (V - tg[0]) ** 2 + 0.5 * self.m * (A - tg[1]) ** 2

    def nonlinear(self, vh, tg):
        v, f, V, A, _ = self.integrals(vh)
        t1 = v * (v * v - 1 - KAPPA)
        s = D * t1 / self.eps ** 3 + (3 * v * v - D - 1) * f / self.eps ** 2
        N = -self.m * (A - tg[1]) * AREA * _fwd(f) - _fwd(s) - self.k2 * _fwd(t1) / self.eps
        N[0, 0, 0] -= 0.5 * self.m * (V - tg[0])
        return N

    def evaluate(self, u, h, tg):
        e1, q, e2, fa, fb, fc, c2 = self.table(h)
        N = self.nonlinear(u, tg)
        if self.scheme == 2:
            a = e1 * u + q * N
            return a + c2 * (self.nonlinear(a, tg) - N)
        a = e1 * u + q * N
        Na = self.nonlinear(a, tg)
        b = e1 * u + q * Na
        Nb = self.nonlinear(b, tg)
        c = e1 * a + q * (2 * Nb - N)
        # the reference's combine takes N^a in the first bracket (Calc.cu:559)
        return e2 * u + Na * fa + (Na + Nb) * fb + self.nonlinear(c, tg) * fc

    def euler_rhs(self, u, tg):
        v, f, V, A, _ = self.integrals(u)
        lf = _inv(-self.k2 * _fwd(f), self.shape)
        g0 = -lf + (3 * v * v - 1) * f / self.eps ** 2
        return 0.5 * self.m * (V - tg[0]) + self.m * (A - tg[1]) * f + g0


def _exact_solve(n, nz, eps, phi, scheme, dt, drift, steps):
    M = _Model(n, nz, eps, scheme, 0.0 if scheme == 2 else 1e4)
    u = _fwd(torch.from_numpy(phi).cuda())
    _, _, V, A, Eb = M.integrals(u)
    tg0 = (V, A)
    tg, h, t = [V, A], dt or 1e-7, 0.0
    out = dict(steps=steps, rejections=0, status=0)
    evals = 0
    if scheme == 1:
        out["residual"] = (M.euler_rhs(u, tg) ** 2).mean().item() * M.L3
    E = M.energy(V, A, Eb, tg)
    for k in range(steps):
        if scheme == 1:
            u = _fwd(_inv(u, M.shape) - h * M.euler_rhs(u, tg))
            evals += 1
        elif not dt:
            if k % 4 == 0:
                h = 2 * h if h * 1.4 < 1e-3 else 1e-3
            while True:
                new = M.evaluate(u, h, tg)
                evals += 1
                En = M.energy(*M.integrals(new)[2:], tg)
                if En <= E:
                    break
                h /= 2
                out["rejections"] += 1
            u, E = new, En
        elif drift:
            for _ in range(2):
                new = M.evaluate(u, h, tg)
                evals += 1
                _, _, V, A, _ = M.integrals(new)
                tg = [tg[0] - (V - tg0[0]), tg[1] - (A - tg0[1])]
            u = new
        else:
            u = M.evaluate(u, h, tg)
            evals += 1
        t += h
    _, _, V, A, Eb = M.integrals(u)
    out.update(evaluations=evals, alpha=tg[0], beta=tg[1], time_step=h, time_current=t, E=M.energy(V, A, Eb, tg), V=V,
               A=A, Eb=Eb, phi=_inv(u, M.shape).cpu().numpy())
    return out


def exact(case, seed):
    if case["kind"] == "solve":
        n, nz = case["n"], case["nz"]
        if n * n * nz * _evaluations(case) > 170 * 256 ** 3:
            return None     # over 20 seconds
        eps, phi = _field(n, nz, seed)
        out = _exact_solve(n, nz, eps, phi, case["scheme"], case["dt"], case["drift"], case["steps"])
        if case["fp32"]:
            for k in ("E", "V", "A", "Eb"):
                out.pop(k)
        return out
    if case["kind"] == "batch":
        phis = []
        for n, dt, sd in _members(case, seed):
            eps, phi = _field(n, n, sd)
            phis.append(_exact_solve(n, n, eps, phi, 4, dt, case["drift"], case["steps"])["phi"])
        return dict(steps=[_evaluations(case)], phi=phis)
    n, nz = case["n"], case["nz"]
    eps, d = _calc_field(n, nz, seed)
    if case["kind"] == "transform":
        d = d.float().double() if case["fp32"] else d
        return _fwd(d), d
    M = _Model(n, nz, eps, 4, 1e4)
    lap = lambda s: _inv(-M.k2 * s, M.shape)
    fd = _fwd(d)
    _, k = _grid(n, nz)
    dx, dy, dz = (_inv(1j * kk * fd, M.shape) for kk in k)
    st = 0.5 * eps * (dx * dx + dy * dy + dz * dz) + 0.25 / eps * (d * d - 1) ** 2
    lp = lap(fd)
    f = -lp * eps + (d * d - 1) * d / eps
    t1 = d * (d * d - 1 - KAPPA)
    nld = -lap(_fwd(t1)) / eps + D * t1 / eps ** 3 + (3 * d * d - D - 1) * f / eps ** 2
    nl = -2.5 * 0.5 + 1.5 * f * AREA - nld
    fn = _fwd(nl)
    e1, q = M.table(case["dt"])[:2]
    b = e1 * fd + q * fn
    return dict(V=(d.mean().item() + 1) * 0.5 * M.L3, A=st.mean().item() * AREA * M.L3,
                Eb=(f * f).mean().item() / (2 * eps) * M.L3, fd=fd, dx=dx, dy=dy, dz=dz, st=st, lap=lp, f=f, ff=f * f,
                tmp1=t1, nld=nld, nl=nl, fn=fn, d1=_inv(b, M.shape), b=b)

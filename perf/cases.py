"""Performance cases: what a modelling or inversion program has this framework do.

Every case is a whole pass through the public binding (dnhip): a shot of a
shot loop (source set, forward run, seismograms read), the gradient of one
shot in an inversion (model set, forward run with snapshots, residuals,
adjoint run, assembly, gradients read), or a batch of uneven shots through
the multi-shot engine.  Grids, time steps and lengths follow the tests, the
example inputs and the benchmark of this repository; runs of thousands of
steps are shortened where a pass would take seconds (a step costs the same).

exact() integrates the same difference equations in 64 bits with torch.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "denise-black-edition_amd"))
import dnhip  # noqa: E402

DEV = "cuda" if torch.cuda.is_available() else "cpu"
# physics of dn_params: P/SV, acoustic, VTI, SH
PSV, AC, VTI, SH = 1, 2, 3, 5
FL = [10.0, 40.0, 2.5]  # relaxation frequencies of the viscoelastic cases
Q = 50.0
# Holberg operators of 0.1 % group-velocity error, FDORDER 2..12
HOLBERG = {
    2: [1.0010],
    4: [1.1382, -0.046414],
    6: [1.1965, -0.078804, 0.0081781],
    8: [1.2257, -0.099537, 0.018063, -0.0026274],
    10: [1.2415, -0.11231, 0.026191, -0.0064682, 0.001191],
    12: [1.2508, -0.12034, 0.032131, -0.010142, 0.0029857, -0.00066667],
}


def _case(name, kind="shot", physics=PSV, nx=0, ny=0, nt=0, dh=10.0, order=8, L=0, free=1, fw=20, dtinv=2,
          water=0, every=2, tune=0, shots=1):
    return dict(name=name, kind=kind, physics=physics, nx=nx, ny=ny, nt=nt, dh=dh, order=order, L=L, free=free,
                fw=fw, dtinv=dtinv, water=water, every=every, tune=tune, shots=shots)


def listed():
    return [
        # the smoke shot: the smallest calls, launches and latency
        _case("tiny_120x80", nx=120, ny=80, nt=300, fw=10),
        # the plain CPU benchmark's grid: a desk-size survey shot
        _case("shot_400x200", nx=400, ny=200, nt=2000),
        # a shot and an inversion gradient of the shipped Marmousi example
        # (marine: water on top)
        _case("marmousi_shot", nx=500, ny=174, nt=3000, dh=20.0, fw=10, water=22, every=1),
        _case("marmousi_gradient", kind="gradient", nx=500, ny=174, nt=3000, dh=20.0, fw=10, dtinv=3, water=22,
              every=1),
        # the elastic gradient benchmark: snapshots every second step
        _case("gradient_2000x600", kind="gradient", nx=2000, ny=600, nt=1000, dtinv=2),
        # the roofline shots, shapes tuned once for the model as the benchmark does
        _case("elastic_4000x1200", nx=4000, ny=1200, nt=600, dh=5.0, every=5, tune=10),
        _case("visco_4000x1200", nx=4000, ny=1200, nt=400, dh=5.0, L=2, every=5, tune=10),
        # odd sizes, the longest operator, absorbing on all sides, one mechanism
        _case("visco_odd_1237x431", nx=1237, ny=431, nt=800, order=12, L=1, free=0),
        # marine streamer modelling: pressure only
        _case("acoustic_1501x601", physics=AC, nx=1501, ny=601, nt=1200, every=1),
        # shear-wave (engineering) line: low order
        _case("sh_811x303", physics=SH, nx=811, ny=303, nt=1500, dh=1.0, order=4, every=1),
        # anisotropic modelling
        _case("vti_1800x700", physics=VTI, nx=1800, ny=700, nt=700),
        # independent uneven shots through the multi-shot engine
        _case("batch_12", kind="batch", nx=3000, ny=800, nt=800, shots=12),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["shot", "shot", "shot", "gradient", "batch"])
    physics = rng.choice([PSV, PSV, AC, VTI, SH]) if kind == "shot" else PSV
    L = rng.choice([0, 0, 1, 2, 3]) if physics == PSV and kind == "shot" else 0
    c = _case("", kind=kind, physics=physics, L=L, order=rng.choice([2, 4, 6, 8, 8, 8, 10, 12]),
              free=rng.choice([0, 1, 1]), fw=rng.choice([10, 20]), dh=rng.choice([2.0, 5.0, 10.0, 20.0]),
              dtinv=rng.choice([1, 2, 3]), every=rng.choice([1, 2, 5]))
    del c["name"]
    if kind == "batch":
        c.update(nx=log(500, 3000), ny=log(200, 800), nt=log(300, 800), shots=rng.randint(2, 12), free=1, fw=20)
        return c
    c["nx"], c["ny"] = log(110, 4000), log(80, 1200)
    if kind == "gradient":
        c["nx"], c["ny"] = min(c["nx"], log(110, 2000)), min(c["ny"], 600)
    # no more cell-updates than the largest listed case of its kind
    most = 1.0e9 if kind == "gradient" else 1.9e9 / (1 + L)
    c["nt"] = max(100, min(log(200, 3000), int(most / (c["nx"] * c["ny"]))))
    if kind == "shot" and c["nx"] * c["ny"] > 1000000:
        c["tune"] = rng.choice([0, 10])
    return c


# ---------------------------------------------------------------- inputs
def _noise(rng, nx, ny, scale=16):
    """Smooth random field of maximum 1: noise on a coarse grid, interpolated."""
    cx, cy = -(-nx // scale) + 2, -(-ny // scale) + 2
    z = torch.from_numpy(rng.standard_normal((1, 1, cx, cy)).astype(np.float32)).to(DEV)
    f = torch.nn.functional.interpolate(z, size=(nx, ny), mode="bilinear", align_corners=True)[0, 0]
    return f / f.abs().max()


def _shot(case, seed, nx=None, ny=None, nt=None, order=None):
    """One shot's inputs as a program holds them: parameters and host arrays.

    vp from 1500 to 4000 m/s with depth and a smooth random +-5 %,
    vs = vp/sqrt(3) (0 in the water), rho = 310 vp^0.25; one Ricker source
    near the surface, a line of receivers."""
    rng = np.random.default_rng(seed)
    nx, ny, nt, order = nx or case["nx"], ny or case["ny"], nt or case["nt"], order or case["order"]
    phys, L, dh = case["physics"], case["L"], case["dh"]

    def model():
        v0 = torch.linspace(1500.0, 4000.0, ny, device=DEV)[None, :]
        vp = v0 * (1.0 + 0.05 * _noise(rng, nx, ny))
        vs, rho = vp / math.sqrt(3.0), 310.0 * vp ** 0.25
        w = case["water"]
        if w:
            vp[:, :w], vs[:, :w], rho[:, :w] = 1500.0, 0.0, 1000.0
        if phys == VTI:
            f = 1.0 + 0.5 * _noise(rng, nx, ny)
            c33, c44 = rho * vp ** 2, rho * vs ** 2
            c11 = c33 * (1.0 + 0.4 * f)
            c13 = torch.sqrt(0.2 * f * c33 * (c33 - c44) + (c33 - c44) ** 2) - c44
            return [a.cpu().numpy() for a in (rho, c11, c13, c33, c44)]
        return [a.cpu().numpy() for a in (vp, vs, rho)]

    m = model()
    true = model() if case["kind"] == "gradient" else None
    vmax = 4200.0 * (1.27 if phys == VTI else 1.0 + 0.04 * L)
    if phys == SH:
        vmax /= math.sqrt(3.0)
    dt = float(np.float32(0.85 * dh / (math.sqrt(2.0) * sum(abs(h) for h in HOLBERG[order]) * vmax)))
    fc = 800.0 / (10.0 * dh) * (1.7 if phys == AC else 1.0)
    p = dnhip.Params(nx=nx, ny=ny, nt=nt, dh=dh, dt=dt, fdorder=order, maxrelerror=1, fw=case["fw"],
                     free_surf=case["free"], L=L, seismo=2 if phys == AC else 1, mode=int(case["kind"] == "gradient"),
                     dtinv=case["dtinv"], ts=float(np.float32(1.0 / fc)), damping=1500.0, fpml=fc, fl=FL[:L],
                     physics=phys)
    z = 2 if case["free"] else case["fw"] + 3
    src = np.zeros((8, 1), np.float32)
    src[:, 0] = [nx // 2 + rng.integers(-nx // 8, nx // 8), z, 1, 0.0, fc, 1.0, 0.0, 1]
    t = (np.arange(1, nt + 1) * dt - 1.5 / fc) * (math.pi / (1.5 / fc))
    sig = ((1.0 - 4.0 * t * t) * np.exp(-2.0 * t * t)).astype(np.float32)[None, :]
    ix = np.arange(3, nx - 2, case["every"])
    rec = np.stack([ix, np.full_like(ix, case["water"] + z)]).astype(np.int32)
    tau = [np.full((nx, ny), 2.0 / Q, np.float32)] * 2 if L else [None, None]
    return dict(p=p, model=m, tau=tau, true=true, src=src, sig=sig, rec=rec)


def _set_model(ctx, s, model):
    if s["p"].physics == VTI:
        ctx.set_model_aniso(*model)
    else:
        ctx.set_model(*model, *s["tau"])


def _context(s, model, mode=None):
    p = s["p"]
    if mode is not None:
        p = dnhip.Params(**{**p.__dict__, "mode": mode})
    ctx = dnhip.Context(p)
    _set_model(ctx, s, model)
    ctx.set_sources(s["src"], s["sig"])
    ctx.set_receivers(s["rec"])
    return ctx


def _batch(case, seed):
    """Uneven shots: grid sizes and lengths uniform up to the case's."""
    rng = np.random.default_rng(1000 + case["nx"] * 7 + case["ny"] * 3 + case["shots"])  # sizes belong to the case
    out = []
    for k in range(case["shots"]):
        nx, ny = int(rng.integers(case["nx"] // 6, case["nx"] + 1)), int(rng.integers(case["ny"] // 4, case["ny"] + 1))
        nt, order = int(rng.integers(case["nt"] * 3 // 8, case["nt"] + 1)), int(rng.choice([4, 8]))
        out.append(_shot(case, seed * 64 + k, max(nx, 100), max(ny, 80), nt, order))
    return out


def prepare(case, seed):
    if case["kind"] == "batch":
        shots = _batch(case, seed)
        return dict(kind="batch", engine=dnhip.Engine(0), ctx=[_context(s, s["model"]) for s in shots])
    s = _shot(case, seed)
    if case["kind"] == "gradient":  # the recorded data of the true model
        with _context(s, s["true"], mode=0) as t:
            t.forward()
            s["obs"] = t.seismogram(0), t.seismogram(1)
    s.update(kind=case["kind"], ctx=_context(s, s["model"]))
    if case["tune"]:
        s["ctx"].autotune(case["tune"])
    return s


def run(state):
    if state["kind"] == "batch":
        for c in state["ctx"]:
            state["engine"].attach(c)
        state["engine"].run()
        out = [(c.seismogram(0), c.seismogram(1)) for c in state["ctx"]]
        for c in state["ctx"]:
            state["engine"].forget(c)
        return out
    ctx = state["ctx"]
    if state["kind"] == "gradient":
        _set_model(ctx, state, state["model"])
        ctx.forward()
        l2 = ctx.residuals(state["obs"][0], state["obs"][1])
        ctx.adjoint()
        ctx.assemble()
        return dict(l2=l2, vp=ctx.gradient(3), vs=ctx.gradient(4), rho=ctx.gradient(5))
    ctx.set_sources(state["src"], state["sig"])
    ctx.forward()
    physics = state["p"].physics
    return [ctx.seismogram(k) for k in ((2,) if physics == AC else (1,) if physics == SH else (0, 1))]


def _work(physics, L, order, nx, ny, nt, nrec, gradient=0, dtinv=1):
    """Of each time step: every coefficient plane and every wavefield read
    once, every wavefield written once; the sampled traces written once."""
    coef = {PSV: 5, AC: 3, VTI: 6, SH: 3}[physics]
    state = {PSV: 5 + 3 * L, AC: 3, VTI: 5, SH: 3}[physics]
    nder = 4 if physics in (AC, SH) else 8
    cells, ncomp = nx * ny * nt, 1 if physics in (AC, SH) else 2
    nbytes = 4 * cells * (coef + 2 * state) + 4 * nrec * nt * ncomp
    flops = cells * (nder * (3 * (order // 2) - 1) + 8 * nder // 2 + 30 * L)
    if gradient:  # snapshots out and in, vxp1 / vyp1, sums, moduli
        nbytes = 2 * nbytes + 4 * cells * 4 + 4 * cells // dtinv * (5 + 5 + 6 + 2)
        flops = 2 * flops + 4 * cells + 25 * cells // dtinv
    return nbytes, flops


def work(case):
    if case["kind"] == "batch":
        w = [_work(PSV, 0, s["p"].fdorder, s["p"].nx, s["p"].ny, s["p"].nt, s["rec"].shape[1]) for s in _sizes(case)]
        return {"bytes": sum(b for b, _ in w), "flops": sum(f for _, f in w)}
    nrec = len(range(3, case["nx"] - 2, case["every"]))
    b, f = _work(case["physics"], case["L"], case["order"], case["nx"], case["ny"], case["nt"], nrec,
                 case["kind"] == "gradient", case["dtinv"])
    return {"bytes": b, "flops": f}


def _sizes(case):
    return _batch(case, 1)


# ---------------------------------------------------------------- 64 bits
H = 8  # zero border around every field


class _Grid:
    def __init__(self, p):
        self.p, self.hc = p, [float(np.float32(h)) for h in HOLBERG[p.fdorder]]
        self.nx, self.ny, self.F = p.nx, p.ny, len(self.hc)
        self.dt, self.dh = float(np.float32(p.dt)), float(np.float32(p.dh))
        self.pml = {k: self._profile(k) for k in ("x", "xh", "y", "yh")}
        self.psi = {}

    def _profile(self, k):
        """CPML coefficients (b, a, 1/K) of the near and far band of an axis."""
        p, fw = self.p, self.p.fw
        n, half = (p.nx if k[0] == "x" else p.ny), (0.5 if k.endswith("h") else 0.0)
        thick, npow = fw * self.dh, p.npower
        d0 = -(npow + 1) * p.damping * math.log(np.float32(0.001)) / (2.0 * thick)
        amax = 2.0 * math.pi * (p.fpml / 2.0)
        out = []
        for cells in (range(1, fw + 1), range(n - fw + 1, n + 1)):
            b, a, ik = [], [], []
            for i in cells:
                x = self.dh * (i - 1 + half)
                s = thick - x if i <= fw and cells[0] == 1 else x - ((n - 1) * self.dh - thick)
                d, K, al = 0.0, 1.0, 0.0
                if s >= -1e-9:
                    s = max(s, 0.0) / thick
                    d, K = d0 * s ** npow, 1.0 + (p.k_max_pml - 1.0) * s ** npow
                    al = amax * (1.0 - s) + (0.1 * amax if p.physics == SH else 0.0)
                if k[0] == "x":
                    al = max(al, 0.0)
                bb = math.exp(-(d / K + al) * self.dt)
                b.append(bb)
                a.append(d * (bb - 1.0) / (K * (d + K * al)) if d >= 1.0 else 0.0)
                ik.append(1.0 / K)
            v = [torch.tensor(q, dtype=torch.float64, device=DEV) for q in (b, a, ik)]
            out.append([q[None, :] if k[0] == "x" else q[:, None] for q in v])
        return out

    def field(self):
        return torch.zeros(self.ny + 2 * H, self.nx + 2 * H, dtype=torch.float64, device=DEV)

    def put(self, a):
        """x-major host array -> [row, column] tensor."""
        return torch.from_numpy(np.ascontiguousarray(a.T)).to(DEV).double()

    def inner(self, f, dy=0, dx=0):
        return f[H + dy:H + dy + self.ny, H + dx:H + dx + self.nx]

    def diff(self, f, axis, fwd):
        """Staggered difference of the inner cells, forward or backward half."""
        out = None
        for m, h in enumerate(self.hc, 1):
            hi, lo = (m, 1 - m) if fwd else (m - 1, -m)
            a = self.inner(f, 0, hi) if axis == "x" else self.inner(f, hi, 0)
            b = self.inner(f, 0, lo) if axis == "x" else self.inner(f, lo, 0)
            out = (a - b) * h if out is None else out.add_(a - b, alpha=h)
        return out

    def damp(self, name, d, k):
        """Applies the CPML of axis profile k to the derivative d, in place."""
        fw = self.p.fw
        for side in (0, 1):
            if k[0] == "y" and side == 0 and self.p.free_surf:
                continue
            if k[0] == "x":
                v = d[:, :fw] if side == 0 else d[:, d.shape[1] - fw:]
            else:
                v = d[:fw] if side == 0 else d[self.ny - fw:]
            b, a, ik = self.pml[k][side]
            psi = self.psi.get((name, side))
            psi = self.psi[name, side] = v * a if psi is None else psi.mul_(b).add_(v * a)
            v.mul_(ik).add_(psi)
        return d


def _ring(f):
    """Cell values with the periodic ghost row and column after the last."""
    f = torch.cat([f, f[:1]], 0)
    return torch.cat([f, f[:, :1]], 1)


def _amp(sig, n, dt):
    """Central difference of the source signal at step n (0-based)."""
    if n == 0:
        return sig[1] / dt
    return ((sig[n + 1] if n + 1 < len(sig) else 0.0) - sig[n - 1]) / dt


def _psv64(s, model, adj=None, fwd=None, mode=0):
    """P/SV, acoustic, VTI and SH runs in 64 bits.  mode 1: snapshots kept
    and returned; adj: the adjoint run with these vx, vy sources, correlated
    with the snapshots fwd."""
    p = s["p"]
    g = _Grid(p)
    phys, L, dt, dh, dtinv = p.physics, p.L, g.dt, g.dh, p.dtinv
    ixr = torch.from_numpy(s["rec"][0].astype(np.int64) - 1 + H).to(DEV)
    iyr = torch.from_numpy(s["rec"][1].astype(np.int64) - 1 + H).to(DEV)
    ixs, iys = int(s["src"][0, 0]) - 1 + H, int(s["src"][1, 0]) - 1 + H
    sig = s["sig"][0].astype(np.float64)
    m = [g.put(a) for a in model]
    rho = m[0] if phys == VTI else m[2]
    R = _ring(rho)
    if phys == SH:
        ri = 1.0 / rho
    else:
        ri, rj = 2.0 / (R[:-1, :-1] + R[:-1, 1:]), 2.0 / (R[:-1, :-1] + R[1:, :-1])

    def harm(x, four=True):
        x = _ring(x)
        return 4.0 / (1 / x[:-1, :-1] + 1 / x[:-1, 1:] + 1 / x[1:, :-1] + 1 / x[1:, 1:])  # 1/0 -> inf -> 0

    if phys == PSV:
        mu, pi = rho * m[1] ** 2, rho * m[0] ** 2
        muh, f, gm = harm(mu), mu, pi - 2.0 * mu
        if L:
            tau = 2.0 / Q
            tau = float(np.float32(tau))
            ts = [1.0 / (2.0 * math.pi * v) for v in FL[:L]]
            eta = [dt / v for v in ts]

            def relax(w):
                return 1.0 / (1.0 + sum((w * v) ** 2 / (1.0 + (w * v) ** 2) for v in ts) * tau)

            r0 = relax(2.0 * math.pi * FL[0])
            muv, piv, muhv = mu * r0, pi * r0, muh * r0
            fip, f, gm = muhv * dt * (1 + L * tau), muv * dt * (1 + L * tau), piv * dt * (1 + L * tau)
            bq, cq = [1.0 / (1.0 + 0.5 * e) for e in eta], [1.0 - 0.5 * e for e in eta]
            mr, mp, mq = ([torch.zeros_like(mu) for _ in range(L)] for _ in range(3))
            rf = relax(2.0 * math.pi / float(np.float32(p.ts)))
            fjm, gfs = 2.0 * mu[0] * rf * (1 + L * tau), pi[0] * rf * (1 + L * tau)
            dme = 2.0 * mu[0] * rf * tau - pi[0] * rf * tau
    elif phys == AC:
        gm = rho * m[0] ** 2
    elif phys == VTI:
        c11, c13, c33, c44 = m[1], m[2], m[3], harm(m[4])
    else:
        x = _ring(rho * m[1] ** 2)
        uip, ujp = 2.0 / (1 / x[:-1, :-1] + 1 / x[:-1, 1:]), 2.0 / (1 / x[:-1, :-1] + 1 / x[1:, :-1])
    vx, vy, sxx, syy, sxy = (g.field() for _ in range(5))
    I, mirror = g.inner, p.free_surf and phys in (PSV, AC)
    nr, nt = len(ixr), p.nt
    sec = torch.zeros(2, nt, nr, dtype=torch.float64, device=DEV)
    keep = []
    if adj is not None:
        wc, wcu, wcr, p1x, p1y = (torch.zeros(g.ny, g.nx, dtype=torch.float64, device=DEV) for _ in range(5))
        mu0, lam0 = rho * m[1] ** 2, rho * (m[0] ** 2 - 2.0 * m[1] ** 2)
        wet, imm, ilm = mu0 > 0, 1.0 / mu0 ** 2, 0.25 / (lam0 + mu0) ** 2
    for n in range(nt):
        if phys == SH:
            d = g.damp("a", g.diff(sxx, "x", False), "x") + g.damp("b", g.diff(syy, "y", False), "y")
            I(vx).add_(ri * d, alpha=dt / dh)
            vx[iys, ixs] += sig[n]
            sec[0, n] = vx[iyr, ixr]
            I(sxx).add_(uip * g.damp("c", g.diff(vx, "x", True) * (dt / dh), "xh"))
            I(syy).add_(ujp * g.damp("d", g.diff(vx, "y", True) * (dt / dh), "yh"))
            continue
        if phys == AC:
            if mirror:
                for k in range(1, g.F + 1):
                    sxx[H - k] = -sxx[H + k]
            fx = g.damp("a", g.diff(sxx, "x", True), "xh")
            fy = g.damp("b", g.diff(sxx, "y", True), "yh")
            # the ghost rows belong to the velocity update alone
            I(vx).add_(ri * fx, alpha=dt / dh)
            I(vy).add_(rj * fy, alpha=dt / dh)
            d = g.damp("c", g.diff(vx, "x", False) * (dt / dh), "x") + \
                g.damp("d", g.diff(vy, "y", False) * (dt / dh), "y")
            I(sxx).add_(gm * d)
            sxx[iys, ixs] += _amp(sig, n, dt)
            if mirror:
                sxx[H] = 0.0
            sec[0, n] = sxx[iyr, ixr]
            continue
        if mirror:
            for k in range(1, g.F + 1):
                syy[H - k] = -syy[H + k]
                sxy[H - k] = -sxy[H + k - 1]
        fx = g.damp("a", g.diff(sxx, "x", True), "xh") + g.damp("b", g.diff(sxy, "y", False), "y")
        fy = g.damp("c", g.diff(sxy, "x", False), "x") + g.damp("d", g.diff(syy, "y", True), "yh")
        ax, ay = ri * fx, rj * fy
        store = mode == 1 and n % dtinv == 0
        snap = [ax / dh, ay / dh] if store else None
        if adj is not None:
            k = (nt - 1 - n) // dtinv if (nt - 1 - n) % dtinv == 0 else -1
            p1x.add_(I(vx), alpha=dt)
            p1y.add_(I(vy), alpha=dt)
            if k >= 0:
                wcr.addcmul_(p1x, fwd[k][0]).addcmul_(p1y, fwd[k][1])
        I(vx).add_(ax, alpha=dt / dh)
        I(vy).add_(ay, alpha=dt / dh)
        if adj is not None:
            vx[iyr, ixr] += adj[0][:, n]
            vy[iyr, ixr] += adj[1][:, n]
        sec[0, n] = vx[iyr, ixr]
        sec[1, n] = vy[iyr, ixr]
        sc = 1.0 / dh if L else dt / dh
        dxx, dyy = g.diff(vx, "x", False), g.diff(vy, "y", False)
        sx, sy = dxx[0] / dh, dyy[0] / dh
        vxx, vyy = g.damp("e", dxx * sc, "x"), g.damp("f", dyy * sc, "y")
        sh = g.damp("g", g.diff(vy, "x", True) * sc, "xh") + g.damp("h", g.diff(vx, "y", True) * sc, "yh")
        if phys == VTI:
            I(sxy).add_(c44 * sh)
            I(sxx).add_(c11 * vxx + c13 * vyy)
            I(syy).add_(c13 * vxx + c33 * vyy)
        elif L == 0:
            I(sxy).add_(muh * sh)
            gd = gm * (vxx + vyy)
            I(sxx).add_(gd + 2.0 * f * vxx)
            I(syy).add_(gd + 2.0 * f * vyy)
        else:
            gd = gm * (vxx + vyy)
            h2 = 0.5 * dt
            I(sxy).add_(fip * sh + h2 * sum(mr))
            I(sxx).add_(gd - 2.0 * f * vyy + h2 * sum(mp))
            I(syy).add_(gd - 2.0 * f * vxx + h2 * sum(mq))
            for l in range(L):
                e = eta[l] * tau
                ev = piv * e * (vxx + vyy)
                mr[l] = bq[l] * (mr[l] * cq[l] - muhv * e * sh)
                mp[l] = bq[l] * (mp[l] * cq[l] - ev + 2.0 * muv * e * vyy)
                mq[l] = bq[l] * (mq[l] * cq[l] - ev + 2.0 * muv * e * vxx)
            I(sxy).add_(h2 * sum(mr))
            I(sxx).add_(h2 * sum(mp))
            I(syy).add_(h2 * sum(mq))
        if adj is None:
            a = _amp(sig, n, dt)
            sxx[iys, ixs] += a
            syy[iys, ixs] += a
        if mirror:
            syy[H] = 0.0
            sx = g.damp("s", sx[None, :].clone(), "x")[0]
            row = sxx[H, H:H + g.nx]
            if L == 0:
                g0, f0 = gm[0], 2.0 * f[0]
                row.sub_(dt * (g0 * g0 / (g0 + f0) * sx + g0 * sy))
            else:
                for l in range(L):
                    mq[l][0] = 0.0
                row.sub_(dt * (gfs - fjm) ** 2 * sx / gfs + dt * (gfs - fjm) * sy + 0.5 * dt * sum(q[0] for q in mp))
                for l in range(L):
                    mp[l][0] += eta[l] * bq[l] * (dme * (fjm / gfs - 1.0) * sx - dme * sy)
                row.add_(0.5 * dt * sum(q[0] for q in mp))
        if store:
            keep.append(snap + [I(sxx).clone(), I(syy).clone(), I(sxy).clone()])
        if adj is not None and k >= 0:
            qx, qy, qs = fwd[k][2:]
            a, b = I(sxx), I(syy)
            pp = (qx + qy) * (a + b)
            wc.add_(pp)
            wcu.add_(torch.where(wet, (qs * I(sxy) + 0.25 * (qx - qy) * (a - b)) * imm + pp * ilm, 0.0))
    if adj is not None:
        return wc, wcu, wcr, m, dt
    return [sec[k].T.contiguous() for k in range(2)], keep


def _gradient64(s):
    p = s["p"]
    obs, _ = _psv64(s, s["true"])
    syn, keep = _psv64(s, s["model"], mode=1)
    adj = []
    for o, y in zip(obs, syn):
        d = y - o
        d[:, 0] = 0.0
        adj.append(torch.flip(torch.cumsum(d * float(np.float32(p.dt)), 1), [1]))
    l2 = sum(0.5 * float((a * a).sum()) for a in adj)
    wc, wcu, wcr, (vp, vs, rho), dt = _psv64(s, s["model"], adj=adj, fwd=keep)
    lam0, mu0 = rho * (vp ** 2 - 2 * vs ** 2), rho * vs ** 2
    lam, mu, rs = -dt * wc / (4.0 * (lam0 + mu0) ** 2), -dt * wcu, -dt * wcr
    gvp, gvs = 2 * vp * rho * lam, -4 * rho * vs * lam + 2 * rho * vs * mu
    grho = (vp ** 2 - 2 * vs ** 2) * lam + vs ** 2 * mu + rs
    return dict(l2=l2, vp=gvp.T.cpu().numpy(), vs=gvs.T.cpu().numpy(), rho=grho.T.cpu().numpy())


def exact(case, seed):
    if case["kind"] == "batch":
        return [tuple(a.cpu().numpy() for a in _psv64(s, s["model"])[0]) for s in _batch(case, seed)]
    s = _shot(case, seed)
    if case["kind"] == "gradient":
        return _gradient64(s)
    out, _ = _psv64(s, s["model"])
    return [a.cpu().numpy() for a in out[:1 if case["physics"] in (AC, SH) else 2]]

"""Performance cases of the library: the calls a user of it makes, over the
sizes this repository configures, tests and benchmarks.

Kinds of case, each through the public Python entry points (mlegs_amd.hip,
mlegs_amd.adjoint):

* ``steps``     -- a program that steps one run by itself, one ``time_step``
  call (and its DIAGNOST check) per step: the smallest calls, where launches
  and host latency count.
* ``march``     -- ``Solver.time_stepping`` over several steps, AB2-CN from a
  saved state and history, or ETD2 from ``initialize`` on.
* ``sweep``     -- many runs of different resolution stepped together.
* ``gradient``  -- the optimal-perturbation gradient: a trajectory forward and
  its adjoint backward through torch.autograd.
* ``pointwise`` -- transforms both ways: velocities of (psi, chi) to physical
  space, their product |u|^2 there, and that back to coefficients.
* ``operators`` -- spectral operators and band solves on coefficients: DEL2,
  IDEL2LN, IHELM, GRAD, PC2VEL, PROJECT.
* ``force``     -- CALC_BOUSSI_FORCE, the right-hand side of the march.
* ``monitor``   -- what a run prints at its output cadence: energies per
  (m, k), spectra, DIAGNOST's integrals.

Sizes are the benchmark workloads' (64x32x32, 128x64x64, 384x256x256, the
48-run sweep), the shipped read.input's (408x204x608: lengths that are not
powers of two) and sizes between and beside them.
"""
import math
from collections import OrderedDict

import numpy as np
import torch

from mlegs_amd import adjoint, hip as H
from mlegs_amd.configs import LAMB_OSEEN_Q

PARAMS = dict(minc=1, mklink=0, ell=1.0, zlen=2 * math.pi, nu=1e-3, kappa=1e-3, nup=0.0, kappap=0.0, visc_sw=1,
              visc_p=0, omega=0.5, bv0=1.0, adams=1, hyper_cn=0, dt=1e-3)
PRODUCTION = dict(ell=2.0, zlen=4 * math.pi, nu=1e-4, kappa=1e-4, nup=1e-14, kappap=1e-14, visc_p=4, omega=1.0,
                  bv0=2.0, adams=0, hyper_cn=1, dt=5e-4)
SHIPPED = dict(ell=8.0, zlen=6 * math.pi, nu=2e-7, kappa=2e-7, nup=1.0, kappap=1.0, visc_sw=3, visc_p=8, omega=0.0,
               bv0=0.1, adams=0, dt=0.1)


def listed():
    return [
        # a script or a coupled program that calls the library step by step on a small grid
        dict(name="steps 32x16x16", kind="steps", nr=32, nth=16, nx=16, nrchop=22, ntchop=6, nxchop=5, steps=4),
        # the reference's CPU-sized case
        dict(name="march 64x32x32", kind="march", nr=64, nth=32, nx=32, nrchop=48, ntchop=11, nxchop=11, steps=10,
             params="plain", graph=True),
        # the adjoint workload's forward march, a common exploratory size
        dict(name="march 128x64x64", kind="march", nr=128, nth=64, nx=64, nrchop=96, ntchop=22, nxchop=22, steps=10,
             params="plain", graph=True),
        # the production workload: ETD2 from the start on, captured steps
        dict(name="march 384x256x256", kind="march", nr=384, nth=256, nx=256, nrchop=256, ntchop=86, nxchop=86,
             steps=16, params="production", graph=True),
        # the reference's shipped read.input, with its axial sponge: lengths with factors 17 and 19
        dict(name="march 408x204x608", kind="march", nr=408, nth=204, nx=608, nrchop=400, ntchop=136, nxchop=304,
             steps=2, params="shipped", graph=False),
        # a parameter study: one run of every grid of the 48-run workload
        dict(name="sweep 12 runs", kind="sweep", runs=12, nr_lo=64, nr_hi=192, n_lo=32, n_hi=128, steps=8),
        # optimal perturbations: forward and backward, checkpointed
        dict(name="gradient 128x64x64", kind="gradient", nr=128, nth=64, nx=64, nrchop=96, ntchop=22, nxchop=22,
             steps=6, every=3),
        # transforms both ways at the production size
        dict(name="pointwise 384x256x256", kind="pointwise", nr=384, nth=256, nx=256, nrchop=256, ntchop=86, nxchop=86,
             split=False),
        # composite lengths at a middling size, as a resolution study picks them
        dict(name="pointwise 150x90x100", kind="pointwise", nr=150, nth=90, nx=100, nrchop=97, ntchop=31, nxchop=34,
             split=False),
        # band solves and operators at the production size
        dict(name="operators 384x256x256", kind="operators", nr=384, nth=256, nx=256, nrchop=256, ntchop=86, nxchop=86),
        # the march's right-hand side beyond the production lengths: theta and z longer than 256
        dict(name="force 192x512x384", kind="force", nr=192, nth=512, nx=384, nrchop=128, ntchop=171, nxchop=129),
        # what a run prints every few steps
        dict(name="monitor 128x64x64", kind="monitor", nr=128, nth=64, nx=64, nrchop=96, ntchop=22, nxchop=22),
    ]


# ------------------------------------------------------------------ drawn cases
def _length(rng, lo, hi):
    """A transform length: half the time a power of two, else a product of
    primes up to 19, odd ones among them."""
    while True:
        n = round(math.exp(rng.uniform(math.log(lo), math.log(hi))))
        if rng.random() < 0.5:
            n = 2 ** round(math.log2(n))
        r = n
        for p in (2, 3, 5, 7, 11, 13, 17, 19):
            while r % p == 0:
                r //= p
        if r == 1 and lo <= n <= hi:
            return n


def _sizes(rng, nr_lo, nr_hi, lo, hi, most):
    while True:
        nr = 2 * round(math.exp(rng.uniform(math.log(nr_lo), math.log(nr_hi))) / 2)
        nth, nx = _length(rng, lo, hi), _length(rng, lo, hi)
        if nr * nth * nx <= most:
            break
    # the 2/3 rule in r; a third (dealiased products) or, as read.input does, more of theta and z
    nrchop = rng.choice((2 * nr // 3, 2 * nr // 3 + 1, nr - 8))
    ntchop = min(rng.choice((nth // 3 + 1, nth // 3 + 1, 2 * nth // 3)), nrchop - 4)
    nxchop = rng.choice((nx // 3 + 1, nx // 3 + 1, nx // 2))
    return dict(nr=nr, nth=nth, nx=nx, nrchop=nrchop, ntchop=ntchop, nxchop=nxchop)


def draw(rng):
    kind = rng.choice(("steps", "march", "march", "sweep", "gradient", "pointwise", "pointwise", "operators", "force",
                       "monitor"))
    if kind == "steps":
        return dict(kind=kind, steps=4, **_sizes(rng, 24, 64, 12, 32, 64 * 32 * 32))
    if kind == "march":
        params = rng.choice(("plain", "plain", "production"))
        return dict(kind=kind, steps=rng.randint(4, 8), params=params, graph=rng.random() < 0.7,
                    **_sizes(rng, 48, 408, 24, 320, 384 * 256 * 256 // 2))
    if kind == "sweep":
        return dict(kind=kind, runs=rng.randint(6, 16), nr_lo=rng.choice((48, 64)), nr_hi=rng.choice((128, 192, 200)),
                    n_lo=rng.choice((24, 32)), n_hi=rng.choice((64, 96, 128)), steps=rng.randint(4, 8))
    if kind == "gradient":
        return dict(kind=kind, steps=rng.randint(3, 6), every=3, **_sizes(rng, 48, 192, 24, 100, 192 * 96 * 96))
    most = 384 * 256 * 256
    if kind == "pointwise":
        return dict(kind=kind, split=rng.random() < 0.2, **_sizes(rng, 48, 408, 32, 608, most))
    if kind == "monitor":
        return dict(kind=kind, **_sizes(rng, 48, 256, 24, 256, most // 4))
    return dict(kind=kind, **_sizes(rng, 48, 408, 32, 608, most))


# ------------------------------------------------------------------ inputs
def _cfg(case):
    # the longer the lines, the smaller the plain runs' step (their explicit products)
    plain = dict(dt=1e-3 if max(case["nth"], case["nx"]) <= 64 else 2.5e-4)
    extra = {"plain": plain, "production": PRODUCTION, "shipped": SHIPPED}[case.get("params", "plain")]
    return {**PARAMS, **extra, **{k: case[k] for k in ("nr", "nth", "nx", "nrchop", "ntchop", "nxchop")}}


class _Plan:
    """What a program keeps for one resolution: the grid and the coefficients
    of the Lamb-Oseen vortex on it (the m = 0, k = 0 column, and its log term)."""

    def __init__(self, cfg, split=False):
        self.cfg, self.stream = cfg, None
        self.grid = H.Grid(dict(cfg, split=1) if split else cfg)
        one = H.Grid(dict(cfg, nth=2, nx=2, ntchop=1, nxchop=1))
        psi, chi = one.scalar(), one.scalar()
        H.qvortex(one, LAMB_OSEEN_Q, psi, chi)
        col, _, ln = psi.download()
        e = np.zeros(self.grid.shape(H.FFF), dtype=np.complex128, order="F")
        e[:, 0, 0] = col[:, 0, 0]
        self.vortex = self.grid.scalar(H.FFF, e, ln)
        self.column, self.ln = col[:, 0, 0], ln
        for f in (psi, chi):
            f.close()
        one.close()


_plans = OrderedDict()


def _plan(cfg, split=False):
    key = (tuple(sorted(cfg.items())), split)
    if key not in _plans:
        while len(_plans) >= 1:  # one resolution at a time: its device memory goes with its last field
            _plans.popitem()
        _plans[key] = _Plan(cfg, split)
    return _plans[key]


def _noise(cfg, seed, amp, full):
    """Complex Gaussian coefficients inside the truncation as a numpy array
    (n, m, k): the workloads' envelope exp(-(n/16)^2-(m/4)^2-(k/4)^2), or,
    with full, a slow decay over every kept coefficient.  m = 0 is Hermitian
    in k, its k = 0 column real and falling off fast in n."""
    nrd, ntd = min(cfg["nrchop"] + 6, cfg["nr"]), min(cfg["ntchop"], cfg["nth"])
    nxc, nxd = cfg["nxchop"], 2 * cfg["nxchop"] - 1
    nb, mb, kb = (nrd, ntd, nxc) if full else (min(nrd, 96), min(ntd, 24), min(nxc, 24))
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    z = torch.randn((2 * kb - 1, mb, nb), dtype=torch.complex128, device="cuda", generator=g)
    n = torch.arange(nb, dtype=torch.float64, device="cuda")[None, None, :]
    m = torch.arange(mb, dtype=torch.float64, device="cuda")[None, :, None]
    k = torch.arange(2 * kb - 1, dtype=torch.float64, device="cuda")
    k = torch.where(k < kb, k, 2 * kb - 1 - k)[:, None, None]
    z *= amp * (1.0 / ((1 + n) * (1 + m) * (1 + k)) ** 1.5 if full else torch.exp(-((n / 16) ** 2) - (m / 4) ** 2 - (k / 4) ** 2))
    z *= (n < cfg["nrchop"] - m) & ~((n == cfg["nrchop"] - 1 - m) & (m == 1))  # DEL2 wants the top m = 1 row empty
    z[0, 0] = z[0, 0].real.to(z.dtype)
    if kb > 1:
        z[kb:, 0] = z[1:kb, 0].flip(0).conj()
    pos = list(range(kb)) + [nxd - kb + 1 + i for i in range(kb - 1)]
    return z, pos, nb, mb


def _set(field, vortex, cfg, seed, amp, full):
    """field = (the vortex or zero) + noise, on the device."""
    if vortex is not None:
        H.copy(field, vortex)
    else:
        field.zero(H.FFF)
    field.grid.synchronize()
    z, pos, nb, mb = _noise(cfg, seed, amp, full)
    t = field.as_tensor().permute(2, 1, 0)
    t[torch.tensor(pos, device="cuda"), :mb, :nb] += z
    torch.cuda.synchronize()


def _state(plan, cfg, seed, amp, full=False):
    f = [plan.grid.scalar() for _ in range(3)]
    for i in range(3):
        _set(f[i], plan.vortex if i == 0 else None, cfg, 7 * seed + i, amp, full)
    return f


class _Memory:
    """Device memory of a field as torch sees it; the tensor made of it keeps
    this object, and with it the state that owns the memory."""

    def __init__(self, ptr, n, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2, "strides": None}


def _value(f, state):
    """The field's coefficients or values, and its log-term coefficient."""
    e, ln = f.device_ptrs()
    shape = f.grid.shape(f.space)
    t = torch.as_tensor(_Memory(e, math.prod(shape), "<c16", state), device="cuda")
    return [t.view(shape[::-1]).permute(2, 1, 0), torch.as_tensor(_Memory(ln, 1, "<f8", state), device="cuda")]


def _sweep_cfgs(case):
    """The sweep's runs: NR over its range fastest, then theta and z lengths;
    parameters spread over the runs."""
    rng = np.random.default_rng(20261204)
    nrs = [v for v in (48, 64, 96, 128, 192, 200) if case["nr_lo"] <= v <= case["nr_hi"]]
    ns = [v for v in (24, 32, 64, 96, 128) if case["n_lo"] <= v <= case["n_hi"] and (v in (32, 64, 128) or v in (case["n_lo"], case["n_hi"]))]
    out = []
    for i in range(case["runs"]):
        nr, n = nrs[i % len(nrs)], ns[(i // len(nrs)) % len(ns)]
        out.append(dict(PARAMS, nr=nr, nth=n, nx=n, nrchop=2 * nr // 3, ntchop=n // 3 + 1, nxchop=n // 3 + 1, nu=5e-4,
                        kappa=5e-4, dt=2.5e-4, ell=float(rng.uniform(1, 3)), omega=float(rng.uniform(0, 2)),
                        bv0=float(rng.uniform(0, 4))))
    return out


def _started(plan, cfg, seed, params="plain"):
    """A run under way: the solver, its fields, and a saved state and history."""
    f = _state(plan, cfg, seed, {"plain": 1e-5, "production": 1e-4, "shipped": 1e-6}[params])
    s = H.Solver(plan.grid)
    if params == "shipped":
        s.set_march_controls(2, 1000, 1, 100)
    saved = [plan.grid.scalar() for _ in range(3)]
    if cfg["adams"]:
        s.initialize(*f)
        f = list(f) + list(s.history())
        saved += [plan.grid.scalar() for _ in range(3)]
    for a, b in zip(saved, f):
        H.copy(a, b)
    plan.grid.synchronize()
    return dict(solver=s, f=f, saved=saved)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sweep":
        plans = [_Plan(c) for c in _sweep_cfgs(case)]
        runs = [_started(p, p.cfg, 1000 * seed + i) for i, p in enumerate(plans)]
        sw = H.Sweep([(r["solver"], *r["f"][:3]) for r in runs], grouped=False, tune=False, streams=True)
        sw.steps(2, check=False)  # records the runs' steps
        return dict(case=case, runs=runs, sweep=sw, plans=plans)
    cfg = _cfg(case)
    plan = _plan(cfg, bool(case.get("split")))
    g = plan.grid
    if kind in ("steps", "march"):
        return dict(case=case, plan=plan, **_started(plan, cfg, seed, case.get("params", "plain")))
    if kind == "gradient":
        plan.stream = plan.stream or torch.cuda.Stream()
        f = _state(plan, cfg, seed, 1e-5)
        with torch.cuda.stream(plan.stream):
            m = adjoint.March(g)
            x0 = m.state_from(*[a.download()[0] for a in f], psi_ln=f[0].ln).requires_grad_(True)
        return dict(case=case, plan=plan, march=m, x0=x0, stream=plan.stream)
    f = _state(plan, cfg, seed, 1e-2 if kind != "monitor" else 1e-4, full=kind != "monitor")
    return dict(case=case, plan=plan, f=f, w=[g.scalar() for _ in range({"pointwise": 4, "operators": 11, "force": 3, "monitor": 0}[kind])])


# ------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("steps", "march"):
        s, f = state["solver"], state["f"]
        for a, b in zip(f, state["saved"]):
            H.copy(a, b)
        u = f[:3]
        if len(f) == 3:
            s.initialize(*u)
        if kind == "steps":
            for _ in range(case["steps"]):
                s.time_step(*u)
        else:
            s.time_stepping(*u, case["steps"], graph=case["graph"])
        return [_value(a, state) for a in f]
    if kind == "sweep":
        for r in state["runs"]:
            for a, b in zip(r["f"], r["saved"]):
                H.copy(a, b)
        state["sweep"].steps(case["steps"], check=False)
        return [[_value(a, state)[0] for a in r["f"][:3]] + _value(r["f"][0], state)[1:] for r in state["runs"]]
    if kind == "gradient":
        with torch.cuda.stream(state["stream"]):
            x = state["x0"]
            x.grad = None
            J = adjoint.trajectory_energy(state["march"], x, case["steps"], every=case["every"])
            J.backward()
        return [J.detach(), x.grad]
    f, w = state["f"], state["w"]
    if kind == "pointwise":
        H.pc2vel(f[0], f[1], *w[:3])
        for a in w[:3]:
            H.tofp(a)
        H.vdotpsub(*w[:3], *w[:3], w[3])
        H.toff(w[3])
        return [_value(a, state) for a in w]
    if kind == "operators":
        H.del2(f[1], w[0])
        H.idel2ln(f[2], w[1])
        H.ihelm(f[2], w[2], 2.0 / (1e-3 * 1e-3))
        H.grad(f[2], *w[3:6])
        H.pc2vel(f[0], f[1], *w[6:9])
        H.project(*w[6:9], w[9], w[10], 0.0)
        return [_value(a, state) for a in w[:6] + w[9:]]
    if kind == "force":
        H.calc_boussi_force(*f, *w)
        return [_value(a, state) for a in w]
    ke, pe, dke = H.calc_boussi_energy(*f)
    em, ek = H.enemon(*f[:2])
    d = H.diagnost_it1(*f[:2])
    return [ke, pe, dke, em, ek, [d[k] for k in H.DIAGNOST_IT1_KEYS]]


# ------------------------------------------------------------------ work and tolerance
def _costs(c):
    """Of one field: FFF elements, Legendre transform, z and theta transforms in flops."""
    sn = sum(max(0, c["nrchop"] - m) for m in range(c["ntchop"]))
    nk = 2 * c["nxchop"] - 1
    leg = 2.0 * c["nr"] * sn * nk
    fz = 5.0 * c["nr"] * c["ntchop"] * c["nx"] * math.log2(c["nx"])
    ft = 5.0 * c["nr"] * c["nx"] * c["nth"] * math.log2(c["nth"])
    return float(sn) * nk, leg, fz, ft


def work(case):
    kind = case["kind"]
    if kind == "sweep":
        w = [work(dict(c, kind="march", steps=case["steps"], params="plain")) for c in _sweep_cfgs(case)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    n, leg, fz, ft = _costs(case)
    # the right-hand side: ten fields to physical space, the products, four back (five Legendre products for PROJECT, one for N_b)
    force = 16 * leg + 14 * (fz + ft) + 30.0 * case["nr"] * case["nth"] * case["nx"] * 2
    solve = 40.0 * n
    if kind in ("steps", "march"):
        etd = case.get("params", "plain") != "plain"
        # state and history in and out; ETD: ten fields, and five more Legendre products for its second projection
        passes = case["steps"] + (3 if etd else 0)
        return {"bytes": passes * 16.0 * n * (20 if etd else 12), "flops": passes * (force + 4 * solve + (5 * leg if etd else 0))}
    if kind == "gradient":
        # forward, the segments again, and the adjoint steps at twice a force each
        return {"bytes": case["steps"] * 16.0 * n * 36, "flops": case["steps"] * 4 * (force + 4 * solve)}
    if kind == "pointwise":
        ppp = float(case["nr"]) * case["nth"] * case["nx"]
        return {"bytes": 16.0 * (2 * n + 3 * ppp + n), "flops": 4 * (leg + fz + ft) + 10 * ppp}
    if kind == "operators":
        # eight results of three fields; the velocities' transforms and the five products of PROJECT
        return {"bytes": 16.0 * n * (3 + 8), "flops": 8 * leg + 3 * solve}
    if kind == "force":
        return {"bytes": 16.0 * n * 6, "flops": force + solve}
    return {"bytes": 16.0 * n * 3, "flops": 10 * leg + 10 * (fz + ft)}


def tolerance(case):
    """About four times the difference from plain numpy (exact) and from
    another order of the Legendre sums, whichever was seen larger over the
    ranges: FP64 throughout, but chi is an inverse Laplacian of a projection
    and amplifies the rounding of the sums before it (up to 5e-9 relative in
    one right-hand side, 1.6e-9 per step at 384x256x256), and a march carries
    it on; IDEL2LN likewise (7e-10 at NRCHOP 238).  Split products: 34 significant bits."""
    return {"steps": {"rel": 6e-11}, "march": {"rel": 2e-8}, "sweep": {"rel": 1e-9}, "gradient": {"rel": 1e-10},
            "pointwise": {"rel": 1e-9 if case.get("split") else 1.5e-12}, "operators": {"rel": 3e-9},
            "force": {"rel": 2e-8}, "monitor": {"rel": 1e-10}}[case["kind"]]


# ------------------------------------------------------------------ the same in plain numpy
class _Plain:
    """The discretisation from its definition: mapped associated Legendre
    functions x = (r^2 - L^2)/(r^2 + L^2), orthonormal on the Gauss nodes,
    Fourier in theta (2 NTH points) and z; a field is (coefficients [m, n, k],
    LN) with LN the coefficient of -log(1 - x)."""

    def __init__(self, cfg):
        self.c = cfg
        self.L2 = cfg["ell"] ** 2
        self.nt, self.nk = min(cfg["ntchop"], cfg["nth"]), 2 * cfg["nxchop"] - 1
        self.rows = min(cfg["nrchop"] + 6, cfg["nr"]) + 3
        x, w = np.polynomial.legendre.leggauss(cfg["nr"])
        lx = x.astype(np.longdouble)
        for _ in range(2):  # the nodes and weights to more than 64 bits by Newton
            p0, p1 = np.ones_like(lx), lx.copy()
            for j in range(2, cfg["nr"] + 1):
                p0, p1 = p1, ((2 * j - 1) * lx * p1 - (j - 1) * p0) / j
            dp = cfg["nr"] * (lx * p1 - p0) / (lx * lx - 1)
            lx = lx - p1 / dp
        self.x, self.w = lx.astype(np.float64), (2 / ((1 - lx * lx) * dp * dp)).astype(np.float64)
        self.r2 = (self.L2 * (1 + lx) / (1 - lx)).astype(np.float64)
        m = np.arange(self.nt, dtype=np.longdouble)[:, None]
        n = m + np.arange(self.rows + 1, dtype=np.longdouble)[None, :]
        al = np.sqrt((n * n - m * m) / (4 * n * n - 1) * (n > m))
        self.al, self.n, self.m = al.astype(np.float64), n.astype(np.float64)[:, :-1], m.astype(np.float64)
        P = np.zeros((self.nt, self.rows + 1, cfg["nr"]), dtype=np.longdouble)
        pmm = np.full(cfg["nr"], np.sqrt(np.longdouble(0.5)))
        s = np.sqrt(1 - lx * lx)
        for mm in range(self.nt):
            if mm:
                pmm = -pmm * s * np.sqrt(np.longdouble(2 * mm + 1) / (2 * mm))
            P[mm, 0] = pmm
            for j in range(1, self.rows + 1):
                P[mm, j] = (lx * P[mm, j - 1] - (al[mm, j - 1] * P[mm, j - 2] if j > 1 else 0)) / al[mm, j]
        self.P = P[:, :-1].astype(np.float64)
        dP = np.zeros((self.nt, self.rows, cfg["nr"]))  # (1 - x^2) P'
        nn = n[:, :-1]
        dP += (-(nn * al[:, 1:])[:, :, None] * P[:, 1:]).astype(np.float64)
        dP[:, 1:] += (((nn + 1) * al[:, :-1])[:, 1:, None] * P[:, :-2]).astype(np.float64)
        self.dP = dP
        k = np.arange(self.nk)
        self.k = (2 * math.pi / cfg["zlen"] * np.where(k < cfg["nxchop"], k, k - self.nk))[None, None, :]
        self.norm = np.sqrt((2 * np.arange(3) + 1) / 2.0)
        self.at1 = np.sqrt((2 * np.arange(self.rows) + 1) / 2.0)

    def keep(self, iof=0):
        """Rows inside the truncation NRCHOP + iof, (m, n, 1)."""
        return (np.arange(self.rows)[None, :] < self.c["nrchop"] + iof - np.arange(self.nt)[:, None])[:, :, None]

    @staticmethod
    def _shift(a, d):
        b = np.zeros_like(a)
        n = a.shape[1]
        b[:, max(d, 0):n + min(d, 0)] = a[:, max(-d, 0):n - max(d, 0)]
        return b

    def mulxm(self, a, iof):
        al0, al1 = self.al[:, :-1, None], self.al[:, 1:, None]
        return (a - self._shift(al1 * a, 1) - self._shift(al0 * a, -1)) * self.keep(iof)

    def xxdx(self, a, ln, iof):
        al0, al1, n = self.al[:, :-1, None], self.al[:, 1:, None], self.n[:, :, None]
        b = self._shift(-n * al1 * a, 1) + self._shift((n + 1) * al0 * a, -1)
        b = b * self.keep(iof)
        b[0, 0, 0] += ln / self.norm[0]
        b[0, 1, 0] += ln / self.norm[1]
        return b

    def delsqh(self, a, ln, iof):
        n = self.n[:, :, None]
        b = -a * n * (n + 1) / self.L2 * self.keep(iof)
        b[0, 0, 0] = ln / self.L2 / self.norm[0]
        return b

    def band(self):
        """Diagonals -2..2 of L^-2 (1 - x)^2 (-n (n + 1)), [m, row]."""
        al, n = self.al, self.n
        a0, a1 = al[:, :-1], al[:, 1:]
        e = -n * (n + 1) / self.L2
        up = lambda v, d: self._shift(v[:, :, None], d)[:, :, 0]
        return [up(e * a1, 2) * up(a1, 1), -2 * up(e * a1, 1), (1 + a0 ** 2 + a1 ** 2) * e, -2 * up(e * a0, -1),
                up(e * a0, -2) * up(a0, -1)]

    def log_rows(self):
        return np.array([4.0 / 3 / self.norm[0], -2.0 / self.norm[1], 2.0 / 3 / self.norm[2]]) / self.L2

    def del2(self, a, ln, iof):
        a = a * self.keep(iof)
        b = sum(d[:, :, None] * self._shift(a, 2 - i) for i, d in enumerate(self.band())) - self.k ** 2 * a
        b = b * self.keep(iof)
        b[0, :3, 0] += self.log_rows() * ln
        return b

    def _penta(self, rhs, alp):
        """(del^2 - alp) x = rhs for m >= 1, all systems side by side (m = 0: zero)."""
        d = [v[:, :, None] + 0 * self.k for v in self.band()]
        keep = self.keep() & (np.arange(self.nt) > 0)[:, None, None]
        d[2] = d[2] - alp - self.k ** 2
        d = [np.where(keep, v, 1.0 if i == 2 else 0.0) for i, v in enumerate(d)]
        nn = self.c["nrchop"] - np.arange(self.nt)[:, None, None]
        j = np.arange(self.rows)[None, :, None]
        d[3], d[4] = np.where(j + 1 < nn, d[3], 0), np.where(j + 2 < nn, d[4], 0)
        x = rhs * keep
        n = self.rows
        for i in range(n):  # elimination of the two rows below
            for q in (1, 2):
                if i + q < n:
                    f = d[2 - q][:, i + q] / d[2][:, i]
                    x[:, i + q] -= f * x[:, i]
                    d[2 - q + 1][:, i + q] -= f * d[3][:, i]
                    d[2 - q + 2][:, i + q] -= f * d[4][:, i]
        for i in range(n - 1, -1, -1):
            t = x[:, i].copy()
            if i + 1 < n:
                t -= d[3][:, i] * x[:, i + 1]
            if i + 2 < n:
                t -= d[4][:, i] * x[:, i + 2]
            x[:, i] = t / d[2][:, i]
        return x

    def _dense0(self, np_):
        A = np.zeros((np_, np_))
        for i, d in enumerate(self.band()):
            o = i - 2
            for r in range(np_):
                if 0 <= r + o < np_:
                    A[r, r + o] = d[0, r]
        return A

    def fix(self, a):
        nn = self.c["nrchop"]
        a[0, 0] -= (self.at1[:nn, None] * a[0, :nn]).sum(0) / self.at1[0]
        return a

    def idel2ln(self, b):
        nn = self.c["nrchop"]
        x = self._penta(b, 0.0)
        A = self._dense0(nn)
        for k in range(self.nk):
            M = A - self.k[0, 0, k] ** 2 * np.eye(nn)
            if k == 0:
                M[:3, 0] += self.log_rows() * self.norm[0]
            x[0, :nn, k] = np.linalg.solve(M, b[0, :nn, k])
        ln = x[0, 0, 0].real * self.norm[0]
        x[0, 0, 0] = 0
        return self.fix(x * self.keep()), ln

    def ihelm(self, b, bln, alp):
        nn = self.c["nrchop"]
        ln = -bln / alp
        b = b.copy()
        b[0, :3, 0] -= self.log_rows() * ln
        x = self._penta(b, alp)
        X = np.eye(nn + 1) - np.diag(self.al[0, 1:nn + 1], 1) - np.diag(self.al[0, 1:nn + 1], -1)
        A = self._dense0(nn + 1) - alp * np.eye(nn + 1)
        for k in range(self.nk):
            M = (A - self.k[0, 0, k] ** 2 * np.eye(nn + 1)) @ X
            y = np.zeros(nn + 1, dtype=complex)
            y[:nn - 1] = np.linalg.solve(M[:nn - 1, :nn - 1], b[0, :nn - 1, k])
            x[0, :nn, k] = (X @ y)[:nn]
        return x * self.keep(), ln

    def grad(self, a, ln, iof):
        a1 = a * self.keep(iof)
        return self.xxdx(a, ln, iof), 1j * self.m[:, :, None] * a1, 1j * self.k * a1

    def pc2vel(self, psi, ln, chi, lnc, iof):
        m, k = self.m[:, :, None], self.k
        ur = 1j * m * psi * self.keep(iof) + 1j * k * self.xxdx(chi, lnc, iof)
        up = -self.xxdx(psi, ln, iof) - m * k * chi * self.keep(iof)
        return ur, up, -self.mulxm(self.mulxm(self.delsqh(chi, lnc, iof), iof), iof)

    def pc2vor(self, psi, ln, chi, lnc, iof):
        m, k = self.m[:, :, None], self.k
        d = self.del2(chi, lnc, iof)
        ur = -1j * m * d + 1j * k * self.xxdx(psi, ln, iof)
        up = self.xxdx(d, 0.0, iof) - k * m * psi * self.keep(iof)
        return ur, up, -self.mulxm(self.mulxm(self.delsqh(psi, ln, iof), iof), iof)

    def tofp(self, a, ln, iof=0):
        """Samples at the 2 NTH angles, (r, theta, z)."""
        c = self.c
        u = np.matmul(self.P.transpose(0, 2, 1), a * self.keep(iof))  # m, r, k
        u[0, :, 0] += ln * -np.log1p(-self.x)
        z = np.zeros((self.nt, c["nr"], c["nx"]), dtype=complex)
        z[:, :, :c["nxchop"]] = u[:, :, :c["nxchop"]]
        if c["nxchop"] > 1:
            z[:, :, -(c["nxchop"] - 1):] = u[:, :, c["nxchop"]:]
        z = np.fft.ifft(z, axis=2) * c["nx"]
        z[0] = z[0].real
        return np.fft.irfft(z.transpose(1, 0, 2), n=2 * c["nth"], axis=1) * 2 * c["nth"]

    def to_pff(self, v):
        c = self.c
        s = np.fft.rfft(v, axis=1)[:, :self.nt] / (2 * c["nth"])
        s[:, 0] = s[:, 0].real
        s = np.fft.fft(s, axis=2) / c["nx"]
        s = np.concatenate([s[:, :, :c["nxchop"]], s[:, :, c["nx"] - c["nxchop"] + 1:]], axis=2)
        return s.transpose(1, 0, 2)  # m, r, k

    def toff(self, v):
        return np.matmul(self.P * self.w, self.to_pff(v)) * self.keep()

    def project(self, ur, up, uz):
        """PROJECT of PFF velocities with psi's log term set to 0."""
        m, k, n = self.m[:, :, None], self.k, np.maximum(1, self.n)[:, :, None]
        col = np.matmul(self.P[0] * self.w, up[0, :, 0].real)[:self.c["nrchop"]]
        ln = -0.5 * (col * np.sqrt((2 * np.arange(len(col)) + 1) / 2.0)).sum()
        up = up.copy()
        up[0, :, 0] += ln * (1 + self.x)
        V = self.P * self.w / (1 - self.x ** 2) / (n * (n + 1))
        D = self.dP * self.w / (1 - self.x ** 2) / (n * (n + 1))
        psi = -1j * m * np.matmul(V, ur) - np.matmul(D, up)
        chi = 1j * k * np.matmul(D, ur) + m * k * np.matmul(V, up) - np.matmul(self.P * self.w, uz)
        return self.fix(psi * self.keep()), chi * self.keep()

    def force(self, psi, ln, chi, lnc, b):
        u = [self.tofp(a, 0.0, 3) for a in self.pc2vel(psi, ln, chi, lnc, 3)]
        o = [self.tofp(a, 0.0, 3) for a in self.pc2vor(psi, ln, chi, lnc, 3)]
        g = [self.tofp(a, 0.0, 3) for a in self.grad(b, 0.0, 3)]
        r2, om, n2 = self.r2[:, None, None], 2 * self.c["omega"], self.c["bv0"] ** 2
        x = u[1] * o[2] - u[2] * o[1] + om * u[1]
        y = u[2] * o[0] - u[0] * o[2] - om * u[0]
        z = (u[0] * o[1] - u[1] * o[0]) / r2 - self.tofp(b, 0.0)
        bn = -((u[0] * g[0] + u[1] * g[1]) / r2 + u[2] * g[2]) + n2 * u[2]
        pn, w = self.project(*[self.to_pff(v) for v in (x, y, z)])
        cn, cln = self.idel2ln(w)
        return (pn, 0.0), (cn, cln), (self.toff(bn), 0.0)

    def field(self, a, ln=0.0):
        """[coefficients as the library lays them out, LN]."""
        nrd = min(self.c["nrchop"] + 6, self.c["nr"])
        return [torch.from_numpy(np.ascontiguousarray(a[:, :nrd].transpose(1, 0, 2))), torch.tensor([float(ln)], dtype=torch.float64)]

    def slots(self, v):
        """Samples as the library lays them out: pairs of angles, padding zero."""
        c = self.c
        out = np.zeros((c["nr"] + 3, c["nth"] + 1, c["nx"]), dtype=complex)
        out[:c["nr"], :c["nth"]] = v[:, 0::2] + 1j * v[:, 1::2]
        return [torch.from_numpy(out), torch.zeros(1, dtype=torch.float64)]


def exact(case, seed):
    """numpy's answer for the transforms, operators, the right-hand side and
    the AB2-CN step; None where that takes too long (the big grids, long
    marches) and for sweeps, gradients, monitors and ETD2 marches."""
    kind = case["kind"]
    if kind not in ("pointwise", "operators", "force", "steps", "march") or case.get("params", "plain") != "plain":
        return None
    n, leg, fz, ft = _costs(case)
    per = {"pointwise": 4, "operators": 10}.get(kind, 18 * case.get("steps", 1))
    if per * (leg / 20 + fz + ft) > 1.2e10 or case["nrchop"] * case["ntchop"] * case["nr"] > 6e6:
        return None
    cfg = _cfg(case)
    p = _Plain(cfg)
    st = prepare(case, seed)

    def arr(f):
        a, _, ln = f.download()
        v = np.zeros((p.nt, p.rows, p.nk), dtype=complex)
        v[:, :a.shape[0]] = a.transpose(1, 0, 2)
        return v, ln

    if kind in ("steps", "march"):
        u = [arr(a) for a in st["saved"]]
        h, u = u[3:], u[:3]
        dt = cfg["dt"]
        for _ in range(case["steps"]):
            N = p.force(*u[0], *u[1], u[2][0])
            new = []
            for (a, ln), (x, xl), (y, yl), nu in zip(u, N, h, (cfg["nu"], cfg["nu"], cfg["kappa"])):
                al = 2 / nu / dt
                s = a + dt * (1.5 * x - 0.5 * y)
                sl = ln + dt * (1.5 * xl - 0.5 * yl)
                new.append(p.ihelm(-p.del2(a, ln, 2) * p.keep() - al * s, -al * sl, al))
            u, h = new, N
        return [p.field(*a) for a in list(u) + list(h)]
    (psi, ln), (chi, lnc), (b, _) = [arr(a) for a in st["f"]]
    if kind == "force":
        return [p.field(*a) for a in p.force(psi, ln, chi, lnc, b)]
    v = p.pc2vel(psi, ln, chi, lnc, 0)
    if kind == "pointwise":
        v = [p.tofp(a, 0.0) for a in v]
        e = (v[0] ** 2 + v[1] ** 2) / p.r2[:, None, None] + v[2] ** 2
        return [p.slots(a) for a in v] + [p.field(p.toff(e))]
    d = p.del2(chi, lnc, 0)
    x = p.idel2ln(b)
    pj, w = p.project(*[np.matmul(p.P.transpose(0, 2, 1), a) for a in v])
    return [p.field(d), p.field(*x), p.field(*p.ihelm(b, 0.0, 2.0 / (1e-3 * 1e-3))), *[p.field(a) for a in p.grad(b, 0.0, 0)],
            p.field(pj), p.field(w)]

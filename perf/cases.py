"""Workloads whose speed matters: what programs built on nrqcd_amd do, through
its public entry points, from single 16^3 time steps to 128^3 runs.

``listed()`` names the standing cases, ``draw(rng)`` gives one more of the same
ranges, ``prepare(case, seed)`` makes what a program holds before the call,
``run(state)`` is one pass with its results, ``work(case)`` the bytes and
floating-point operations such a pass cannot do without, and
``exact(case, seed)`` the same results in plain 64-bit torch arithmetic.

Kinds of case:

* ``evolve``: a stretch of real-time evolution of one gauge configuration with
  energy, Gauss law and plaquette logged along the way, then the transverse
  electric spectrum of the state it reaches (with ``back``, the last steps are
  taken backwards, as the fixed-centre correlator mode does).
* ``ensemble``: the same for several configurations in one batched call.
* ``meson``: the inner loop of the meson-correlator drivers on a lattice that
  fits a CPU run: heavy-quark step, gauge step, correlators, norms and
  observables every step, the whole state downloaded at the end.
* ``heavy``: one heavy-quark Crank-Nicolson step (of one or several masses on
  one gauge configuration) with the correlators and norms that drivers write.
* ``hamiltonian``: that step with all four terms of the Hamiltonian.
* ``learned``: that step preconditioned by the trained network.
* ``gluon``: a gluon-occupation measurement: a copy is brought to Coulomb
  gauge, then both transverse correlators.
* ``thermal``: the thermal initial condition with its Gauss-law projection.

The state of a large lattice stays in HBM between calls, as in the drivers;
what comes back is what they read: log rows, correlators and spectra (per
momentum), and at the small sizes links, fields and propagators whole.
"""
import math

import numpy as np
import torch

import nrqcd_amd as nrq

SOLVERS = {"gmres": nrq.NRQ_SOLVER_GMRES_FP64, "gmres_mixed": nrq.NRQ_SOLVER_GMRES_MIXED,
           "chebyshev": nrq.NRQ_SOLVER_CHEBYSHEV_FP64, "chebyshev_mixed": nrq.NRQ_SOLVER_CHEBYSHEV_MIXED,
           "learned_mixed": nrq.NRQ_SOLVER_FGMRES_CNN_MIXED}
MASSES = (2.0, 1.0, 5.0, 10.0)
KSP_TOL = 1e-10
A0 = 0.05  # time step of the standing runs
REUNIT = 10  # FP32 storage: reunitarisation interval
GLUON_AGE = 20  # time steps before a gluon-occupation measurement


def _case(kind, name=None, n0=16, n1=16, n2=16, **more):
    c = {"kind": kind, "n0": n0, "n1": n1, "n2": n2}
    if name:
        c["name"] = name
    c.update(more)
    return c


def listed():
    return [
        # the 16^3 configuration of a CPU run, as the meson driver orders it: the smallest calls
        _case("meson", "meson_16", precision=64, steps=10, solver="gmres", anisotropy=1.0),
        # reference precision at 64^3: a stretch of the energy-log driver, logging every 10 steps
        _case("evolve", "evolve_64_fp64", 64, 64, 64, precision=64, steps=50, log_every=10, back=0, anisotropy=1.0),
        # ragged extents with unequal spacings, the last steps backwards
        _case("evolve", "evolve_ragged_fp32", 54, 37, 45, precision=32, steps=30, log_every=10, back=2, anisotropy=1.25),
        # the mixed-precision production run: FP32 storage, reunitarised, logged every 50 steps
        _case("evolve", "evolve_128_fp32", 128, 128, 128, precision=32, steps=50, log_every=50, back=0, anisotropy=1.0),
        # a quarter of the 32-member 48^3 ensemble
        _case("ensemble", "ensemble_8x48_fp32", 48, 48, 48, precision=32, members=8, steps=20, anisotropy=1.0),
        # the reference's own solver (PETSc's GMRES(30)) at 64^3
        _case("heavy", "heavy_64_gmres", 64, 64, 64, precision=64, masses=1, solver="gmres", anisotropy=1.0),
        # the fast solver of the production run
        _case("heavy", "heavy_128_mixed", 128, 128, 128, precision=64, masses=1, solver="chebyshev_mixed", anisotropy=1.0),
        # four masses on one member of the ensemble: 48 right-hand sides
        _case("heavy", "heavy_48_four_masses", 48, 48, 48, precision=32, masses=4, solver="chebyshev_mixed", anisotropy=1.0),
        # the network as preconditioner
        _case("learned", "learned_64", 64, 64, 64, precision=64, solver="learned_mixed", anisotropy=1.0),
        # all Wilson coefficients, as the job templates set them; odd extents
        _case("hamiltonian", "hamiltonian_ragged", 33, 30, 27, precision=64, anisotropy=1.0),
        # the gluon-occupation driver's measurement with its default tolerance and cap
        _case("gluon", "gluon_64", 64, 64, 64, precision=64, iterations=100, anisotropy=1.0),
        # thermal start of the equilibrium driver
        _case("thermal", "thermal_16", 16, 16, 16, precision=64, beta=16.0, rounds=1, steps=10, anisotropy=1.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("meson", "evolve", "evolve", "evolve", "ensemble", "heavy", "heavy", "heavy", "hamiltonian",
                       "learned", "gluon", "gluon", "thermal"))
    an = rng.choice((1.0, 1.0, 1.25, 0.8))
    prec = rng.choice((64, 32))
    lo, hi = {"meson": (8, 24), "evolve": (12, 128), "ensemble": (12, 48), "heavy": (12, 112), "hamiltonian": (8, 40),
              "learned": (16, 64), "gluon": (12, 64), "thermal": (6, 18)}[kind]
    ext = [_log_int(rng, lo, hi) for _ in range(3)]
    if rng.random() < 0.4:
        # extents in use are often multiples of 16
        ext = [max(16, 16 * round(e / 16)) if hi >= 32 else 4 * max(1, round(e / 4)) for e in ext]
    if kind == "learned":
        ext[0] = max(16, 16 * round(ext[0] / 16))  # the network needs it
    more = {}
    if kind == "meson":
        more = dict(steps=rng.randint(2, 10), solver=rng.choice(("gmres", "gmres_mixed", "chebyshev", "chebyshev_mixed")))
        prec = 64
    elif kind == "evolve":
        more = dict(steps=rng.randint(5, 50), log_every=rng.choice((5, 10, 25, 50)), back=rng.choice((0, 0, 1, 2)))
    elif kind == "ensemble":
        more = dict(members=rng.randint(2, 8), steps=rng.randint(4, 20))
    elif kind == "heavy":
        more = dict(masses=rng.choice((1, 1, 2, 4)) if max(ext) <= 64 else 1,
                    solver=rng.choice(("gmres", "gmres_mixed", "chebyshev", "chebyshev_mixed", "chebyshev_mixed")))
    elif kind == "learned":
        more = dict(solver="learned_mixed")
        prec = 64
    elif kind == "hamiltonian":
        prec = 64
    elif kind == "gluon":
        more = dict(iterations=rng.randint(10, 100))
    elif kind == "thermal":
        more = dict(beta=rng.choice((8.0, 16.0, 32.0)), rounds=1, steps=rng.randint(1, 10))
        prec = 64
    return _case(kind, None, *ext, precision=prec, anisotropy=an, **more)


# ---------------------------------------------------------------------------
# inputs: links exp(i A) and E of a transverse box occupation, made on the GPU
# ---------------------------------------------------------------------------
def _spacings(case):
    an = case["anisotropy"]
    return (A0, 1.0, an, 1.0 if an == 1.0 else 0.9)


def _ext(case):
    return case["n0"], case["n1"], case["n2"]


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _momentum(ext, sp, dev):
    """Backward-derivative lattice momentum (3, n2, n1, n0) complex, and |p|."""
    p = torch.zeros((3, ext[2], ext[1], ext[0]), dtype=torch.complex128, device=dev)
    for d in range(3):
        arg = math.pi * torch.arange(ext[d], dtype=torch.float64, device=dev) / ext[d]
        mag = 2.0 * torch.sin(arg) / sp[d + 1]
        shape = [1, 1, 1]
        shape[2 - d] = ext[d]
        p[d] += torch.complex(mag * torch.cos(arg), -mag * torch.sin(arg)).reshape(shape)
    return p, torch.sqrt((p.real ** 2 + p.imag ** 2).sum(0))


def _fields(case, seed):
    """A (coordinates of a_i A_i) and lattice E, each (3, 8, n2, n1, n0)."""
    dev = _device()
    ext, sp = _ext(case), _spacings(case)
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    p, pn = _momentum(ext, sp, dev)
    safe = torch.where(pn > 1e-9, pn, torch.ones_like(pn))
    box = ((pn > 1e-9) & (pn <= 1.0)).to(torch.float64)
    out = []
    for power in (-0.5, 0.5):
        # 24 components at a time, one direction each, to bound the memory
        f = torch.empty((3, 8, ext[2], ext[1], ext[0]), dtype=torch.float64, device=dev)
        f.normal_(generator=gen)
        amp = box * math.sqrt(2.0) * safe ** power
        res = torch.empty_like(f)
        for a in range(8):
            k = torch.fft.fftn(f[:, a], dim=(1, 2, 3)) * amp
            long = (p * k).sum(0) / safe ** 2
            k = k - p.conj() * long
            res[:, a] = torch.fft.ifftn(k, dim=(1, 2, 3)).real
        vol = sp[1] * sp[2] * sp[3]
        out.append(res / math.sqrt(vol))
    a, e = out
    for d in range(3):
        a[d] *= sp[d + 1]
        e[d] *= sp[d + 1] * sp[0]
    return a, e


def _algebra(c):
    """alpha^a T^a of coordinates (8, ...) as (3, 3, ...)."""
    h, s = 0.5, 0.5 / math.sqrt(3.0)
    z = torch.zeros_like(c[0])
    cx = torch.complex
    return torch.stack([
        torch.stack([cx(h * c[2] + s * c[7], z), cx(h * c[0], h * c[1]), cx(h * c[3], h * c[4])]),
        torch.stack([cx(h * c[0], -h * c[1]), cx(-h * c[2] + s * c[7], z), cx(h * c[5], h * c[6])]),
        torch.stack([cx(h * c[3], -h * c[4]), cx(h * c[5], -h * c[6]), cx(-2.0 * s * c[7], z)])])


def _mm(a, b):
    """Product of (3, 3, ...) matrices."""
    out = torch.empty_like(a)
    for r in range(3):
        for c in range(3):
            out[r, c] = a[r, 0] * b[0, c] + a[r, 1] * b[1, c] + a[r, 2] * b[2, c]
    return out


def _dag(a):
    return a.transpose(0, 1).conj().resolve_conj()


def _unit(like):
    one = torch.zeros_like(like)
    for k in range(3):
        one[k, k] = 1.0
    return one


def _exp_i(h):
    """exp(i H) of (3, 3, ...): Taylor series of H / 2^6, squared six times."""
    x = 1j * h / 64.0
    out = _unit(h)
    for k in range(14, 0, -1):
        out = _unit(h) + _mm(x, out) / k
    for _ in range(6):
        out = _mm(out, out)
    return out


def _configuration(case, seed):
    """Links (3 dirs, 3, 3, n2, n1, n0) and E (3, 8, ...), as stored at the case's precision."""
    a, e = _fields(case, seed)
    u = torch.stack([_exp_i(_algebra(a[d])) for d in range(3)])
    if case["precision"] == 32:
        u = u.to(torch.complex64).to(torch.complex128)
        e = e.to(torch.float32).to(torch.float64)
    return u, e


def _host_links(u):
    v = u[0, 0, 0].numel()
    return u.reshape(3, 3, 3, v).permute(3, 0, 2, 1).contiguous().cpu().numpy().transpose()


def _host_efield(e):
    v = e[0, 0].numel()
    return e.reshape(3, 8, v).permute(2, 0, 1).contiguous().cpu().numpy().transpose()


# The lattice and the heavy-quark module are set up once per program and kept.
_now = {"lattice": None, "nrqcd": None}


def _modules(case):
    lattice = (_ext(case), _spacings(case))
    heavy = None
    if "solver" in case or case["kind"] == "hamiltonian":
        kind = case.get("solver", "gmres")
        heavy = (kind, 20 if kind == "learned_mixed" else 30)
    if _now["nrqcd"] is not None and (_now["lattice"] != lattice or _now["nrqcd"] != heavy):
        nrq.nrqcd_finalize()
        _now["nrqcd"] = None
    if _now["lattice"] != lattice:
        if _now["lattice"] is not None:
            nrq.lattice_finalize()
            _now["lattice"] = None
        nrq.lattice_init(*lattice)
        _now["lattice"] = lattice
    if heavy is not None and _now["nrqcd"] is None:
        nrq.nrqcd_init(MASSES[0], [1, 0, 0, 0], 1.0, KSP_TOL)
        nrq.nrqcd_set_solver(SOLVERS[heavy[0]], heavy[1])
        _now["nrqcd"] = heavy


def _gauge(case, seed):
    g = nrq.GaugeConfiguration(case["precision"])
    u, e = _configuration(case, seed)
    g.upload(_host_links(u), _host_efield(e))
    if case["precision"] == 32:
        g.SetReunitarisationInterval(REUNIT)
    return g


def _source(case, seed):
    """Lattice index of the point sources (1-based)."""
    return 1 + seed * 7919 % (case["n0"] * case["n1"] * case["n2"])


def prepare(case, seed):
    _modules(case)
    kind = case["kind"]
    s = {"case": case}
    if kind == "thermal":
        s["g"] = nrq.GaugeConfiguration(case["precision"])
        s["seed"] = 1 + seed % (2 ** 31 - 2)
        return s
    if kind == "ensemble":
        s["members"] = [_gauge(case, 31 * seed + k) for k in range(case["members"])]
        return s
    s["g"] = _gauge(case, seed)
    if kind == "gluon":
        s["g"].Update(1.0, GLUON_AGE)  # measured along a run, not on the initial condition
    if kind in ("meson", "heavy", "hamiltonian", "learned"):
        n = case.get("masses", 1)
        s["heavy"] = []
        for _ in range(n):
            f = nrq.NRQCDField()
            f.InitSinglePoint(_source(case, seed), _source(case, seed))
            s["heavy"].append(f)
        s["mass"] = list(MASSES[:n])
    if kind == "learned":
        net = nrq.PreconditionerNet(seed=1 + seed % 1000)
        net.harvest(s["g"], 1.0, 1, seed=1 + seed)
        net.train(2, 1e-3, seed=1)
        s["net"] = net
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _rows(log, case):
    """Energy, Gauss maximum and plaquette of log rows (the reference's Gauss
    sum is zero up to rounding), in the precision of the stored links."""
    return np.ascontiguousarray(np.asarray(log)[:, [0, 2, 3]], dtype=np.float64 if case["precision"] == 64 else np.float32)


def _stored(x, case):
    return x if case["precision"] == 64 else x.astype(np.float32)


def _correlators(f):
    c, cg = f.correlators(), f.correlators(gconjg=True)
    return np.array([c[k] for k in sorted(c)] + [cg[k] for k in sorted(cg)]), np.array(f.norms())


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "evolve":
        g, left = state["g"], case["steps"] - case["back"]
        while left > 0:
            n = min(left, case["log_every"])
            g.Update(1.0, n)
            g.log_observables()
            left -= n
        if case["back"]:
            g.Update(-1.0, case["back"])
            g.log_observables()
        return {"log": _rows(g.read_log(), case), "ee": _stored(g.GetTransverseEECorrelator(), case)}
    if kind == "ensemble":
        nrq.leapfrog_batch(state["members"], 1.0, case["steps"])
        for g in state["members"]:
            g.log_observables()
        return {"log": np.stack([_rows(g.read_log(), case) for g in state["members"]]),
                "ee": np.stack([_stored(g.GetTransverseEECorrelator(), case) for g in state["members"]])}
    if kind == "meson":
        g, f = state["g"], state["heavy"][0]
        corr, norms, obs = [], [], []
        for _ in range(case["steps"]):
            f.Update(g, state["mass"][0], [1, 0, 0, 0], 1.0)
            g.Update(1.0, 1)
            c, n = _correlators(f)
            o = g.observables()
            corr.append(c)
            norms.append(n)
            obs.append([o["energy"], o["gauss_max"], o["plaquette"]])
        links, efield = g.download()
        quark, antiq = f.download()
        return {"correlators": np.array(corr), "norms": np.array(norms), "observables": np.array(obs), "links": links,
                "efield": efield, "quark": quark, "antiquark": antiq}
    if kind in ("heavy", "learned"):
        if kind == "learned":
            nrq.nrqcd_set_preconditioner(state["net"])
        if len(state["heavy"]) == 1:
            state["heavy"][0].Update(state["g"], state["mass"][0], [1, 0, 0, 0], 1.0)
        else:
            nrq.update_batch(state["heavy"], state["g"], state["mass"], [1, 0, 0, 0], 1.0)
        got = [_correlators(f) for f in state["heavy"]]
        return {"correlators": np.array([c for c, _ in got]), "norms": np.array([n for _, n in got])}
    if kind == "hamiltonian":
        f = state["heavy"][0]
        f.Update(state["g"], state["mass"][0], [1, 1, 1, 1], 1.0)
        corr, norms = _correlators(f)
        return {"correlators": corr, "norms": norms}
    if kind == "gluon":
        fixed = state["g"].copy()
        iterations, deviation = fixed.CoulombGaugefixing(1e-8, 0.08, case["iterations"])
        aa, ee = fixed.transverse_correlators()
        return {"aa": _stored(aa, case), "ee": _stored(ee, case), "deviation": float(deviation), "iterations": iterations}
    g = state["g"]
    nrq.random_init(state["seed"])
    energy, deviation, sweeps = g.EquilibriumInit(case["beta"], case["rounds"], case["steps"])
    links, efield = g.download()
    return {"energy": energy, "deviation": deviation, "sweeps": sweeps, "links": links, "efield": efield}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    v = case["n0"] * case["n1"] * case["n2"]
    kind = case["kind"]
    real = case["precision"] / 8
    config = (54 + 24) * real * v  # links and E once
    link_flops = 2600.0            # staples, force, exponential and product of one link update
    hop_flops = 6 * 72 + 30.0      # covariant Laplacian of one colour vector at one site
    if kind == "evolve":
        return {"bytes": case["steps"] * 2 * config + 24 * real * v + 8 * v, "flops": 3 * v * case["steps"] * link_flops}
    if kind == "ensemble":
        m = case["members"]
        return {"bytes": m * (case["steps"] * 2 * config + 24 * real * v + 8 * v),
                "flops": m * 3 * v * case["steps"] * link_flops}
    fields = 12 * case.get("masses", 1)
    # a step to 1e-10 takes about eight applications of the operator: right-hand side, six solver steps, residual
    cn = {"bytes": fields * 2 * 48.0 * v + 54 * real * v, "flops": 8 * fields * v * hop_flops}
    if kind == "meson":
        n = case["steps"]
        return {"bytes": n * (2 * config + cn["bytes"]) + config + 1152.0 * v, "flops": n * (3 * v * link_flops + cn["flops"])}
    if kind in ("heavy", "learned"):
        return cn
    if kind == "hamiltonian":
        # 12 columns of 6 complex numbers; per column and application six hops with the links and two spin-orbit blocks each
        return {"bytes": 12 * 2 * 96.0 * v + config, "flops": 8 * 12 * v * (6 * 144 + 14 * 144.0)}
    if kind == "gluon":
        # per iteration the links read and written, the divergence written and read once
        n = case["iterations"]
        fft = 5 * math.log2(max(v, 2)) * v
        return {"bytes": n * (108 * real * v + 288.0 * v) + config + 16 * v, "flops": n * (18 * fft + 3000.0 * v) + 48 * fft}
    # thermal: the number of projection sweeps depends on the draw; a few thousand at these sizes
    return {"bytes": case["rounds"] * (2000 * (24 * 2 + 54 + 36) * real * v + case["steps"] * 2 * config),
            "flops": case["rounds"] * (2000 * 2500.0 * v + case["steps"] * 3 * v * link_flops)}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _up(x, d, n=1):
    """x shifted so that entry s holds the value at s + n d^."""
    return torch.roll(x, -n, dims=x.dim() - 1 - d)


def _two_im_trace(w):
    """2 Im Tr(T^a W), a = 1..8."""
    return torch.stack([
        w[0, 1].imag + w[1, 0].imag, w[1, 0].real - w[0, 1].real, w[0, 0].imag - w[1, 1].imag,
        w[0, 2].imag + w[2, 0].imag, w[2, 0].real - w[0, 2].real, w[1, 2].imag + w[2, 1].imag,
        w[2, 1].real - w[1, 2].real, (w[0, 0].imag + w[1, 1].imag - 2.0 * w[2, 2].imag) / math.sqrt(3.0)])


def _two_re_trace(w):
    """2 Tr(T^a W) of a Hermitian W."""
    return _two_im_trace(1j * w)


def _links_step(u, e, dt):
    return torch.stack([_mm(_exp_i(_algebra(dt * e[i])), u[i]) for i in range(3)])


def _efield_step(u, e, dt, sp):
    e = e.clone()
    for i in range(3):
        total = torch.zeros_like(u[0])
        for k in range(3):
            if k == i:
                continue
            ui_dn, uk_dn = _up(u[i], k, -1), _up(u[k], k, -1)
            ahead = _mm(_mm(_up(u[k], i), _dag(_up(u[i], k))), _dag(u[k]))
            behind = _mm(_mm(_dag(_up(uk_dn, i)), _dag(ui_dn)), uk_dn)
            total += dt * (sp[0] / sp[k + 1]) ** 2 * (ahead + behind)
        e[i] -= _two_im_trace(_mm(u[i], total))
    return e


def _project(u):
    """Rows 1 and 2 orthonormalised, row 3 the conjugated cross product."""
    r0 = u[:, 0] / torch.sqrt((u[:, 0].real ** 2 + u[:, 0].imag ** 2).sum(1, keepdim=True))
    r1 = u[:, 1] - (r0.conj() * u[:, 1]).sum(1, keepdim=True) * r0
    r1 = r1 / torch.sqrt((r1.real ** 2 + r1.imag ** 2).sum(1, keepdim=True))
    r2 = torch.stack([(r0[:, (c + 1) % 3] * r1[:, (c + 2) % 3] - r0[:, (c + 2) % 3] * r1[:, (c + 1) % 3]).conj()
                      for c in range(3)], 1)
    return torch.stack([r0, r1, r2], 1)


class _Evolution:
    """Leapfrog steps with the reunitarisation interval of the FP32 storage."""

    def __init__(self, case, u, e):
        self.sp, self.u, self.e, self.done = _spacings(case), u, e, 0
        self.every = REUNIT if case["precision"] == 32 else 0

    def step(self, dt, n):
        for _ in range(n):
            if dt > 0:
                self.u = _links_step(self.u, self.e, dt)
                self.e = _efield_step(self.u, self.e, dt, self.sp)
            else:
                self.e = _efield_step(self.u, self.e, dt, self.sp)
                self.u = _links_step(self.u, self.e, dt)
            self.done += 1
            if self.every and self.done % self.every == 0:
                self.u = _project(self.u)

    def observables(self):
        """Energy, Gauss maximum and mean plaquette."""
        u, e, sp = self.u, self.e, self.sp
        energy, plaq = 0.0, 0.0
        gauss = torch.zeros_like(u[0])
        for i in range(3):
            energy += 0.5 * float(((e[i] / sp[i + 1] / sp[0]) ** 2).sum())
            m = _algebra(e[i])
            um, em = _up(u[i], i, -1), _up(m, i, -1)
            gauss += (m - _mm(_mm(_dag(um), em), um)) / sp[i + 1]
            for j in range(i + 1, 3):
                tr = (_mm(_mm(u[i], _up(u[j], i)), _dag(_up(u[i], j))) * u[j].conj()).sum((0, 1)).real
                energy += float((2.0 * 3.0 * (1.0 - tr / 3.0) / sp[i + 1] / sp[j + 1]).sum())
                plaq += float((tr / 3.0).sum())
        dev = float(_two_re_trace(gauss / sp[0]).abs().max())
        return [energy, dev, plaq / (3.0 * e[0, 0].numel())]


def _transverse(f, ext, sp):
    """Transverse correlator of fields f (3, 8, n2, n1, n0) per momentum."""
    p, pn = _momentum(ext, sp, f.device)
    zero = pn < 1e-12
    p2 = torch.where(zero, torch.ones_like(pn), pn ** 2)
    k = torch.fft.fftn(f.to(torch.complex128), dim=(2, 3, 4))
    acc = torch.zeros_like(pn)
    for i in range(3):
        for j in range(3):
            w = (1.0 if i == j else 0.0) - (p[i].conj() * p[j]).real / p2
            acc += 0.5 * w * (k[i] * k[j].conj()).real.sum(0)
    cell = sp[1] * sp[2] * sp[3]
    acc = torch.where(zero, torch.zeros_like(acc), acc) * cell ** 2 / (cell * ext[0] * ext[1] * ext[2]) / 8.0
    return acc.reshape(-1).cpu().numpy()


def _ee(case, e):
    sp = _spacings(case)
    f = torch.stack([e[i] / sp[i + 1] / sp[0] for i in range(3)])
    return _transverse(f, _ext(case), sp)


def _inverse(m):
    """Inverse of (3, 3, ...) matrices by cofactors."""
    out = torch.empty_like(m)
    for r in range(3):
        for c in range(3):
            a, b, d, e = (r + 1) % 3, (r + 2) % 3, (c + 1) % 3, (c + 2) % 3
            out[c, r] = m[a, d] * m[b, e] - m[a, e] * m[b, d]
    return out / (m[0, 0] * out[0, 0] + m[0, 1] * out[1, 0] + m[0, 2] * out[2, 0])


def _log(u):
    """-i log U of unitary (3, 3, ...): three square roots (the unitary polar
    factor of 1 + U), then the series of the inverse Cayley transform."""
    w = u
    for _ in range(3):
        w = w + _unit(w)
        for _ in range(9):
            w = 0.5 * (w + _dag(_inverse(w)))
    x = _mm(w - _unit(w), _inverse(w + _unit(w)))
    x2, out, power = _mm(x, x), torch.zeros_like(x), x
    for k in range(14):
        out = out + power / (2 * k + 1)
        power = _mm(power, x2)
    return -1j * 16.0 * out


# heavy quarks: psi (12 fields, 3 colours, n2, n1, n0); field (j, s) of a point source has j - s even
def _live():
    return [(p, j, s) for p in range(2) for j in range(6) for s in range(2) if (j - s) % 2 == 0]


def _point(case, seed):
    ext = _ext(case)
    s = _source(case, seed) - 1
    at = (s // (ext[0] * ext[1]), s // ext[0] % ext[1], s % ext[0])
    psi = torch.zeros((12, 3, ext[2], ext[1], ext[0]), dtype=torch.complex128, device=_device())
    for f, (_, j, sp) in enumerate(_live()):
        psi[f, (j - sp) // 2][at] = 1.0 / math.sqrt(6.0)
    return psi


def _laplacian(u, x, sp):
    """K x of fields x (..., 3, n2, n1, n0)."""
    out = torch.zeros_like(x)
    for i in range(3):
        xp, m = _up(x, i), _up(u[i], i, -1)
        xm = _up(x, i, -1)
        for r in range(3):
            h = sum(u[i][r, c] * xp[..., c, :, :, :] + m[c, r].conj() * xm[..., c, :, :, :] for c in range(3))
            out[..., r, :, :, :] += (x[..., r, :, :, :] - 0.5 * h) / sp[i + 1] ** 2
    return out


def _crank_nicolson(u, psi, mass, sp):
    """Solves (1 + conj(alpha) K) x = (1 + alpha K) psi by fixed-point iteration."""
    alpha = torch.tensor([-0.5j * sp[0] / (mass if f < 6 else -mass) for f in range(12)], dtype=torch.complex128,
                         device=psi.device).reshape(12, 1, 1, 1, 1)
    y = psi + alpha * _laplacian(u, psi, sp)
    x = psi
    for _ in range(80):
        new = y - alpha.conj() * _laplacian(u, x, sp)
        far = float((new - x).abs().max())
        x = new
        if far < 1e-16:
            break
    return x


def _propagators(psi):
    """(6, 6, V) quark and antiquark matrices, row 2 colour + spin."""
    v = psi[0, 0].numel()
    out = torch.zeros((2, 6, 6, v), dtype=torch.complex128, device=psi.device)
    for f, (p, j, s) in enumerate(_live()):
        for c in range(3):
            out[p, 2 * c + s, j] = psi[f, c].reshape(-1)
    return out[0], out[1]


def _traces(q, a):
    """The eight zero-momentum correlators (sorted by name, then their _gconjg
    variants) and the two norms of propagators (6, 6, V)."""
    v = q.shape[2]

    def one(p):
        pr, qr = p.reshape(3, 2, 3, 2, v), q.reshape(3, 2, 3, 2, v)
        t0 = (p * q.transpose(0, 1)).sum()
        tx = (p.diagonal(dim1=0, dim2=1).sum(1) * q.diagonal(dim1=0, dim2=1).sum(1)).sum()
        ps = pr[0, :, 0] + pr[1, :, 1] + pr[2, :, 2]
        qs = qr[0, :, 0] + qr[1, :, 1] + qr[2, :, 2]
        pc, qc = pr[:, 0, :, 0] + pr[:, 1, :, 1], qr[:, 0, :, 0] + qr[:, 1, :, 1]
        tc, ts = (ps * qs.transpose(0, 1)).sum(), (pc * qc.transpose(0, 1)).sum()
        return [complex(1j * t0), complex(1j * (2 * ts - t0) / 3), complex(0.375j * (tc - t0 / 3)),
                complex(0.125j * (2 * tx - tc - (2 * ts - t0) / 3))]

    corr = one(a.transpose(0, 1).conj()) + one(a.conj())
    return np.array(corr), np.array([float((q.abs() ** 2).sum().sqrt()), float((a.abs() ** 2).sum().sqrt())])


_EPS = [(i, (i + 1) % 3, (i + 2) % 3) for i in range(3)]


class _FullHamiltonian:
    """S - 1 and its adjoint - 1 on columns x (2 spins, 3 colours, n2, n1, n0), all Wilson coefficients 1."""

    def __init__(self, u, e, sp):
        self.u, self.sp = u, sp
        cx = torch.complex128
        f0 = [_log(_exp_i(_algebra(e[j]))).real / (sp[0] * sp[j + 1]) for j in range(3)]
        self.b = torch.zeros_like(f0[0])
        for _, j, k in _EPS:
            for sign, (m, n) in ((0.5, (j, k)), (-0.5, (k, j))):
                plaq = _mm(_mm(_mm(u[m], _up(u[n], m)), _dag(_up(u[m], n))), _dag(u[n]))
                self.b += sign * _log(plaq).real / (sp[m + 1] * sp[n + 1])
        self.b = self.b.to(cx)
        ef = [-f.to(cx) for f in f0]
        self.d = torch.zeros_like(u[0])
        self.hop = {}
        for i, j, k in _EPS:
            um = _up(u[i], i, -1)
            self.d += (_mm(_mm(u[i], _up(ef[i], i)), _dag(u[i])) - _mm(_mm(_dag(um), _up(ef[i], i, -1)), um)) / (2 * sp[i + 1])
            for eps, jj, kk in ((1.0, j, k), (-1.0, k, j)):
                w = _dag(um)
                self.hop[i, kk, 1] = eps * (_mm(ef[jj], u[i]) + _mm(u[i], _up(ef[jj], i))) / (2 * sp[i + 1])
                self.hop[i, kk, -1] = -eps * (_mm(ef[jj], w) + _mm(w, _up(ef[jj], i, -1))) / (2 * sp[i + 1])
        self.sigma = torch.tensor([[[0, 1], [1, 0]], [[0, 1j], [-1j, 0]], [[1, 0], [0, -1]]], dtype=cx, device=e.device)

    def _colour(self, m, x):
        return torch.stack([sum(m[r, c] * x[:, c] for c in range(3)) for r in range(3)], 1)

    def _spin(self, k, x):
        s = self.sigma[k]
        return torch.stack([s[0, 0] * x[0] + s[0, 1] * x[1], s[1, 0] * x[0] + s[1, 1] * x[1]])

    def apply(self, x, mass, adjoint):
        pre = -0.5j * self.sp[0]
        a = [pre / mass, -pre / (2 * mass), -pre / (8 * mass ** 2), -pre * 1j / (8 * mass ** 2)]
        t4 = torch.zeros_like(x)
        for (i, k, sign), g in self.hop.items():
            if adjoint:
                # the transposed hop: from x to x + sign i with G^+ of the site it leaves
                t4 += _up(self._spin(k, self._colour(_dag(g), x)), i, -sign)
            else:
                t4 += self._spin(k, self._colour(g, _up(x, i, sign)))
        diag = [self._colour(_dag(m) if adjoint else m, x) for m in (self.b, self.d)]
        terms = [_laplacian(self.u, x, self.sp)] + diag + [t4]
        return sum((np.conj(c) if adjoint else c) * t for c, t in zip(a, terms))

    def step(self, x, mass):
        y = x + self.apply(x, mass, False)
        for _ in range(120):
            new = y - self.apply(x, mass, True)
            far = float((new - x).abs().max())
            x = new
            if far < 1e-16:
                break
        return x


def _coulomb(u, ext, sp, iterations):
    """Fourier-accelerated Coulomb gauge fixing: (links, transformations, final deviation)."""
    p, pn = _momentum(ext, sp, u.device)
    acc = torch.where(pn > 1e-12, (float(pn.max()) / torch.where(pn > 1e-12, pn, torch.ones_like(pn))) ** 2,
                      torch.ones_like(pn))
    done = 0
    while True:
        delta = torch.zeros_like(u[0])
        for i in range(3):
            d = _up(u[i], i, -1) - u[i]
            delta += 0.5 * (d - _dag(d))
        dev = float(torch.sqrt((delta.real ** 2 + delta.imag ** 2).sum((0, 1))).max()) / 9.0
        if dev <= 1e-8 or done >= iterations:
            return u, done, dev
        delta = 0.08 * torch.fft.ifftn(torch.fft.fftn(delta, dim=(2, 3, 4)) * acc, dim=(2, 3, 4))
        delta = 0.5 * (delta - _dag(delta))
        g = _exp_i(-1j * delta)
        u = torch.stack([_mm(_mm(g, u[i]), _dag(_up(g, i))) for i in range(3)])
        done += 1


def _flat(psi, case):
    """Propagators as download() returns them."""
    return [m.cpu().numpy() for m in _propagators(psi)]


def exact(case, seed):
    kind, ext, sp = case["kind"], _ext(case), _spacings(case)
    v = ext[0] * ext[1] * ext[2]
    if kind == "thermal":
        return None  # its random numbers are the library's own stream
    if kind in ("evolve", "ensemble"):
        if v * case["steps"] * case.get("members", 1) > 3e7:
            return None  # over 20 seconds
        log, ee = [], []
        for k in range(case.get("members", 1)):
            ev = _Evolution(case, *_configuration(case, 31 * seed + k if kind == "ensemble" else seed))
            rows, left = [], case["steps"] - case.get("back", 0)
            while left > 0:
                n = min(left, case.get("log_every", left))
                ev.step(1.0, n)
                rows.append(ev.observables())
                left -= n
            if case.get("back", 0):
                ev.step(-1.0, case["back"])
                rows.append(ev.observables())
            log.append(rows)
            ee.append(_ee(case, ev.e))
        return {"log": np.array(log if kind == "ensemble" else log[0]), "ee": np.array(ee if kind == "ensemble" else ee[0])}
    u, e = _configuration(case, seed)
    if kind == "meson":
        ev, psi = _Evolution(case, u, e), _point(case, seed)
        corr, norms, obs = [], [], []
        for _ in range(case["steps"]):
            psi = _crank_nicolson(ev.u, psi, MASSES[0], sp)
            ev.step(1.0, 1)
            c, n = _traces(*_propagators(psi))
            corr.append(c)
            norms.append(n)
            obs.append(ev.observables())
        quark, antiq = _flat(psi, case)
        return {"correlators": np.array(corr), "norms": np.array(norms), "observables": np.array(obs),
                "links": _host_links(ev.u), "efield": _host_efield(ev.e), "quark": quark, "antiquark": antiq}
    if kind in ("heavy", "learned"):
        got = [_traces(*_propagators(_crank_nicolson(u, _point(case, seed), m, sp))) for m in MASSES[:case.get("masses", 1)]]
        return {"correlators": np.array([c for c, _ in got]), "norms": np.array([n for _, n in got])}
    if kind == "hamiltonian":
        ham, psi = _FullHamiltonian(u, e, sp), _point(case, seed)
        out = torch.zeros((2, 6, 6, v), dtype=torch.complex128, device=psi.device)
        for f, (p, j, s) in enumerate(_live()):
            x = torch.zeros((2,) + tuple(psi[f].shape), dtype=torch.complex128, device=psi.device)
            x[s] = psi[f]
            x = ham.step(x, MASSES[0] if p == 0 else -MASSES[0])
            for t in range(2):
                for c in range(3):
                    out[p, 2 * c + t, j] += x[t, c].reshape(-1)
        corr, norms = _traces(out[0], out[1])
        return {"correlators": corr, "norms": norms}
    # gluon
    if v * case["iterations"] > 3e7:
        return None  # over 20 seconds
    ev = _Evolution(case, u, e)
    ev.step(1.0, GLUON_AGE)
    u, e = ev.u, ev.e
    if case["precision"] == 32:
        return {"aa": None, "ee": _ee(case, e), "deviation": None, "iterations": None}  # links rounded every transformation
    u, done, dev = _coulomb(u, ext, sp, case["iterations"])
    a = torch.stack([_two_re_trace(_log(u[i])) / sp[i + 1] for i in range(3)])
    return {"aa": _transverse(a, ext, sp), "ee": _ee(case, e), "deviation": dev, "iterations": done}

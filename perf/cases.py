"""The work a user of the package has it do, through its public entry points.

A case is one pass of such a program: stepping a dwarf galaxy (small, as the
sample work units have it, and large; every walk form), a batch of dwarfs, a
whole likelihood evaluation from bodies to histograms, the reverse sweep of
the adjoint (direct sum and tree), sampling initial conditions, and the
histograms of a final state.  Bodies are drawn on the GPU from the seed: a
two-component dwarf (Plummer baryons in a Plummer or NFW dark halo, isotropic
velocities) at the Orphan stream's (l, b, r) in the Milky Way potential, or
isolated.  `exact` evaluates the same step by the direct sum in 64 bits.
"""
import math

import numpy as np
import torch

from milkywayathome_client_amd import adjoint as adj
from milkywayathome_client_amd import nbody as nb
from milkywayathome_client_amd.histogram import HistogramParams

# the sample work units' orbit point: (l, b, r) = (218 deg, 53.5 deg, 28.6 kpc), Sun at x = -8
POS = (28.6 * math.cos(math.radians(53.5)) * math.cos(math.radians(218.0)) - 8.0,
       28.6 * math.cos(math.radians(53.5)) * math.sin(math.radians(218.0)),
       28.6 * math.sin(math.radians(53.5)))
VEL = (-156.0, 79.0, 107.0)
DT = 1e-3


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a test-sized isolated sphere stepped one st:step(ctx) at a time: launches and latency
        dict(name="step_small", kind="run", n=1021, steps=1, precision="fp64", criterion="bh86",
             theta=0.5, quad=True, mw=False, graph=False, dark="plummer", eps2=2.9e-2),
        # the sample work unit's 20000 bodies, replayed steps of the default precision
        dict(name="workunit_fp64", kind="run", n=20000, steps=10, precision="fp64",
             criterion="bh86", theta=0.5, quad=True, mw=True, graph=True, dark="plummer",
             eps2=6.2e-3),
        # the same search with the mixed walk that keeps the reference's lists, an odd size
        dict(name="mixed_mid", kind="run", n=100003, steps=10, precision="mixed",
             criterion="bh86", theta=0.5, quad=True, mw=True, graph=True, dark="nfw",
             eps2=2.9e-3),
        # the benchmark harness's other opening rule, monopoles only, wave-coherent lists, eager
        dict(name="coherent_sw93", kind="run", n=65537, steps=5, precision="mixed_coherent",
             criterion="sw93", theta=0.6, quad=False, mw=True, graph=False, dark="plummer",
             eps2=3.0e-3),
        # a million bodies, plain FP64
        dict(name="large_fp64", kind="run", n=1000000, steps=4, precision="fp64",
             criterion="bh86", theta=0.5, quad=True, mw=True, graph=True, dark="nfw",
             eps2=8.9e-4),
        # a million bodies, the group walk with open scale 1.45 and far-field ratio 0.1
        dict(name="large_group", kind="run", n=1000000, steps=20, precision="mixed_group",
             criterion="bh86", theta=0.5, quad=True, mw=True, graph=True, dark="nfw",
             eps2=8.9e-4, scale=1.45, ratio=0.1),
        # a search's generation: 64 dwarfs of 2000 to 40000 bodies in one state
        dict(name="batch_fp64", kind="batch", sims=64, lo=2000, hi=40000, steps=2,
             precision="fp64", theta=0.5, quad=True),
        # one likelihood evaluation: new state, force, steps, histogram, dispersions, release
        dict(name="evaluate", kind="evaluate", n=40000, steps=10, precision="fp64", theta=0.5,
             eps2=4.2e-3),
        # the gradient of a short run by the direct sum: checkpointed forward and reverse sweep
        dict(name="gradient_exact", kind="adjoint", n=20000, steps=4, every=2,
             criterion="exact", theta=0.5, quad=False, eps2=6.2e-3),
        # the same with the tree held fixed per step
        dict(name="gradient_tree", kind="adjoint", n=20000, steps=4, every=2, criterion="bh86",
             theta=0.5, quad=True, eps2=6.2e-3),
        # initial conditions of a Plummer + NFW dwarf into host arrays
        dict(name="sample_dwarf", kind="sample", n=200000, dark="nfw"),
        # counts and outlier-rejected dispersions of a million bodies' final state
        dict(name="histograms", kind="hist", n=1000000, lbins=50, bbins=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _theta(rng, criterion):
    """An opening angle at which no body can accept a cell that holds it (BH86: below 1/sqrt 3)."""
    lo, hi = {"bh86": (0.45, 0.57), "sw93": (0.5, 1.0), "treecode": (0.6, 1.0)}[criterion]
    return round(rng.uniform(lo, hi), 3)


def draw(rng):
    kind = rng.choice(["run"] * 6 + ["batch", "evaluate", "adjoint", "adjoint", "sample", "hist"])
    if kind == "run":
        precision = rng.choice(["fp64", "fp64", "mixed", "mixed_coherent", "mixed_group"])
        n = _log(rng, 500, 600000)
        criterion = rng.choice(["bh86", "bh86", "sw93", "treecode"])
        c = dict(kind=kind, n=n, steps=rng.randint(1, max(1, min(8, 1000000 // n))),
                 precision=precision, criterion=criterion, theta=_theta(rng, criterion),
                 quad=rng.random() < 0.75, mw=rng.random() < 0.8,
                 graph=rng.random() < 0.5, dark=rng.choice(["plummer", "nfw"]),
                 eps2=round(0.03 * (1000.0 / n) ** 0.5, 9))
        if precision == "mixed_group" and rng.random() < 0.5:
            c["scale"] = round(rng.uniform(1.0, 1.6), 3)
            c["ratio"] = round(rng.uniform(0.0, 0.12), 3)
        return c
    if kind == "batch":
        lo = _log(rng, 500, 4000)
        return dict(kind=kind, sims=_log(rng, 2, 64), lo=lo, hi=_log(rng, lo, 20000),
                    steps=rng.randint(1, 2), precision=rng.choice(["fp64", "mixed"]),
                    theta=_theta(rng, "bh86"), quad=True)
    if kind == "evaluate":
        n = _log(rng, 1000, 100000)
        return dict(kind=kind, n=n, steps=rng.randint(1, 10),
                    precision=rng.choice(["fp64", "fp64", "mixed"]), theta=_theta(rng, "bh86"),
                    eps2=round(0.03 * (1000.0 / n) ** 0.5, 9))
    if kind == "adjoint":
        n = _log(rng, 500, 20000)
        steps = rng.randint(1, 4)
        exact = rng.random() < 0.5
        criterion = rng.choice(["bh86", "sw93"])
        return dict(kind=kind, n=n, steps=steps, every=rng.randint(1, steps),
                    criterion="exact" if exact else criterion,
                    theta=min(_theta(rng, criterion), 0.7), quad=not exact and rng.random() < 0.75,
                    eps2=round(0.03 * (1000.0 / n) ** 0.5, 9))
    if kind == "sample":
        return dict(kind=kind, n=_log(rng, 1000, 1000000), dark=rng.choice(["plummer", "nfw"]))
    return dict(kind=kind, n=_log(rng, 1000, 1000000), lbins=rng.choice([25, 50, 100, 131]),
                bbins=rng.choice([1, 1, 2, 5]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _inverse(table_x, table_y, u):
    """x with y(x) = u, linear between the table's points (y rising)."""
    k = torch.searchsorted(table_y, u).clamp(1, table_y.numel() - 1)
    y0, y1, x0, x1 = table_y[k - 1], table_y[k], table_x[k - 1], table_x[k]
    return x0 + (x1 - x0) * (u - y0) / (y1 - y0)


def _dwarf(n, seed, dark="plummer", mw=True, mass_b=12.0, a_b=0.2, mass_d=48.0, a_d=0.8):
    """A two-component dwarf, baryons first: (pos, vel, mass) float64 on the GPU.  Radii from
    each component's mass profile (the NFW halo's mass is 60 inside r200, cut at 5 r200, the
    Plummer spheres cut at 50 (a_b + a_d)); speeds q v_esc with q from q^2 (1 - q^2)^(7/2)."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    f = dict(device="cuda", dtype=torch.float64)
    nbar = n // 2
    u = torch.rand(n, generator=g, **f) * (1.0 - 1e-9) + 5e-10
    cut = 50.0 * (a_b + a_d)

    def plummer_r(u, a):
        top = (cut / math.sqrt(cut * cut + a * a)) ** 3
        return a / torch.sqrt((u * top) ** (-2.0 / 3.0) - 1.0)

    r = torch.empty(n, **f)
    r[:nbar] = plummer_r(u[:nbar], a_b)
    if dark == "nfw":
        m200, r200 = 60.0, (60.0 / 0.568910904587397) ** (1.0 / 3.0)
        x = torch.logspace(-5, math.log10(5.0 * r200 / a_d), 8192, **f)
        m = torch.log1p(x) - x / (1.0 + x)
        c = r200 / a_d
        scale = m200 / (math.log1p(c) - c / (1.0 + c))       # 4 pi rho0 a^3
        mass_d = scale * float(m[-1])
        r[nbar:] = a_d * _inverse(x, m / m[-1], u[nbar:])
        psi_d = scale * torch.log1p(r / a_d) / r
    else:
        r[nbar:] = plummer_r(u[nbar:], a_d)
        psi_d = mass_d / torch.sqrt(r * r + a_d * a_d)
    psi = mass_b / torch.sqrt(r * r + a_b * a_b) + psi_d
    q = torch.linspace(0.0, 0.99, 4096, **f)
    w = torch.cumsum(q * q * (1.0 - q * q) ** 3.5, 0)
    speed = _inverse(q, w / w[-1], torch.rand(n, generator=g, **f)) * torch.sqrt(2.0 * psi)

    def directions():
        d = torch.randn(n, 3, generator=g, **f)
        return d / torch.linalg.norm(d, dim=1, keepdim=True)

    pos, vel = directions() * r[:, None], directions() * speed[:, None]
    for s in (slice(0, nbar), slice(nbar, n)):
        pos[s] -= pos[s].mean(0)
        vel[s] -= vel[s].mean(0)
    if mw:
        pos += torch.tensor(POS, **f)
        vel += torch.tensor(VEL, **f)
    mass = torch.empty(n, **f)
    mass[:nbar] = mass_b / max(nbar, 1)
    mass[nbar:] = mass_d / max(n - nbar, 1)
    return pos, vel, mass


def _members(case, seed):
    """The batch's dwarfs: body counts over [lo, hi], scale radii and masses of the search's
    ranges, each with its softening."""
    sizes = np.random.default_rng([case["sims"], case["lo"], case["hi"]])
    sizes = sizes.integers(case["lo"], case["hi"] + 1, size=case["sims"])
    rng = np.random.default_rng(int(seed))
    out = []
    for k in range(case["sims"]):
        n = int(sizes[k])
        a_b, rr = rng.uniform(0.1, 0.5), rng.uniform(0.1, 0.5)
        m_b, mr = rng.uniform(1.0, 30.0), rng.uniform(0.1, 0.9)
        b = _dwarf(n, 1000003 * int(seed) + k, mass_b=m_b, a_b=a_b, mass_d=m_b / mr * (1.0 - mr),
                   a_d=a_b / rr * (1.0 - rr))
        out.append((b, 0.03 * (1000.0 / n) ** 0.5 * (a_b / 0.2) ** 2))
    return out


def _host(bodies):
    return tuple(t.cpu().numpy() for t in bodies)


def _ctx(case, eps2=None):
    return nb.NBodyCtx.create(timestep=DT, timeEvolve=4.0,
                              eps2=case.get("eps2", 1e-3) if eps2 is None else eps2,
                              theta=case["theta"], criterion=case.get("criterion", "bh86"),
                              useQuad=case.get("quad", True), treeRSize=4.0)


def _hist_params(case):
    return HistogramParams(lambdaBins=case.get("lbins", 50), betaBins=case.get("bbins", 1))


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "run":
        pos, vel, mass = _host(_dwarf(case["n"], seed, case["dark"], case["mw"]))
        pot = nb.milky_way_potential() if case["mw"] else None
        st = nb.NBodyState(_ctx(case), pot, pos, vel, mass, precision=case["precision"],
                           prestep=False)
        if case.get("scale", 1.0) != 1.0:
            st.set_open_scale(case["scale"])
        if case.get("ratio", 0.0):
            st.set_group_expansion(case["ratio"])
        st.gravity()
        if case["graph"]:
            st.set_graph(True)
        s["state"] = st
    elif kind == "batch":
        mem = _members(case, seed)
        st = nb.NBodyBatch(_ctx(case), nb.milky_way_potential(), [_host(b) for b, _ in mem],
                           eps2=[e for _, e in mem], precision=case["precision"])
        st.set_graph(True)
        s["state"] = st
    elif kind == "evaluate":
        s["bodies"] = _host(_dwarf(case["n"], seed))
        s["ignore"] = np.arange(case["n"]) >= case["n"] // 2
        s["ctx"], s["pot"] = _ctx(case), nb.milky_way_potential()
    elif kind == "adjoint":
        s["inputs"] = [t.cpu().requires_grad_(True) for t in _dwarf(case["n"], seed)]
        s["inputs"].append(torch.tensor(DT, dtype=torch.float64, requires_grad=True))
        s["grads"] = [t.cpu() for t in _grads(case, seed)]
        s["cfg"] = adj.EvolveConfig(nsteps=case["steps"], eps2=case["eps2"], theta=case["theta"],
                                    criterion=case["criterion"], use_quad=case["quad"],
                                    every=case["every"], potential=nb.milky_way_potential())
    elif kind == "sample":
        rng = np.random.default_rng(int(seed))
        dark = (("nfw", 60.0, 0.8) if case["dark"] == "nfw" else ("plummer", 48.0, 0.8))
        s["model"] = dict(light=("plummer", float(rng.uniform(8.0, 16.0)), 0.2), dark=dark,
                          seed=int(seed), position=POS, velocity=VEL)
    else:
        n = case["n"]
        pos, vel, mass = _host(_stream(n, seed))
        st = nb.NBodyState(_ctx(dict(theta=0.5)), nb.milky_way_potential(), pos, vel, mass,
                           prestep=False)
        st.set_ignore(np.arange(n) >= n // 2)
        s["state"] = st
    return s


def _grads(case, seed):
    """dL/d(final pos, vel) of a loss: random vectors."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 77)
    f = dict(device="cuda", dtype=torch.float64, generator=g)
    return torch.randn(case["n"], 3, **f), torch.randn(case["n"], 3, **f)


def _stream(n, seed):
    """A disrupted dwarf: the bodies spread along an orbit, so that they fill many bins."""
    pos, vel, mass = _dwarf(n, seed)
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 5)
    f = dict(device="cuda", dtype=torch.float64)
    t = (0.06 * torch.randn(n, generator=g, **f))[:, None]
    v = torch.tensor(VEL, **f)
    return pos + t * v, vel - 300.0 * t * pos / torch.linalg.norm(pos, dim=1, keepdim=True), mass


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _out(case, state):
    """The bodies as a program writes them out: positions and velocities, and in FP64 states
    the accelerations (a mixed walk's are FP32 sums, of use inside the step only)."""
    pos, vel, acc = state.bodies()
    return (pos, vel, acc) if case["precision"] == "fp64" else (pos, vel)


def _dispersions(state, hp):
    d = state.histogram_dispersion(hp)
    return [a for k in sorted(d) for a in d[k]]


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "run":
        st = s["state"]
        if case["graph"] or case["steps"] > 1:
            st.steps(case["steps"])
        else:
            st.step()
        return _out(case, st)
    if kind == "batch":
        s["state"].steps(case["steps"])
        return _out(case, s["state"])
    if kind == "evaluate":
        pos, vel, mass = s["bodies"]
        st = nb.NBodyState(s["ctx"], s["pot"], pos, vel, mass, precision=case["precision"],
                           prestep=False)
        st.run(case["steps"])
        st.set_ignore(s["ignore"])
        hp = _hist_params(case)
        counts, totals = st.histogram(hp)
        out = [counts.astype(np.int64), totals.astype(np.int64)] + _dispersions(st, hp)
        st.close()
        return out
    if kind == "adjoint":
        # a gradient through the run, as a torch model takes it: final state, then the sweep
        end = adj.KDKRun.apply(*s["inputs"], s["cfg"])
        return [t.detach() for t in end] + list(torch.autograd.grad(end, s["inputs"], s["grads"]))
    if kind == "sample":
        pos, vel, mass, typ, cm = nb.mixed_dwarf(case["n"], case["n"] // 2, **s["model"])
        return pos, vel, mass, typ, cm
    hp = _hist_params(case)
    counts, totals = s["state"].histogram(hp)
    return [counts.astype(np.int64), totals.astype(np.int64)] + _dispersions(s["state"], hp)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _step_work(n, precision, quad, theta, exact=False):
    """One force and step: the bodies' state in and out, the Morton order and a tree of 1.5
    nodes a body written and read once; interactions by the walk, about 100 log2 n a body at
    theta 0.5 (fewer as theta grows), 18 flops each and 38 more with a quadrupole."""
    if exact:
        return n * 200.0, 20.0 * n * n
    per = min(n, 100.0 * math.log2(max(n, 4)) * (0.5 / theta) ** 2)
    node = 96.0 if precision == "fp64" else 64.0
    return n * (24 + 72 + 72 + 24 + 2 * 1.5 * node), n * per * (56.0 if quad else 18.0)


def work(case):
    kind = case["kind"]
    n = case.get("n", 0)
    if kind in ("run", "evaluate"):
        b, f = _step_work(n, case["precision"], case.get("quad", True), case["theta"])
        k = case["steps"] + (kind == "evaluate")
        return {"bytes": k * b + (72.0 * n if kind == "run" else 16.0 * 50), "flops": k * f}
    if kind == "batch":
        m = (case["lo"] + case["hi"]) // 2
        b, f = _step_work(m, case["precision"], True, case["theta"])
        k = case["steps"] * case["sims"]
        return {"bytes": k * b + 72.0 * m * case["sims"], "flops": k * f}
    if kind == "adjoint":
        # forward, the segments again, and a force adjoint (about three times a force) per state
        b, f = _step_work(n, "fp64", case["quad"], case["theta"], case["criterion"] == "exact")
        k = case["steps"]
        return {"bytes": (5 * k + 4) * b + 200.0 * n, "flops": (2 * k + 1 + 3 * (k + 1)) * f}
    if kind == "sample":
        return {"bytes": 60.0 * n, "flops": 4000.0 * n + 2 * 2048 * 128 * 200.0}
    return {"bytes": n * (48.0 + 1.0 + 24.0), "flops": n * 0.5 * 400.0}


# ---------------------------------------------------------------------------
# the same in 64 bits, without the package
# ---------------------------------------------------------------------------
def _mw(x):
    """The sample work units' Milky Way: Miyamoto-Nagai disk, Hernquist bulge, log halo."""
    X, Y, Z = x[:, 0], x[:, 1], x[:, 2]
    zp = torch.sqrt(Z * Z + 0.26 ** 2)
    az = 6.5 + zp
    k = -4.45865888e5 / (X * X + Y * Y + az * az) ** 1.5
    disk = torch.stack([k * X, k * Y, k * Z * az / zp], 1)
    halo = x * (-2.0 * 74.61 ** 2 / (144.0 + (x * x).sum(1)))[:, None]
    r = torch.linalg.norm(x, dim=1)
    bulge = x * (-1.52954402e5 / (r * (0.7 + r) ** 2))[:, None]
    return disk + halo + bulge


def _direct(x, m, eps2, mw):
    out = torch.empty_like(x)
    step = max(1, 25_000_000 // x.shape[0])
    for i in range(0, x.shape[0], step):
        d = [x[None, :, k] - x[i:i + step, k, None] for k in range(3)]
        w = d[0] * d[0]
        w.addcmul_(d[1], d[1]).addcmul_(d[2], d[2]).add_(eps2)
        w = m[None, :] / (w * torch.sqrt(w))
        for k in range(3):
            out[i:i + step, k] = (w * d[k]).sum(1)
    return out + _mw(x) if mw else out


def _direct_vjp(x, m, eps2, g):
    """(dL/dx, dL/dm) of the force for dL/da = g, the potential's part by autograd."""
    gx, gm = torch.empty_like(x), torch.empty_like(m)
    step = max(1, 12_000_000 // x.shape[0])
    for i in range(0, x.shape[0], step):
        s = slice(i, i + step)
        d = [x[None, :, k] - x[s, k, None] for k in range(3)]
        s2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] + eps2
        s3 = 1.0 / (s2 * torch.sqrt(s2))
        w = [m[s, None] * g[None, :, k] - m[None, :] * g[s, k, None] for k in range(3)]
        dw = 3.0 * (d[0] * w[0] + d[1] * w[1] + d[2] * w[2]) / s2
        for k in range(3):
            gx[s, k] = (s3 * (w[k] - dw * d[k])).sum(1)
        gm[s] = -(s3 * (d[0] * g[None, :, 0] + d[1] * g[None, :, 1] + d[2] * g[None, :, 2])).sum(1)
    y = x.detach().clone().requires_grad_(True)
    with torch.enable_grad():
        (e,) = torch.autograd.grad((_mw(y) * g).sum(), y)
    return gx + e, gm


def _leapfrog(x, v, m, eps2, mw, dt, steps):
    """[(x, v, a)] of every state of the KDK run."""
    a = _direct(x, m, eps2, mw)
    states = [(x, v, a)]
    for _ in range(steps):
        v = v + 0.5 * dt * a
        x = x + dt * v
        a = _direct(x, m, eps2, mw)
        v = v + 0.5 * dt * a
        states.append((x, v, a))
    return states


def _exact_hist(case, seed):
    """Counts and histograms 1 to 7 (six rounds of outlier rejection at 2.5 sigma, correction
    1.111) of the baryons, per bin."""
    n, hp = case["n"], _hist_params(case)
    pos, vel, _ = _stream(n, seed)
    x, v = pos[: n // 2] + torch.tensor([8.0, 0.0, 0.0], device="cuda", dtype=pos.dtype), vel[: n // 2]
    f, t, s = (math.radians(a) for a in (hp.phi, hp.theta, hp.psi))
    cf, sf, ct, st, cs, ss = (math.cos(f), math.sin(f), math.cos(t), math.sin(t), math.cos(s),
                              math.sin(s))

    def frame(rows):
        return torch.tensor(rows, device="cuda", dtype=x.dtype).T

    y = x @ frame([[cs * cf - ct * sf * ss, cs * sf + ct * cf * ss, ss * st],
                   [-ss * cf - ct * sf * cs, -ss * sf + ct * cf * cs, cs * st],
                   [st * sf, -st * cf, ct]])
    dist = torch.linalg.norm(x, dim=1)
    lam = torch.rad2deg(torch.atan2(y[:, 1], y[:, 0]))
    beta = torch.rad2deg(torch.asin(-y[:, 2] / torch.linalg.norm(y, dim=1)))
    li = torch.floor((lam + 150.0) / (300.0 / hp.lambdaBins))
    bi = torch.floor((beta + 15.0) / (30.0 / hp.betaBins))
    ok = (li >= 0) & (li < hp.lambdaBins) & (bi >= 0) & (bi < hp.betaBins)
    nbin = hp.lambdaBins * hp.betaBins
    b = (li * hp.betaBins + bi)[ok].long()
    vlos = ((x * v).sum(1) / dist)[ok]
    # proper motions in the equatorial frame
    l, d, a = math.pi - math.radians(123.0), math.pi / 2 - math.radians(27.4), math.radians(192.0)
    cl, sl, cd, sd, ca, sa = (math.cos(l), math.sin(l), math.cos(d), math.sin(d), math.cos(a),
                              math.sin(a))
    eq = frame([[ca * cd * cl - sa * sl, -ca * cd * sl - sa * cl, ca * sd],
                [sa * cd * cl + ca * sl, -sa * cd * sl + ca * cl, sa * sd],
                [-sd * cl, sd * sl, cd]])
    p = (x @ eq)[ok]
    u = ((v - torch.tensor(nb.SUN_VEL, device="cuda", dtype=x.dtype)) @ eq)[ok]
    rho, r = torch.linalg.norm(p[:, :2], dim=1), torch.linalg.norm(p, dim=1)
    c, sn, sz, cz = p[:, 0] / rho, p[:, 1] / rho, p[:, 2] / r, rho / r
    mas = 180.0 / math.pi * 3600.0 / 1e6
    mudec = (-u[:, 0] * c * sz - u[:, 1] * sn * sz + u[:, 2] * cz) / r * mas
    mura = (-u[:, 0] * sn + u[:, 1] * c) / r * mas
    raw = torch.bincount(b, minlength=nbin).double()
    var, ave = {}, {}
    for k, q in {"beta": beta[ok], "vlos": vlos, "dist": dist[ok], "dec": mudec, "ra": mura}.items():
        sig, err = torch.zeros(nbin, device="cuda", dtype=x.dtype), torch.zeros(nbin, device="cuda", dtype=x.dtype)
        keep = torch.ones_like(b, dtype=torch.bool)
        for rnd in range(7):
            if rnd:
                keep = (mean[b] - q).abs() < 2.5 * sig[b]
            cnt = torch.bincount(b[keep], minlength=nbin).double()
            tot = torch.bincount(b[keep], weights=q[keep], minlength=nbin)
            sq = torch.bincount(b[keep], weights=q[keep] ** 2, minlength=nbin)
            mean = tot / cnt
            var2 = (sq / (cnt - 1) - cnt / (cnt - 1) * mean ** 2) * (1.111 if rnd else 1.0)
            new = torch.sqrt(var2)
            sig, err = torch.where(cnt > 10, new, sig), torch.where(cnt > 10, torch.sqrt((cnt + 1) / (cnt * (cnt - 1))) * new, err)
        var[k] = (sig, err)
        ave[k] = (torch.where(cnt > 10, mean, torch.zeros_like(mean)),
                  torch.where(cnt > 10, sig / torch.sqrt(cnt), -torch.ones_like(mean)))
    out = [raw.long().reshape(1, -1), torch.tensor([int(ok.sum())])]
    for pair in (var["beta"], var["vlos"], ave["vlos"], ave["beta"], ave["dist"], ave["dec"], ave["ra"]):
        out += list(pair)
    return [o.cpu() for o in out]


def exact(case, seed):
    kind = case["kind"]
    n = case.get("n", 0)
    with torch.no_grad():
        if kind == "run" and n <= 110000 and float(n) * n * (case["steps"] + 1) <= 1.3e11:
            x, v, m = _dwarf(n, seed, case["dark"], case["mw"])
            dt = 4.0 / math.ceil(4.0 / DT)
            out = _leapfrog(x, v, m, case["eps2"], case["mw"], dt, case["steps"])[-1]
            return out if case["precision"] == "fp64" else out[:2]
        if kind == "batch" and case["sims"] * float(case["hi"]) ** 2 <= 1.1e11:
            dt = 4.0 / math.ceil(4.0 / DT)
            ends = [_leapfrog(*b, e, True, dt, case["steps"])[-1] for b, e in _members(case, seed)]
            out = tuple(torch.cat(t) for t in zip(*ends))
            return out if case["precision"] == "fp64" else out[:2]
        if kind == "adjoint":
            x, v, m = _dwarf(n, seed)
            dt, eps2 = DT, case["eps2"]
            states = _leapfrog(x, v, m, eps2, True, dt, case["steps"])
            gx, gv = _grads(case, seed)
            gm, ga, gdt = torch.zeros_like(m), torch.zeros_like(x), 0.0
            for k in range(case["steps"], 0, -1):
                x1, _, a1 = states[k]
                _, v0, a0 = states[k - 1]
                ga = ga + 0.5 * dt * gv
                gdt += 0.5 * (a1 * gv).sum()
                dx, dm = _direct_vjp(x1, m, eps2, ga)
                gx, gm = gx + dx, gm + dm
                gh = gv + dt * gx
                gdt += ((v0 + 0.5 * dt * a0) * gx).sum() + 0.5 * (a0 * gh).sum()
                gv, ga = gh, 0.5 * dt * gh
            dx, dm = _direct_vjp(states[0][0], m, eps2, ga)
            return list(states[-1][:2]) + [gx + dx, gv, gm + dm, torch.as_tensor(gdt)]
        if kind == "hist":
            return _exact_hist(case, seed)
    return None

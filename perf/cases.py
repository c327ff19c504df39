"""Performance cases of the force and integration library: what a program that
uses it has it do, through the public Python binding, from the smallest calls
to the largest. `listed()` names them, `draw()` gives more of the same ranges,
`prepare()` makes the inputs and the context, `run()` is one pass, `work()`
what the pass cannot do without and `exact()` its outputs in plain FP64.

Kinds of pass:
  steps     load a state from device tensors, advance it, read it back
  report    the same through the integration report (energies before and after)
  ensemble  advance a loaded ensemble of small systems, read it back
  fit       trajectory forward and gradients of a snapshot loss (one system)
  fits      the same for an ensemble of three-body systems
"""
import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

import aster_amd as A

METHODS = {"mixed": A.ALLPAIRS_FP32_KAHAN, "fp32": A.ALLPAIRS_FP32, "fp64": A.ALLPAIRS_FP64,
           "group": A.BH_GROUP, "parity": A.BH_PARITY}
INTEGRATORS = {"leapfrog": A.LEAPFROG, "yoshida4": A.YOSHIDA4, "saba4": A.SABA, "wh": A.WH_PLANETARY}
YOSHIDA = (1.3512071919596578, -1.7024143839193153, 1.3512071919596578)


def _steps(name, n, method, integrator, nsteps, dt, **kw):
    return dict(dict(name=name, kind="steps", n=n, ic="plummer", method=method, integrator=integrator, nsteps=nsteps,
                     dt=dt, soft=2.5e-5, theta=0.5, pn1=False, c=1e4), **kw)


def _ensemble(name, nsys, nmax, integrator, nsteps, dt, **kw):
    return dict(dict(name=name, kind="ensemble", nsys=nsys, nmin=3, nmax=nmax, integrator=integrator, nsteps=nsteps,
                     dt=dt, pn1=True, c=1e4, exact_order=False), **kw)


def listed():
    return [
        # A small cluster between two frames of a program that shows or steers it: every launch counts.
        _steps("allpairs_1000_mixed", 1000, "mixed", "leapfrog", 16, 1e-3),
        # The reference's own CPU-sized run, bit-compatible FP64, with its energy report.
        _steps("report_4096_fp64", 4096, "fp64", "leapfrog", 10, 1e-3, kind="report", soft=1e-4),
        # A mid-sized odd body count in plain FP32 through a higher-order integrator, handed on as FP32 (a viewer).
        _steps("allpairs_20011_fp32_saba4", 20011, "fp32", "saba4", 2, 1e-3),
        # The mixed-precision configuration: 65536 bodies, fourth order.
        _steps("allpairs_65536_mixed_yoshida", 65536, "mixed", "yoshida4", 2, 2.5e-4),
        # The Barnes-Hut configuration: 2^20 bodies, 10 steps.
        _steps("bh_1m_group", 1 << 20, "group", "leapfrog", 10, 5e-4, ic="mixed"),
        # A small Barnes-Hut run at a wide angle, where the tree costs as much as the walk.
        _steps("bh_50000_group_wide", 50000, "group", "leapfrog", 10, 5e-4, ic="mixed", theta=0.7),
        # Barnes-Hut with first post-Newtonian terms, odd body count.
        _steps("bh_100003_group_pn1", 100003, "group", "leapfrog", 2, 5e-4, ic="mixed", pn1=True, c=100.0),
        # The reference's default solver (its own opening test, FP64, bit-compatible), odd body count.
        _steps("bh_150001_parity_fp64", 150001, "parity", "leapfrog", 4, 5e-4, ic="mixed"),
        # The ensemble configuration: 8192 planetary systems with 1PN terms, between two snapshots.
        _ensemble("ensemble_8192_pn1", 8192, 64, "yoshida4", 200, 1e-3),
        # A smaller ensemble in the reference's operation order.
        _ensemble("ensemble_1000_exact", 1000, 64, "leapfrog", 200, 1e-3, exact_order=True, pn1=False),
        # One gradient of a trajectory fit: forward, loss, backward.
        dict(name="fit_16384", kind="fit", n=16384, nsteps=32, ckpt=8, nsnap=4, dt=1e-3, soft=2.5e-5),
        # Thousands of three-body fits at once.
        dict(name="fits_4096_threebody", kind="fits", nsys=4096, nsteps=200, nsnap=4, dt=1e-3, soft=1e-2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["allpairs", "allpairs", "report", "bh", "bh", "ensemble", "fit", "fits"])
    if kind in ("allpairs", "report"):
        method = rng.choice(["mixed", "fp32", "fp64"])
        n = _log_int(rng, 64, 16384 if method == "fp64" else 65536)
        nsteps = max(1, min(16, int(4e9 / n / n) if method == "mixed" else int(1e9 / n / n)))
        c = _steps("", n, method, rng.choice(["leapfrog", "yoshida4", "saba4"]), nsteps, 1e-3 if n < 32768 else 2.5e-4)
        if kind == "report":
            c["kind"] = "report"
    elif kind == "bh":
        method = rng.choice(["group", "group", "parity"])
        pn1 = method == "group" and rng.random() < 0.25
        n = _log_int(rng, 2000, 1 << (17 if pn1 else 19))
        c = _steps("", n, method, "leapfrog", 2 if pn1 else rng.randint(2, 8), 5e-4, ic=rng.choice(["mixed", "plummer"]),
                   theta=round(rng.uniform(0.35, 0.75), 3), pn1=pn1, c=100.0)
    elif kind == "ensemble":
        integrator = rng.choice(["leapfrog", "yoshida4", "wh"])
        exact_order = rng.random() < 0.4
        c = _ensemble("", _log_int(rng, 64, 4096), rng.randint(4, 64), integrator, rng.randint(40, 100),
                      2e-2 if integrator == "wh" else 1e-3, exact_order=exact_order,
                      pn1=integrator != "wh" and rng.random() < 0.5)
    elif kind == "fit":
        n = _log_int(rng, 200, 32768)
        c = dict(kind="fit", n=n, nsteps=8 * (1 if n > 8192 else rng.randint(1, 6)), ckpt=rng.choice([4, 8]),
                 nsnap=rng.randint(1, 4), dt=1e-3, soft=2.5e-5)
    else:
        c = dict(kind="fits", nsys=_log_int(rng, 64, 8192), nsteps=rng.randint(40, 200), nsnap=rng.randint(1, 4),
                 dt=1e-3, soft=1e-2)
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ inputs --

def _unit(rng, n):
    z = rng.uniform(-1.0, 1.0, n)
    p = rng.uniform(0.0, 2 * np.pi, n)
    s = np.sqrt(1.0 - z * z)
    return np.stack([s * np.cos(p), s * np.sin(p), z], 1)


def _plummer(n, rng, mtot=1.0, log_masses=False):
    """Plummer sphere in virial equilibrium, scale radius 1, r <= 10 (Aarseth, Henon & Wielen 1974)."""
    umax = (1.0 + 1.0 / 100.0) ** -1.5
    r = 1.0 / np.sqrt((rng.uniform(0.0, 1.0, n) * umax + 1e-12) ** (-2.0 / 3.0) - 1.0)
    q = np.zeros(n)
    todo = np.arange(n)
    while todo.size:
        a, b = rng.uniform(0.0, 1.0, todo.size), rng.uniform(0.0, 0.1, todo.size)
        ok = b < a * a * (1.0 - a * a) ** 3.5
        q[todo[ok]] = a[ok]
        todo = todo[~ok]
    pos = r[:, None] * _unit(rng, n)
    vel = (q * np.sqrt(2.0 * mtot) * (1.0 + r * r) ** -0.25)[:, None] * _unit(rng, n)
    mass = 10.0 ** rng.uniform(0.0, 2.0, n) if log_masses else np.ones(n)
    mass = mass * (mtot / mass.sum())
    pos -= (mass[:, None] * pos).sum(0) / mtot
    vel -= (mass[:, None] * vel).sum(0) / mtot
    return pos, vel, mass


def _bodies(case, seed):
    n, rng = case["n"], np.random.default_rng([seed, 1])
    if case.get("ic") != "mixed":
        return _plummer(n, rng, log_masses=True)
    # half a Plummer sphere, half a uniform cube at rest, equal masses
    h = n // 2
    p, v, _ = _plummer(h, rng, mtot=0.5)
    pos = np.concatenate([p, rng.uniform(-4.0, 4.0, (n - h, 3))])
    vel = np.concatenate([v, np.zeros((n - h, 3))])
    return pos, vel, np.full(n, 1.0 / n)


def _systems(case, seed):
    """Planetary systems about a unit mass: masses log-uniform in [1e-7, 1e-3], semi-major axes log-uniform in
    [0.4, 30], eccentricities up to 0.3, inclinations up to 5 degrees; barycentric. The sizes are the case's own."""
    rng = np.random.default_rng([seed, 2])
    sizes = np.random.default_rng(case["nsys"]).integers(case["nmin"], case["nmax"] + 1, case["nsys"])
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    n = int(off[-1])
    m = 10.0 ** rng.uniform(-7.0, -3.0, n)
    a = np.exp(rng.uniform(math.log(0.4), math.log(30.0), n))
    e, inc = rng.uniform(0.0, 0.3, n), np.radians(rng.uniform(0.0, 5.0, n))
    node, peri, anom = (rng.uniform(0.0, 2 * np.pi, n) for _ in range(3))
    E = anom.copy()
    for _ in range(12):
        E = E - (E - e * np.sin(E) - anom) / (1.0 - e * np.cos(E))
    cn, sn, cw, sw, ci, si = np.cos(node), np.sin(node), np.cos(peri), np.sin(peri), np.cos(inc), np.sin(inc)
    P = np.stack([cn * cw - sn * sw * ci, sn * cw + cn * sw * ci, sw * si], 1)
    Q = np.stack([-cn * sw - sn * cw * ci, -sn * sw + cn * cw * ci, cw * si], 1)
    b, rate = np.sqrt(1.0 - e * e), np.sqrt(1.0 / a) / (1.0 - e * np.cos(E))
    pos = (a * (np.cos(E) - e))[:, None] * P + (a * b * np.sin(E))[:, None] * Q
    vel = (-rate * np.sin(E))[:, None] * P + (rate * b * np.cos(E))[:, None] * Q
    first = off[:-1]
    m[first] = 1.0
    pos[first] = 0.0
    vel[first] = 0.0
    sys = np.repeat(np.arange(case["nsys"]), sizes)
    tot = np.add.reduceat(m, first)
    for w in (pos, vel):
        w -= (np.add.reduceat(m[:, None] * w, first) / tot[:, None])[sys]
    return off, pos, vel, m


def _three(case, seed):
    rng = np.random.default_rng([seed, 3])
    k = case["nsys"]
    m = rng.uniform(0.5, 1.5, (k, 3))
    x, v = rng.uniform(0.0, 1.0, (k, 3, 3)), rng.uniform(-0.5, 0.5, (k, 3, 3))
    v -= (m[:, :, None] * v).sum(1, keepdims=True) / m.sum(1)[:, None, None]
    return np.arange(k + 1, dtype=np.int64) * 3, x.reshape(-1, 3), v.reshape(-1, 3), m.reshape(-1)


def _snaps(case):
    k = case["nsnap"]
    return np.array([(q + 1) * case["nsteps"] // k for q in range(k)], np.int64)


def _target(case, seed, pos):
    """Observed positions that a fit compares its snapshots with."""
    rng = np.random.default_rng([seed, 4])
    return pos[None] + rng.normal(scale=1e-2, size=(case["nsnap"],) + pos.shape)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def prepare(case, seed):
    kind = case["kind"]
    ctx = A.Context(torch.cuda.current_device())
    st = dict(case=case, ctx=ctx)
    if kind in ("steps", "report", "fit"):
        pos, vel, mass = _bodies(case, seed)
        ctx.set_params(G=1.0, softening=case["soft"], theta=case.get("theta", 0.5), c=case.get("c", 1e4),
                       pn_flags=A.NEWTON | (A.PN1 if case.get("pn1") else 0),
                       precision=A.FP64 if case.get("method") == "parity" else A.FP32)
        st.update(pos=_dev(pos), vel=_dev(vel), mass=_dev(mass))
        st.update(out_pos=torch.empty_like(st["pos"]), out_vel=torch.empty_like(st["vel"]))
        if kind == "fit":
            st.update(snaps=_snaps(case), target=_target(case, seed, pos))
    else:
        off, pos, vel, mass = _systems(case, seed) if kind == "ensemble" else _three(case, seed)
        ctx.set_params(G=1.0, softening=case.get("soft", 0.0), c=case.get("c", 1e4),
                       pn_flags=A.NEWTON | (A.PN1 if case.get("pn1") else 0),
                       precision=A.FP64 if case.get("exact_order") else A.FP32)
        ctx.batch_set(off, pos, vel, mass)
        if kind == "fits":
            st.update(snaps=_snaps(case), target=_target(case, seed, pos))
    torch.cuda.synchronize()
    return st


# -------------------------------------------------------------------- pass --

def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind == "ensemble":
        ctx.batch_step(INTEGRATORS[case["integrator"]], case["dt"], case["nsteps"])
        return list(ctx.batch_get())
    if kind == "fits":
        snaps = ctx.batch_traj_forward(case["dt"], case["nsteps"], st["snaps"])
        return [snaps] + list(ctx.batch_traj_backward(2.0 * (snaps - st["target"]) / snaps.size))
    n = case["n"]
    ctx.set_state_device(n, st["pos"].data_ptr(), st["vel"].data_ptr(), st["mass"].data_ptr())
    if kind == "fit":
        snaps = ctx.traj_forward(case["dt"], case["nsteps"], case["ckpt"], st["snaps"])
        return [snaps] + list(ctx.traj_backward(2.0 * (snaps - st["target"]) / snaps.size))
    method, integrator = METHODS[case["method"]], INTEGRATORS[case["integrator"]]
    out = []
    if kind == "report":
        r = ctx.integrate_report(method, integrator, case["dt"], case["nsteps"], order=4)
        out = [r["initial_energy"], r["final_energy"]]
    else:
        ctx.integrate(method, integrator, 4, case["dt"], case["nsteps"])
    ctx.get_state_device(st["out_pos"].data_ptr(), st["out_vel"].data_ptr())
    state = [st["out_pos"], st["out_vel"]]
    if case["method"] == "fp32":  # plain FP32 forces: the state is handed on as FP32
        state = [t.float() for t in state]
    return state + out


# -------------------------------------------------------------------- work --

def _evals(case):
    """Force evaluations of a pass over one system."""
    per = {"leapfrog": 1, "yoshida4": 3, "saba4": 4, "wh": 1}[case["integrator"]] * case["nsteps"]
    if case.get("pn1"):
        return 2 * per
    return per + (0 if case["integrator"] == "saba4" else 1)


def work(case):
    kind = case["kind"]
    if kind in ("ensemble", "fits"):
        if kind == "fits":
            n, pairs, evals, per = 3 * case["nsys"], 6 * case["nsys"], case["nsteps"] + 1, 26 + 60
        else:
            lo, hi = case["nmin"], case["nmax"]
            n = case["nsys"] * (lo + hi) / 2
            pairs = case["nsys"] * sum(k * (k - 1) for k in range(lo, hi + 1)) / (hi - lo + 1)
            evals, per = _evals(case), 113 if case["pn1"] else 26
        return {"bytes": 104.0 * n, "flops": float(per) * pairs * evals}
    n = case["n"]
    if kind == "fit":
        return {"bytes": 8.0 * n * (7 + 6 * case["nsnap"] + 7), "flops": n * (n - 1.0) * case["nsteps"] * (20 + 54)}
    if case["method"] == "group":  # list entries per body of the group traversal, from its counters at 2^18..2^22
        per = min(n - 1.0, max(200.0, 2192 + 130 * math.log2(n / 2 ** 20)) * (0.5 / case["theta"]) ** 2.1)
    elif case["method"] == "parity":
        per = 14.5
    else:
        per = n - 1.0
    flops = n * per * _evals(case) * (107 if case["pn1"] else 20)
    if kind == "report":
        flops += 2 * n * (n - 1.0) * 14
    return {"bytes": 104.0 * n, "flops": float(flops)}


# ------------------------------------------------------------------- exact --

def _pair_sum(xt, vt, mt, x, v, m, soft, ic2):
    """Accelerations of targets (xt, vt, mt) from sources (x, v, m), G = 1; a body's own pair adds nothing."""
    dx, dy, dz = (x[..., None, :, k] - xt[..., :, None, k] for k in range(3))
    d2 = dx * dx + dy * dy + dz * dz
    r2 = torch.where(d2 == 0, torch.ones_like(d2), d2 + soft)
    mj = torch.where(d2 == 0, torch.zeros_like(d2), m[..., None, :].expand_as(d2))
    inv = r2.rsqrt()
    w = mj * inv * inv * inv
    a = [(w * d).sum(-1) for d in (dx, dy, dz)]
    if ic2:
        n = [-d * inv for d in (dx, dy, dz)]
        dot = lambda p, q: p[0] * q[0] + p[1] * q[1] + p[2] * q[2]  # noqa: E731
        v1, v2 = [vt[..., :, None, k] for k in range(3)], [v[..., None, :, k] for k in range(3)]
        n1, n2 = dot(n, v1), dot(n, v2)
        s = -dot(v1, v1) - 2 * dot(v2, v2) + 4 * dot(v1, v2) + 1.5 * n2 * n2 + (5 * mt[..., :, None] + 4 * mj) * inv
        t, k = 4 * n1 - 3 * n2, mj * inv * inv * ic2
        a = [a[q] + ((n[q] * s + (v1[q] - v2[q]) * t) * k).sum(-1) for q in range(3)]
    return torch.stack(a, -1)


def _accel(x, v, m, soft, ic2, grad=False):
    if x.dim() == 3:  # [systems, bodies, 3]
        return _pair_sum(x, v, m, x, v, m, soft, ic2)
    n, out = x.shape[0], []
    step = max(16, int(3e7 / n))
    for i in range(0, n, step):
        args = (x[i:i + step], v[i:i + step], m[i:i + step], x, v, m, soft, ic2)
        out.append(checkpoint(_pair_sum, *args, use_reentrant=False) if grad else _pair_sum(*args))
    return torch.cat(out)


def _advance(case, x, v, m):
    soft, dt = case.get("soft", 0.0), case["dt"]
    ic2 = 1.0 / case["c"] ** 2 if case["pn1"] else 0.0
    if case["integrator"] == "saba4":
        nodes, weights = np.polynomial.legendre.leggauss(4)
        nodes = 0.5 * (nodes + 1.0)
        drifts = np.diff(np.concatenate([[0.0], nodes, [1.0]]))
        for _ in range(case["nsteps"]):
            x = x + v * (drifts[0] * dt)
            for k in range(4):
                v = v + _accel(x, v, m, soft, ic2) * (0.5 * weights[k] * dt)
                x = x + v * (drifts[k + 1] * dt)
        return x, v
    a = None
    for _ in range(case["nsteps"]):
        for w in YOSHIDA if case["integrator"] == "yoshida4" else (1.0,):
            h = w * dt
            if a is None or ic2:
                a = _accel(x, v, m, soft, ic2)
            v = v + 0.5 * h * a
            x = x + h * v
            a = _accel(x, v, m, soft, ic2)
            v = v + 0.5 * h * a
    return x, v


def _energy(x, v, m, soft):
    n, pot = x.shape[0], 0.0
    step = max(16, int(3e7 / n))
    for i in range(0, n, step):
        r = sum((x[i:i + step, None, k] - x[None, :, k]) ** 2 for k in range(3)).sqrt()
        w = torch.where(r == 0, torch.zeros_like(r), 1.0 / (r + soft))
        pot += float((m[i:i + step, None] * w * m[None]).sum())
    return float(0.5 * (m[:, None] * v * v).sum()) - 0.5 * pot


def _fit(case, x, v, m, target):
    """Snapshots and gradients of mean((snapshots - target)^2) by automatic differentiation."""
    x0, v0, m0 = (t.clone().requires_grad_() for t in (x, v, m))
    x, v, soft, dt, at, snaps = x0, v0, case["soft"], case["dt"], set(_snaps(case).tolist()), []
    a = _accel(x, v, m0, soft, 0.0, True)
    for s in range(case["nsteps"]):
        v = v + 0.5 * dt * a
        x = x + dt * v
        if s + 1 in at:
            snaps.append(x)
        if s + 1 < case["nsteps"]:
            a = _accel(x, v, m0, soft, 0.0, True)
            v = v + 0.5 * dt * a
    snaps = torch.stack(snaps)
    ((snaps - target) ** 2).mean().backward()
    return snaps.detach(), x0.grad, v0.grad, m0.grad


def exact(case, seed):
    kind = case["kind"]
    if kind == "fits":
        _, pos, vel, mass = _three(case, seed)
        k = case["nsys"]
        target = _dev(_target(case, seed, pos)).reshape(case["nsnap"], k, 3, 3)
        s, gx, gv, gm = _fit(case, _dev(pos).reshape(k, 3, 3), _dev(vel).reshape(k, 3, 3), _dev(mass).reshape(k, 3),
                             target)
        return [s.reshape(case["nsnap"], -1, 3), gx.reshape(-1, 3), gv.reshape(-1, 3), gm.reshape(-1)]
    if kind == "ensemble":
        if case["integrator"] == "wh":
            return None  # the splitting's own error at this step is far above rounding
        off, pos, vel, mass = _systems(case, seed)
        top = int(np.diff(off).max())
        sys = np.repeat(np.arange(case["nsys"]), np.diff(off))
        at = torch.from_numpy(sys * top + np.arange(off[-1]) - off[:-1][sys]).cuda()
        full = []
        for w in (pos, vel, mass):
            f = torch.zeros((case["nsys"] * top,) + w.shape[1:], dtype=torch.float64, device="cuda")
            f[at] = _dev(w)
            full.append(f.reshape((case["nsys"], top) + w.shape[1:]))
        x, v = _advance(case, *full)
        return [t.reshape(-1, 3)[at] for t in (x, v)]
    pos, vel, mass = (_dev(w) for w in _bodies(case, seed))
    if kind == "fit":
        return list(_fit(case, pos, vel, mass, _dev(_target(case, seed, pos.cpu().numpy()))))
    if float(case["n"]) ** 2 * _evals(case) > 3e11:
        return None  # all pairs would take too long; the tree's error against them is reported by the benchmark
    x, v = _advance(case, pos, vel, mass)
    out = [x, v]
    if kind == "report":
        out += [_energy(pos, vel, mass, case["soft"]), _energy(x, v, mass, case["soft"])]
    return out

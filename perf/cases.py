"""Performance cases of the engine: what its users call, at the sizes they call it.

A case is a dict of plain values; ``kind`` names the way the engine is used:

* ``force``  one force evaluation of particles that already live on the GPU
  (``evaluate_device`` of ``HipDirectSolver`` / ``HipTreeSolver``);
* ``host``   the same through ``evaluate`` on host arrays, the ForceSolver seam a
  host integrator calls;
* ``run``    a device-resident system (``DeviceSystem``): ``steps`` steps, then the
  energy line and the frame that a simulation writes at each output;
* ``batch``  many uneven systems stepped together (``DeviceBatch``), then read back;
* ``serve``  a burst of requests through the continuous-batching ``Server``.

Particles are the workload generators' own (Plummer spheres and two-disc
collisions), made from the seed. Masses are equal, as the generators make them,
or spread over a factor of a hundred (``masses="spread"``).
"""
import math

import numpy as np
import torch

import orrery_amd as E
import orrery_amd.workloads as W

# Runs move through the frame: with a bulk velocity every conserved quantity of
# the energy line is a number of its own rather than rounding noise about zero.
BULK = (0.05, -0.02, 0.03)
STATE = ("x", "y", "z", "vx", "vy", "vz", "ax", "ay", "az")


def listed():
    return [
        # A two-body orbit, the smallest simulation there is: launch latency alone.
        dict(name="run_pair", kind="run", solver="direct", model="pair", n=2, integrator="velocity-verlet",
             softening=0.0, timestep=1e-3, steps=100),
        # A small cluster behind a host integrator: one call, host arrays in and out.
        dict(name="host_direct_1000", kind="host", solver="direct", model="plummer", n=1000,
             masses="equal", softening=0.01),
        # The reference's small benchmark system between two outputs.
        dict(name="run_plummer_4096", kind="run", solver="direct", model="plummer", n=4096,
             integrator="velocity-verlet", softening=0.01, timestep=1e-3, steps=20),
        # A mid-sized direct sum with a mass spectrum and a ragged count.
        dict(name="force_direct_20001", kind="force", solver="direct", model="plummer", n=20001,
             masses="spread", softening=0.02),
        # A production direct run: one fourth-order step and its output.
        dict(name="run_plummer_65536", kind="run", solver="direct", model="plummer", n=65536,
             integrator="yoshida4", softening=0.005, timestep=5e-4, steps=1),
        # The headline direct sum.
        dict(name="force_direct_262144", kind="force", solver="direct", model="plummer", n=262144,
             masses="equal", softening=0.005),
        # The reference's tree accuracy setting from host arrays.
        dict(name="host_tree_16384", kind="host", solver="tree", model="plummer", n=16384,
             masses="equal", softening=0.01, theta=0.5, leaf=32, quadrupole=False),
        # The two-galaxy example run, a few steps and an output.
        dict(name="run_collision_60000", kind="run", solver="tree", model="discs", n=60000,
             integrator="velocity-verlet", softening=0.02, timestep=2e-3, steps=5, theta=0.6,
             leaf=32, quadrupole=False),
        # Barnes-Hut with quadrupoles at the cross-check size.
        dict(name="force_tree_262144", kind="force", solver="tree", model="discs", n=262144,
             masses="equal", softening=0.01, theta=0.5, leaf=16, quadrupole=True),
        # The largest Barnes-Hut evaluation the benchmark reports.
        dict(name="force_tree_2097152", kind="force", solver="tree", model="discs", n=2097152,
             masses="equal", softening=0.01, theta=0.5, leaf=16, quadrupole=True),
        # A parameter study: uneven spheres stepped together, direct ones and trees.
        dict(name="batch_48", kind="batch", systems=48, lo=512, hi=16384, sizes=4, softening=0.02,
             timestep=1e-3, steps=20, theta=0.6, leaf=16),
        # A burst of service requests of mixed size.
        dict(name="serve_12", kind="serve", systems=12, lo=256, hi=8192, sizes=7, softening=0.02,
             timestep=1e-3, steps=20, theta=0.5, leaf=16),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _tree_options(rng):
    return dict(theta=round(rng.uniform(0.4, 0.9), 2), leaf=rng.choice([8, 16, 16, 24, 32]),
                quadrupole=rng.random() < 0.5)


def draw(rng):
    kind = rng.choice(["pair", "force", "force", "host", "host", "run", "run", "run", "batch", "serve"])
    tree = rng.random() < 0.5
    eps = round(rng.uniform(0.005, 0.03), 4)
    if kind == "pair":
        n = _log_int(rng, 2, 64)
        return dict(kind="run", solver="direct", model="pair" if n == 2 else "plummer", n=n,
                    integrator=rng.choice(["velocity-verlet", "yoshida4", "runge-kutta4"]),
                    softening=0.0 if n == 2 else eps, timestep=round(rng.uniform(2e-4, 1e-3), 6),
                    steps=rng.randint(50, 150))
    if kind in ("force", "host"):
        out = dict(kind=kind, solver="tree" if tree else "direct",
                   model=rng.choice(["plummer", "discs"]), masses=rng.choice(["equal", "spread"]),
                   softening=eps)
        top = (1000000 if tree else 150000) if kind == "force" else (60000 if tree else 16000)
        out["n"] = _log_int(rng, 1000 if tree else 65, top)
        return out | (_tree_options(rng) if tree else {})
    if kind == "run":
        n = _log_int(rng, 2000 if tree else 128, 200000 if tree else 60000)
        out = dict(kind="run", solver="tree" if tree else "direct",
                   model=rng.choice(["plummer", "discs"]), n=n,
                   integrator=rng.choice(["velocity-verlet", "yoshida4", "runge-kutta4"]),
                   softening=max(eps, 0.01), timestep=round(rng.uniform(2e-4, 2e-3), 6),
                   steps=max(1, min(30, 40000 // n)))
        return out | (_tree_options(rng) if tree else {})
    lo = rng.randint(128, 800)
    return dict(kind=kind, systems=rng.randint(6, 40 if kind == "batch" else 12), lo=lo,
                hi=_log_int(rng, 4 * lo, 16000 if kind == "batch" else 8000), sizes=rng.randrange(1 << 20),
                softening=eps, timestep=round(rng.uniform(2e-4, 1e-3), 6), steps=rng.randint(5, 20),
                theta=round(rng.uniform(0.4, 0.9), 2), leaf=rng.choice([8, 16, 32]))


# ---- inputs ---------------------------------------------------------------


def _pair(seed):
    """Two bodies on an eccentric orbit about their centre of mass, turned by the seed."""
    r = np.random.default_rng(seed)
    m = np.array([1.0, r.uniform(0.2, 1.0)])
    phase, sep, ecc = r.uniform(0, 2 * np.pi), r.uniform(0.8, 1.2), r.uniform(0.0, 0.5)
    u = np.array([np.cos(phase), np.sin(phase), 0.0])
    t = np.array([-np.sin(phase), np.cos(phase), 0.0])
    speed = np.sqrt(m.sum() * (1 - ecc) / sep)  # at apocentre
    share = np.array([-m[1], m[0]]) / m.sum()
    pos, vel = np.outer(u, share) * sep, np.outer(t, share) * speed
    pos[2] += share * 0.1
    return W.Workload(*(np.ascontiguousarray(a) for a in (*pos, *vel)), m)


def _particles(case, seed):
    if case["model"] == "pair":
        return _pair(seed)
    p = (W.plummer if case["model"] == "plummer" else W.disc_collision)(case["n"], seed)
    if case.get("masses") == "spread":
        w = np.random.default_rng(seed + 1).uniform(0.0, 1.0, p.n)
        m = 100.0 ** w
        p.m = m / m.sum()
    return p


def _moving(p):
    for a, u in zip((p.vx, p.vy, p.vz), BULK):
        a += u
    return p


def _spheres(case, seed):
    ns = W.batched_sizes(case["systems"], case["lo"], case["hi"], case["sizes"])
    return [W.plummer(n, seed * 1009 + k) for k, n in enumerate(ns)]


def _solver(case):
    if case["solver"] == "tree":
        return E.HipTreeSolver(E.TreeParameters(case["theta"], case["leaf"], case["quadrupole"]),
                               E.Softening(case["softening"]))
    return E.HipDirectSolver(E.Softening(case["softening"]))


def _step_config(case):
    c = E.StepConfig(integrator=case["integrator"], softening=case["softening"],
                     solver="barnes-hut" if case["solver"] == "tree" else "direct")
    if case["solver"] == "tree":
        c.opening_angle, c.leaf_capacity, c.quadrupole = case["theta"], case["leaf"], case["quadrupole"]
    return c


def prepare(case, seed):
    s = dict(case=case)
    if case["kind"] in ("force", "host"):
        p = _particles(case, seed)
        s["solver"] = _solver(case)
        if case["kind"] == "host":
            s["x"], s["m"], s["a"] = (p.x, p.y, p.z), p.m, [np.zeros(p.n) for _ in range(3)]
        else:
            s["x"] = [torch.from_numpy(a).cuda() for a in (p.x, p.y, p.z)]
            s["m"] = torch.from_numpy(p.m).cuda()
            s["a"] = [torch.zeros_like(s["m"]) for _ in range(3)]
            torch.cuda.synchronize()
        return s
    s["ctx"] = E.Context(0)
    if case["kind"] == "run":
        s["system"], s["config"] = E.DeviceSystem(s["ctx"], case["n"]), _step_config(case)
        s["system"].upload(*_moving(_particles(case, seed)).arrays())
        s["system"].refresh(s["config"])
    elif case["kind"] == "batch":
        spheres = _spheres(case, seed)
        s["batch"] = E.DeviceBatch(
            s["ctx"], [E.BatchSystem(p.n, case["softening"], case["timestep"]) for p in spheres],
            E.BatchConfig(opening_angle=case["theta"], leaf_capacity=case["leaf"]))
        for k, p in enumerate(spheres):
            s["batch"].upload(k, *p.arrays())
        s["batch"].refresh()
    else:
        s["requests"] = _spheres(case, seed)
        s["server"] = E.Server(s["ctx"], E.ServerConfig(opening_angle=case["theta"],
                                                        leaf_capacity=case["leaf"]))
    return s


# ---- one pass -------------------------------------------------------------


def _energy_line(d):
    return np.array([d["kinetic"], d["potential"], d["total"], *d["momentum"], *d["angular_momentum"]])


def run(state):
    case = state["case"]
    if case["kind"] in ("force", "host"):
        solver = state["solver"]
        solver.reset_interaction_count()
        if case["kind"] == "host":
            solver.evaluate(state["x"], state["m"], state["a"])
        else:
            solver.evaluate_device(*(t.data_ptr() for t in (*state["x"], state["m"], *state["a"])), case["n"])
        c = solver.interaction_count()
        return dict(a=state["a"], counts=[c.particle_particle, c.particle_cell])
    if case["kind"] == "run":
        s = state["system"]
        s.step(state["config"], case["timestep"], case["steps"])
        return dict(energy=_energy_line(s.diagnostics(case["softening"])), **s.download())
    if case["kind"] == "batch":
        b = state["batch"]
        b.step(case["steps"])
        frames = [b.download(k) for k in range(case["systems"])]
        return [np.stack([f[a] for a in STATE]) for f in frames]
    server = state["server"]
    ids = [server.submit(p, "velocity-verlet", case["softening"], case["timestep"], case["steps"])
           for p in state["requests"]]
    server.drain()
    out = []
    for rid in ids:
        r, st = server.result(rid), server.status(rid)
        out.append(dict(state=np.stack([r[a] for a in STATE[:6]]),
                        energy=np.array([st["start"]["total"], st["end"]["total"]])))
    return out


# ---- what a pass cannot do without ----------------------------------------

FLOPS_PER_INTERACTION = 20  # the reference's convention
EVALUATIONS = {"velocity-verlet": 1, "yoshida4": 3, "runge-kutta4": 4}


def _interactions(n, solver, theta=0.5, leaf=16):
    """Pairs of a direct sum; for a tree, about 24 theta^-3 cells and particles per
    target and level of eight (3300 per target at theta 0.5 and two million particles)."""
    if solver == "direct":
        return n * (n - 1)
    return min(n * (n - 1), n * 24 / theta**3 * max(1.0, math.log2(max(2.0, n / leaf))))


def work(case):
    if case["kind"] in ("force", "host"):
        inter = _interactions(case["n"], case["solver"], case.get("theta"), case.get("leaf"))
        return dict(bytes=56 * case["n"], flops=FLOPS_PER_INTERACTION * inter)
    if case["kind"] == "run":
        n = case["n"]
        inter = _interactions(n, case["solver"], case.get("theta"), case.get("leaf"))
        inter = inter * EVALUATIONS[case["integrator"]] * case["steps"] + n * (n - 1) / 2
        return dict(bytes=(80 + 72 + 72) * n, flops=FLOPS_PER_INTERACTION * inter)
    ns = W.batched_sizes(case["systems"], case["lo"], case["hi"], case["sizes"])
    inter = sum(_interactions(n, "direct" if n < 4096 else "tree", case["theta"], case["leaf"]) for n in ns)
    inter *= case["steps"]
    if case["kind"] == "serve":  # each request's energy at its start and end
        inter += sum(n * (n - 1) for n in ns)
    return dict(bytes=224 * sum(ns), flops=FLOPS_PER_INTERACTION * inter)


# ---- the same in 64 bits --------------------------------------------------
#
# Forces are the softened direct sum, which is also what a tree approximates: a
# tree's distance from it is its opening angle's truncation.


def _pairs(x, m, eps2, terms):
    """Per chunk of targets: (slice, 1 / r of every pair with the self term zero)."""
    n = m.numel()
    rows = max(1, min(n, (1 << 28) // n))
    for b in range(0, n, rows):
        t = slice(b, min(n, b + rows))
        r2 = torch.full((t.stop - b, n), eps2, dtype=torch.float64, device=m.device)
        for c in range(3):
            d = x[c][None, :] - x[c][t, None]
            r2.addcmul_(d, d)
        k = torch.arange(t.stop - b, device=m.device)
        r2[k, k + b] = math.inf
        terms(t, r2.rsqrt_())


def _field(x, m, eps):
    a = torch.zeros((3, m.numel()), dtype=torch.float64, device=m.device)

    def terms(t, inv):
        f = (inv * inv).mul_(inv).mul_(m[None, :])
        for c in range(3):
            a[c, t] = ((x[c][None, :] - x[c][t, None]).mul_(f)).sum(dim=1)

    _pairs(x, m, eps * eps, terms)
    return a


def _energies(x, v, m, eps):
    pot = torch.zeros_like(m)

    def terms(t, inv):
        pot[t] = inv @ m

    _pairs(x, m, eps * eps, terms)
    ke, pe = 0.5 * (m * (v * v).sum(0)).sum(), -0.5 * (m * pot).sum()
    p, l = (m * v).sum(1), (m * torch.linalg.cross(x.T, v.T).T).sum(1)
    return torch.stack([ke, pe, ke + pe, *p, *l])


def _advance(x, v, m, eps, integrator, dt, steps):
    a = _field(x, m, eps)
    cube = 2.0 ** (1.0 / 3.0)
    weights = [1 / (2 - cube), -cube / (2 - cube), 1 / (2 - cube)] if integrator == "yoshida4" else [1.0]
    for _ in range(steps):
        if integrator == "runge-kutta4":
            kx, kv = [v], [a]
            for h in (dt / 2, dt / 2, dt):
                xs, vs = x + h * kx[-1], v + h * kv[-1]
                kx.append(vs)
                kv.append(_field(xs, m, eps))
            x = x + dt / 6 * (kx[0] + 2 * kx[1] + 2 * kx[2] + kx[3])
            v = v + dt / 6 * (kv[0] + 2 * kv[1] + 2 * kv[2] + kv[3])
            a = _field(x, m, eps)
            continue
        for w in weights:
            v = v + w * dt / 2 * a
            x = x + w * dt * v
            a = _field(x, m, eps)
            v = v + w * dt / 2 * a
    return x, v, a


def _on_gpu(p):
    x, v = (torch.from_numpy(np.stack(c)).cuda() for c in ((p.x, p.y, p.z), (p.vx, p.vy, p.vz)))
    return x, v, torch.from_numpy(p.m).cuda()


def exact(case, seed):
    if case.get("n", 0) > 300000:
        return None  # minutes of pair terms
    if case["kind"] in ("force", "host"):
        x, _, m = _on_gpu(_particles(case, seed))
        return dict(a=list(_field(x, m, case["softening"])), counts=[None, None])
    if case["kind"] == "run":
        evaluations = 1 + EVALUATIONS[case["integrator"]] * case["steps"]
        if evaluations * case["n"] ** 2 > 2e11:
            return None
        x, v, m = _on_gpu(_moving(_particles(case, seed)))
        x, v, a = _advance(x, v, m, case["softening"], case["integrator"], case["timestep"], case["steps"])
        return dict(energy=_energies(x, v, m, case["softening"]), **dict(zip(STATE, (*x, *v, *a))))
    out = []
    for p in _spheres(case, seed):
        x, v, m = _on_gpu(p)
        before = _energies(x, v, m, case["softening"])[2] if case["kind"] == "serve" else None
        x, v, a = _advance(x, v, m, case["softening"], "velocity-verlet", case["timestep"], case["steps"])
        if case["kind"] == "batch":
            out.append(torch.cat([x, v, a]))
        else:
            after = _energies(x, v, m, case["softening"])[2]
            out.append(dict(state=torch.cat([x, v]), energy=torch.stack([before, after])))
    return out

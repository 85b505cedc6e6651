"""The calls that users of the engine make, as cases to be timed and checked.

A case is a dict of plain values. `prepare` makes the engine, the simulation
handles and the initial states a program holds before it calls; `run` is one
pass through the public entry points, from host state in to host state out
(that is how every caller of the library hands bodies over); `exact` is the
same pass in plain 64-bit torch.

Three forms of pass:
* "call": one transform of a host state (the plugin path of a pipeline whose
  other elements run on the CPU);
* "run": a simulation: upload the initial state, step it on the device,
  download the result (with the energy diagnostic where a run is watched);
* "batch" and "served": many simulations of uneven size stepped together,
  through the batch call or through the request server.
"""
import math

import numpy as np
import torch

import physim_amd as P

FIELDS = ("x", "y", "z", "vx", "vy", "vz", "radius", "mass", "id", "fixed")


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # One transform of a small scene with the plugin's benchmark setting:
        # what a CPU pipeline waits for in each of its iterations.
        dict(name="call_cube_1k", form="call", kind="astro2", precision="mixed", model="cube",
             n=1002, theta=1.5, e=0.5),
        # The same call at the benchmark's largest cube: the state crosses to
        # the device and the accelerations come back.
        dict(name="call_cube_1m", form="call", kind="astro2", precision="mixed", model="cube",
             n=1048578, theta=1.5, e=0.5),
        # The all-pairs element on the benchmark's direct-sum size.
        dict(name="call_direct_131k", form="call", kind="simple_astro", precision="mixed",
             model="cube", n=131074, theta=1.0, e=0.5),
        # The reference's own example pipeline: 10,000 bodies and two stars,
        # 100 iterations.
        dict(name="run_cube_10k", form="run", kind="astro2", precision="mixed", model="cube",
             n=10002, theta=1.5, e=0.5, dt=1e-5, steps=100, integrator="verlet", near=0.0,
             energy=False),
        # The headline simulation: the 1M cube for 1000 iterations.
        dict(name="run_cube_1m", form="run", kind="astro2", precision="mixed", model="cube",
             n=1048578, theta=1.5, e=0.5, dt=1e-5, steps=1000, integrator="verlet", near=0.0,
             energy=False),
        # A large served request taken alone: a Plummer sphere at the
        # workload's smallest opening angle, as few steps as it asks for.
        dict(name="run_plummer_262k", form="run", kind="astro2", precision="mixed",
             model="plummer", n=262144, theta=0.5, e=0.01, dt=1e-5, steps=100,
             integrator="verlet", near=0.0, energy=False),
        # The precision study: two colliding spheres with the direct-sum near
        # field of 2 leaf widths.
        dict(name="run_collision_1m", form="run", kind="astro2", precision="mixed",
             model="collision", n=1048576, theta=0.5, e=1e-3, dt=1e-5, steps=20,
             integrator="verlet", near=2.0, energy=False),
        # The reference's FP64 arithmetic over the tree, an odd count.
        dict(name="run_fp64_65k", form="run", kind="astro2", precision="fp64", model="cube",
             n=65539, theta=0.7, e=0.5, dt=1e-5, steps=50, integrator="verlet", near=0.0,
             energy=False),
        # The all-pairs element under rk4 in FP64, watched by the energy
        # diagnostic: what a small reference run is checked with.
        dict(name="run_rk4_direct_8k", form="run", kind="simple_astro", precision="fp64",
             model="plummer", n=8195, theta=1.0, e=0.01, dt=1e-4, steps=5, integrator="rk4",
             near=0.0, energy=True),
        # The quadtree element under euler.
        dict(name="run_euler_quad_50k", form="run", kind="astro", precision="mixed",
             model="cube", n=50003, theta=0.7, e=0.5, dt=1e-5, steps=20, integrator="euler",
             near=0.0, energy=False),
        # Batched ensembles: spheres of uneven size stepped together.
        dict(name="batch_spheres", form="batch", kind="astro2", precision="mixed",
             model="plummer", members=64, n_min=1024, n_max=65536, theta=0.7, e=0.01, dt=1e-4,
             steps=100),
        # Served requests: cubes and spheres of every opening angle admitted
        # together, their steps co-batched 50 at a time.
        dict(name="served_mix", form="served", kind="astro2", precision="mixed", members=12,
             n_min=4096, n_max=131072, theta=0.5, e=0.01, dt=1e-5, steps_min=100,
             steps_max=400),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a form, a kind and an opening angle in earnest use, and
    a size spread over the form's range (over its logarithm; any number)."""
    form = rng.choice(["call", "run", "run", "run", "batch", "served"])
    precision = rng.choice(["mixed", "mixed", "mixed", "fp64"])
    if form == "call":
        kind = rng.choice(["astro2", "astro2", "astro", "simple_astro"])
        top = {"astro2": 1 << 20, "astro": 1 << 18, "simple_astro": 1 << 16}[kind]
        return dict(form="call", kind=kind, precision=precision,
                    model=rng.choice(["cube", "plummer"]), n=_log_int(rng, 300, top),
                    theta=rng.choice([0.5, 0.7, 1.0, 1.5]), e=rng.choice([0.01, 0.5]))
    if form == "run":
        kind = rng.choice(["astro2", "astro2", "astro2", "astro", "simple_astro"])
        integrator = rng.choice(["verlet", "verlet", "verlet", "euler", "rk4"])
        model = rng.choice(["cube", "plummer", "collision"])
        theta = rng.choice([0.5, 0.7, 1.0, 1.5])
        top = {"astro2": 1 << 19, "astro": 1 << 17, "simple_astro": 1 << 14}[kind]
        n = _log_int(rng, 1000, top)
        # (longer runs of smaller systems)
        rate = 1e11 if precision == "mixed" else 5e10
        step_s = 1e-4 + 1e-9 * n + _pairs(kind, n, theta) / rate
        step_s *= 4 if integrator == "rk4" else 1
        steps = max(2, min(200, int(0.1 / step_s)))
        return dict(form="run", kind=kind, precision=precision, model=model, n=n, theta=theta,
                    e=rng.choice([0.001, 0.01, 0.5]), dt=1e-5, steps=steps,
                    integrator=integrator,
                    near=2.0 if model == "collision" and kind == "astro2" else 0.0,
                    energy=n < 20000)
    if form == "batch":
        return dict(form="batch", kind="astro2", precision="mixed", model="plummer",
                    members=rng.randint(2, 64), n_min=1024,
                    n_max=_log_int(rng, 4096, 65536), theta=rng.choice([0.5, 0.7, 1.5]), e=0.01,
                    dt=1e-4, steps=rng.randint(20, 50))
    return dict(form="served", kind="astro2", precision="mixed", members=rng.randint(2, 12),
                n_min=4096, n_max=_log_int(rng, 8192, 131072), theta=0.5, e=0.01, dt=1e-5,
                steps_min=50, steps_max=rng.randint(100, 300))


# ------------------------------------------------------------- initial states
def _entities(pos, vel, mass, radius):
    s = np.zeros(len(pos), P.ENTITY)
    for k, f in enumerate("xyz"):
        s[f] = pos[:, k]
        s["v" + f] = vel[:, k]
    s["mass"] = mass
    s["radius"] = radius
    s["id"] = np.arange(len(pos))
    return s


def _cube(rng, n, stars=True):
    """The rotating cube (spin 1000, total mass 1) and its two stars of 1e5."""
    m = n - 2 if stars else n
    pos = np.concatenate([rng.uniform(-1.0, 1.0, (m, 2)), rng.uniform(0.0, 1.0, (m, 1))], 1)
    vel = np.stack([pos[:, 1] * 1000.0, -pos[:, 0] * 1000.0, np.zeros(m)], 1)
    mass, radius = np.full(m, 1.0 / m), np.full(m, 0.02)
    if stars:
        pos = np.concatenate([pos, [[0.2, 0.2, 0.5], [-0.2, -0.2, 0.5]]])
        vel = np.concatenate([vel, np.zeros((2, 3))])
        mass, radius = np.append(mass, [1e5, 1e5]), np.append(radius, [0.1, 0.1])
    return _entities(pos, vel, mass, radius)


def _directions(rng, n):
    z, a = rng.uniform(-1.0, 1.0, n), rng.uniform(0.0, 2.0 * math.pi, n)
    s = np.sqrt(1.0 - z * z)
    return np.stack([s * np.cos(a), s * np.sin(a), z], 1)


def _plummer(rng, n, mass=1.0, a=0.1, centre=(0.0, 0.0, 0.0), v=(0.0, 0.0, 0.0)):
    """An isotropic Plummer sphere in virial equilibrium (squared speeds over
    the escape speed's are Beta(3/2, 9/2) distributed)."""
    r = a / np.sqrt(rng.uniform(1e-9, 1.0, n) ** (-2.0 / 3.0) - 1.0)
    speed = np.sqrt(rng.beta(1.5, 4.5, n) * 2.0 * mass / np.sqrt(r * r + a * a))
    pos = _directions(rng, n) * r[:, None] + np.asarray(centre)
    vel = _directions(rng, n) * speed[:, None] + np.asarray(v)
    return _entities(pos, vel, np.full(n, mass / n), np.full(n, 0.01))


def _collision(rng, n):
    """Two Plummer spheres, masses 1.0 and 0.1, 1.0 apart, closing at 0.5."""
    n1 = int(round(n * 10 / 11))
    m1, m2 = 1.0, 0.1
    return P.concat([
        _plummer(rng, n1, m1, centre=(-0.5, 0.0, 0.0), v=(0.5 * m2 / (m1 + m2), 0.0, 0.0)),
        _plummer(rng, n - n1, m2, centre=(0.5, 0.0, 0.0), v=(-0.5 * m1 / (m1 + m2), 0.0, 0.0)),
    ])


def _state(model, rng, n):
    return {"cube": _cube, "plummer": _plummer, "collision": _collision}[model](rng, n)


def _members(case, seed):
    """The simulations of a batch or served case: dicts of state, theta, steps."""
    # (sizes, angles and lengths belong to the case; the states to the seed)
    plan = np.random.default_rng([case["members"], case["n_max"]])
    out = []
    for i in range(case["members"]):
        n = int(round(math.exp(plan.uniform(math.log(case["n_min"]), math.log(case["n_max"])))))
        if case["form"] == "batch":
            out.append(dict(n=n, theta=case["theta"], steps=case["steps"], model="plummer"))
        else:
            out.append(dict(n=n, theta=(0.5, 0.7, 1.5)[int(plan.integers(3))],
                            steps=int(plan.integers(case["steps_min"], case["steps_max"] + 1)),
                            model=("cube", "plummer")[int(plan.integers(2))]))
        if seed is not None:
            rng = np.random.default_rng([seed, i])
            out[-1]["state"] = (_cube(rng, n, stars=False) if out[-1]["model"] == "cube"
                                else _plummer(rng, n))
    return out


# ------------------------------------------------------------ prepare and run
def prepare(case, seed):
    """An engine, the handles and the initial host states, as a program holds
    them; the states differ by seed."""
    eng = P.Engine(0)
    s = dict(case=case, engine=eng)
    if case["form"] in ("call", "run"):
        s["state"] = _state(case["model"], np.random.default_rng(seed), case["n"])
    if case["form"] == "run":
        s["sim"] = P.Sim(eng, n=case["n"], kind=case["kind"], theta=case["theta"], e=case["e"],
                         dt=case["dt"], precision=case["precision"],
                         integrator=case["integrator"])
        if case["near"]:
            s["sim"].set_near_field(case["near"])
    if case["form"] in ("batch", "served"):
        s["members"] = _members(case, seed)
    if case["form"] == "batch":
        s["sims"] = [P.Sim(eng, n=m["n"], kind=case["kind"], theta=m["theta"], e=case["e"],
                           dt=case["dt"], precision=case["precision"]) for m in s["members"]]
    if case["form"] == "served":
        s["server"] = P.Server(eng)
    return s


def _phase(state):
    """Positions and velocities of an Entity array, (n, 6)."""
    return state.view(np.float64).reshape(len(state), 10)[:, :6]


def run(s):
    case = s["case"]
    if case["form"] == "call":
        a = s["engine"].transform(s["state"], kind=case["kind"], theta=case["theta"],
                                  e=case["e"], precision=case["precision"])
        return a.view(np.float64).reshape(-1, 3)
    if case["form"] == "run":
        sim = s["sim"]
        sim.upload(s["state"])
        sim.step(case["steps"])
        out = sim.download()
        out = {f: out[f] for f in FIELDS}
        if case["energy"]:
            out["energy"] = sim.energy()
        return out
    if case["form"] == "batch":
        for m, sim in zip(s["members"], s["sims"]):
            sim.upload(m["state"])
        s["engine"].batch_step(s["sims"], case["steps"])
        return [_phase(sim.download()) for sim in s["sims"]]
    srv = s["server"]
    ids = [srv.submit(m["state"], m["steps"], kind=case["kind"], theta=m["theta"], e=case["e"],
                      dt=case["dt"], precision=case["precision"]) for m in s["members"]]
    active = queued = 1
    while active or queued:
        active, queued = srv.tick(50)
    return [_phase(srv.take(i, m["n"])[0]) for i, m in zip(ids, s["members"])]


# ------------------------------------------------------------------------ work
def _pairs(kind, n, theta):
    """About how many pair terms one force pass of n bodies takes: all of
    them, or cells on each tree level with bodies in it (about 65 a level at an
    opening angle of 0.5, 10 at 0.7; from about 1 on a body's own ancestors are
    taken whole, and 1 or 2 pairs are left)."""
    if kind == "simple_astro":
        return n * float(n)
    per_level = (65.0 if kind == "astro2" else 10.0) * (0.5 / theta) ** 5
    levels = max(1.0, math.log(max(n, 2)) / math.log(8 if kind == "astro2" else 4))
    return n * max(1.5, per_level * levels)


def _pass_bytes(kind, n, mixed_tree_nodes=0.48):
    """Bytes one step cannot do without: position, history and mass read, the
    new state written; over a tree also the keys and indices sorted (written
    and read once) and the internal nodes written and read once."""
    state = (24 + 24 + 8 + 24 + 24) * n
    return state if kind == "simple_astro" else state + (2 * 12 + 2 * 64 * mixed_tree_nodes) * n


def _moves(case):
    """(n, theta, force passes) of each simulation of a case."""
    if case["form"] == "call":
        return [(case["n"], case["theta"], 1)]
    if case["form"] == "run":
        per = 4 if case["integrator"] == "rk4" else 1
        return [(case["n"], case["theta"], case["steps"] * per)]
    return [(m["n"], m["theta"], m["steps"]) for m in _members(case, None)]


def work(case):
    """Bytes and operations of one pass (20 operations per pair term): the
    host states in and out, and each force pass with its update."""
    b = f = 0.0
    for n, theta, passes in _moves(case):
        b += (80 + (24 if case["form"] == "call" else 80)) * n
        b += passes * _pass_bytes(case["kind"], n)
        f += passes * 20.0 * _pairs(case["kind"], n, theta)
        if case.get("energy"):
            f += 20.0 * n * n
    return {"bytes": b, "flops": f}


# ----------------------------------------------------------------------- exact
# The same passes in plain 64-bit torch: the Barnes-Hut sum by expanding
# (body, cell) pairs level by level, the all-pairs sum by blocks of rows.
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _levels(pos, mass, dim, order_levels):
    """The tree over `pos` level by level: bodies sorted along the digits of
    the descent (octant bit set where the coordinate exceeds the cell's
    centre), and for each level the cell of each body, the cells' first
    bodies, counts, centres, masses and centres of mass."""
    extent = float(pos.abs().max())
    n = len(pos)
    key = torch.zeros(n, dtype=torch.int64, device=pos.device)
    c = torch.zeros(n, dim, dtype=torch.float64, device=pos.device)
    h, digits = extent, []
    for _ in range(order_levels):
        up = pos[:, :dim] > c
        o = torch.zeros_like(key)
        for a in range(dim):
            o |= up[:, a].to(torch.int64) << a
        key = (key << dim) | o
        digits.append(up)
        h = h / 2.0
        c = torch.where(up, c + h, c - h)
    order = torch.argsort(key)
    pos, mass, key = pos[order], mass[order], key[order]
    # the cells of every level, then their mass sums from the finest level up
    # (few terms each: a sum over all bodies of the root would collide)
    c = torch.zeros(n, dim, dtype=torch.float64, device=pos.device)
    h, out = extent, []
    leaf = torch.full((n,), order_levels, dtype=torch.int64, device=pos.device)
    for lv in range(order_levels + 1):
        k = key >> (dim * (order_levels - lv))
        new = torch.ones(n, dtype=torch.bool, device=pos.device)
        new[1:] = k[1:] != k[:-1]
        cell = torch.cumsum(new, 0) - 1
        first = torch.nonzero(new).flatten()
        count = torch.diff(first, append=torch.tensor([n], device=pos.device))
        alone = count == 1
        centre = torch.zeros(len(first), 3, dtype=torch.float64, device=pos.device)
        centre[:, :dim] = c[first]
        leaf = torch.where(alone[cell] & (leaf == order_levels), torch.full_like(leaf, lv), leaf)
        out.append(dict(cell=cell, first=first, count=count, centre=centre,
                        hw=extent / 2.0 ** lv, alone=alone))
        if bool(alone.all()):
            break
        if lv < order_levels:
            h = h / 2.0
            up = digits[lv][order]
            c = torch.where(up, c + h, c - h)
    part, at = torch.cat([mass[:, None], pos * mass[:, None]], 1), None
    for t in reversed(out):
        at = t["cell"] if at is None else t["cell"][at]
        part = torch.zeros(len(t["first"]), 4, dtype=torch.float64,
                           device=pos.device).index_add_(0, at, part)
        t["mass"] = torch.where(t["alone"], mass[t["first"]], part[:, 0])
        t["com"] = torch.where(t["alone"][:, None], pos[t["first"]], part[:, 1:] / part[:, :1])
        at = t["first"]
    return order, pos, mass, out, leaf


def _add_pairs(acc, body, pos, src, m, e):
    """acc[body] += the pair terms of (body, source) pairs, body ascending."""
    d = src - pos[body]
    s = d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2]
    w = torch.where(s > 0, m / (torch.sqrt(s) * (s + e)), torch.zeros_like(s))
    if len(body):
        who, num = torch.unique_consecutive(body, return_counts=True)
        for a in range(3):
            acc[who, a] += torch.segment_reduce(d[:, a] * w, "sum", lengths=num)


def _tree_acc(pos, mass, kind, theta, e, near):
    dim = 3 if kind == "astro2" else 2
    order, pos, mass, levels, leaf = _levels(pos, mass, dim, 21 if dim == 3 else 31)
    acc = torch.zeros_like(pos)
    n = len(pos)
    extent = levels[0]["hw"]
    step = 1 << (17 if theta < 1.0 else 20)
    for b0 in range(0, n, step):
        body = torch.arange(b0, min(n, b0 + step), device=pos.device)
        cell = torch.zeros_like(body)
        for lv, t in enumerate(levels):
            d = pos[body] - t["centre"][cell]
            r = torch.sqrt(d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2])
            take = t["hw"] / r < theta
            if near:
                reach = t["hw"] + near * (extent * 2.0) / 2.0 ** leaf[body].double()
                close = (d[:, :dim].abs() < reach[:, None]).all(1)
                take &= ~((lv >= leaf[body]) & (lv <= leaf[body] + 2) & close)
            take |= t["alone"][cell]
            tb, tc = body[take], cell[take]
            _add_pairs(acc, tb, pos, t["com"][tc], t["mass"][tc], e)
            body, cell = body[~take], cell[~take]
            if not len(body):
                break
            start, cnt = t["first"][cell], t["count"][cell]
            if lv + 1 < len(levels):
                nxt = levels[lv + 1]["cell"]
                lo, hi = nxt[start], nxt[start + cnt - 1]
            else:  # (cells past the last level: their bodies)
                lo, hi = start, start + cnt - 1
            num = hi - lo + 1
            body = torch.repeat_interleave(body, num)
            at = torch.arange(len(body), device=pos.device)
            at -= torch.repeat_interleave(torch.cumsum(num, 0) - num, num)
            cell = torch.repeat_interleave(lo, num) + at
            if lv + 1 == len(levels):
                _add_pairs(acc, body, pos, pos[cell], mass[cell], e)
    out = torch.empty_like(acc)
    out[order] = acc
    return out


def _direct_acc(pos, mass, e):
    n = len(pos)
    acc = torch.empty_like(pos)
    rows = max(1, (1 << 27) // n)
    for i in range(0, n, rows):
        d = [pos[None, :, a] - pos[i:i + rows, a, None] for a in range(3)]
        s = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        w = torch.where(s > 0, mass[None, :] / (torch.sqrt(s) * (s + e)), torch.zeros_like(s))
        for a in range(3):
            acc[i:i + rows, a] = (d[a] * w).sum(1)
    return acc


def _energy(pos, vel, mass, e):
    n, se = len(pos), math.sqrt(e)
    v = 0.0
    for i in range(0, n, 1024):
        d = pos[None, :, :] - pos[i:i + 1024, None, :]
        r = torch.sqrt((d * d).sum(-1))
        mm = mass[None, :] * mass[i:i + 1024, None]
        u = torch.where(r > 0, -(mm / se) * torch.atan(se / r), torch.zeros_like(r))
        v += 0.5 * float(u.sum())
    k = float((0.5 * mass * (vel * vel).sum(1)).sum())
    p = (mass[:, None] * vel).sum(0).tolist()
    return np.array([k, v, k + v] + p)


def _fields(state):
    dev = _device()
    get = lambda *f: torch.from_numpy(np.stack([state[k] for k in f], 1)).to(dev)  # noqa: E731
    return get("x", "y", "z"), get("vx", "vy", "vz"), get("mass")[:, 0]


def _simulate(state, case, theta, steps, integrator="verlet", near=0.0):
    pos, vel, mass = _fields(state)
    dt = case["dt"]

    def force(p):
        if case["kind"] == "simple_astro":
            return _direct_acc(p, mass, case["e"])
        return _tree_acc(p, mass, case["kind"], theta, case["e"], near)

    before = None
    for _ in range(steps):
        if integrator == "rk4":
            sp = sv = 0.0
            p, v = pos, vel
            for w, share in ((0.5, 1.0), (0.5, 2.0), (1.0, 2.0), (0.0, 1.0)):
                kp, kv = dt * v, dt * force(p)
                sp, sv = sp + share * kp, sv + share * kv
                p, v = pos + w * kp, vel + w * kv
            pos, vel = pos + sp / 6.0, vel + sv / 6.0
            continue
        a = force(pos)
        if integrator == "euler" or before is None:
            new = pos + vel * dt + 0.5 * a * dt * dt
            vel = vel + a * dt
        else:
            new = 2.0 * pos - before + a * dt * dt
            vel = (new - pos) / dt
        before, pos = pos, new
    return pos, vel, mass


def _exact_s(kind, n, theta, passes):
    """About the seconds that `passes` force passes of n bodies take here."""
    pairs = _pairs(kind, n, theta)
    if kind == "simple_astro":
        return passes * (0.001 + pairs / 1.5e10)
    return passes * (0.01 + 6e-9 * n + pairs / 1.2e9)


def exact(case, seed):
    # (about 20 seconds of a GPU at most; of many simulations, the first ones)
    left = 18.0
    cost = [_exact_s(case["kind"], n, t, k) for n, t, k in _moves(case)]
    if case["form"] in ("call", "run") and cost[0] > left:
        return None
    if case["form"] == "call":
        pos, _, mass = _fields(_state(case["model"], np.random.default_rng(seed), case["n"]))
        if case["kind"] == "simple_astro":
            return _direct_acc(pos, mass, case["e"]).cpu().numpy()
        return _tree_acc(pos, mass, case["kind"], case["theta"], case["e"], 0.0).cpu().numpy()
    if case["form"] == "run":
        state = _state(case["model"], np.random.default_rng(seed), case["n"])
        pos, vel, mass = _simulate(state, case, case["theta"], case["steps"], case["integrator"],
                                   case["near"])
        out = {f: state[f] for f in FIELDS}
        out["id"] = out["fixed"] = None
        for a, f in enumerate("xyz"):
            out[f], out["v" + f] = pos[:, a].cpu().numpy(), vel[:, a].cpu().numpy()
        if case["energy"]:
            out["energy"] = _energy(pos, vel, mass, case["e"])
        return out
    got = []
    for m, c in zip(_members(case, seed), cost):
        left -= c
        if left < 0.0:
            got.append(None)
            continue
        pos, vel, _ = _simulate(m["state"], case, m["theta"], m["steps"])
        got.append(torch.cat([pos, vel], 1).cpu().numpy())
    return got

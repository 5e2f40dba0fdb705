"""Performance cases: the work that users of the engine have it do, through its public
entry points (gpuvoxels_amd.engine.Batch).

Every pass is what a driver program does between two looks at its simulations: it steps
the batch by a number of physics steps, polls the simulations' statuses (time, centre of
mass, fitness) and reads their whole state back.  Simulations go on from pass to pass.

Families (sizes and physics are those of the benchmark, the configuration legs and the
tests; see gpuvoxels_amd/workloads.py):
  cube     one small solid cube: the shortest calls, where latency counts
  robots   a generation of uneven robots, each small enough for one workgroup
           (`collide`: with self-collision, the default of the VXA format)
  big      robots of up to tens of thousands of voxels (the serving stream's large requests)
  slab     one dense body of bilinear material
  arena    many balls in one simulation, thrown at each other (collision lists rebuilt every
           8 steps)
  swarm    ciliated bodies with signals and collisions in one simulation (the xenobot-like
           experiments' options)
"""
import math

import numpy as np

from gpuvoxels_amd import _abi, engine, workloads


# ---------------------------------------------------------------------------- the cases
def listed():
    return [
        # one 6^3 cube stepped a little at a time (interactive use, single evaluations)
        {"name": "cube6_f64", "family": "cube", "n": 6, "steps": 200, "precision": "f64"},
        # a handful of small robots of odd sizes in the fast precision
        {"name": "robots5_f32", "family": "robots", "count": 5, "grid": 7, "steps": 333, "precision": "f32", "collide": False},
        # the evolutionary search's generation, the benchmark's 512 robots on 12^3 grids, over a
        # good part of its 20,000-step horizon
        {"name": "robots512_f64", "family": "robots", "count": 512, "grid": 12, "steps": 8000, "precision": "f64", "collide": False},
        {"name": "robots512_f32", "family": "robots", "count": 512, "grid": 12, "steps": 8000, "precision": "f32", "collide": False},
        # a generation with self-collision on
        {"name": "robots200_collide_f64", "family": "robots", "count": 200, "grid": 12, "steps": 2000, "precision": "f64",
         "collide": True},
        # the large requests of the serving stream: 15 robots of about 13,000 voxels
        {"name": "big15_f64", "family": "big", "count": 15, "grid": 30, "steps": 3000, "precision": "f64"},
        # one of its largest requests alone, in single precision
        {"name": "big1_f32", "family": "big", "count": 1, "grid": 45, "steps": 2500, "precision": "f32"},
        # a dense body with collisions on, the 64x64x32 configuration
        {"name": "slab64_f64", "family": "slab", "nx": 64, "ny": 64, "nz": 32, "steps": 800, "precision": "f64", "collide": True},
        # a thinner plate of odd extents
        {"name": "plate_f32", "family": "slab", "nx": 61, "ny": 47, "nz": 7, "steps": 800, "precision": "f32", "collide": True},
        # the many-body configuration, in both precisions and at two sizes
        {"name": "arena2048_f64", "family": "arena", "count": 2048, "radius": 4, "steps": 200, "precision": "f64"},
        {"name": "arena300_f32", "family": "arena", "count": 300, "radius": 3, "steps": 400, "precision": "f32"},
        # ciliated, signalling bodies among each other
        {"name": "swarm48_f64", "family": "swarm", "count": 48, "radius": 4, "steps": 400, "precision": "f64"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["cube", "robots", "robots", "robots", "big", "big", "slab", "slab", "arena", "arena", "swarm"])
    precision = rng.choice(["f64", "f64", "f32"])
    if family == "cube":
        return {"family": family, "n": rng.randint(3, 9), "steps": _log(rng, 50, 500), "precision": precision}
    if family == "robots":
        collide = rng.random() < 0.4
        return {"family": family, "count": _log(rng, 2, 200 if collide else 512), "grid": rng.randint(6, 12),
                "steps": _log(rng, 300, 2000 if collide else 6000), "precision": precision, "collide": collide}
    if family == "big":
        grid = rng.randint(14, 45)
        return {"family": family, "count": rng.randint(1, max(1, min(15, int(15 * (30 / grid) ** 3)))), "grid": grid,
                "steps": _log(rng, 500, 2500), "precision": precision}
    if family == "slab":
        return {"family": family, "nx": _log(rng, 20, 64), "ny": _log(rng, 20, 64), "nz": _log(rng, 5, 32),
                "steps": _log(rng, 200, 800), "precision": precision, "collide": rng.random() < 0.7}
    if family == "arena":
        return {"family": family, "count": _log(rng, 100, 2048), "radius": rng.randint(2, 4), "steps": _log(rng, 80, 200),
                "precision": precision}
    return {"family": family, "count": _log(rng, 8, 200), "radius": rng.randint(2, 4), "steps": _log(rng, 150, 400),
            "precision": precision}


# ---------------------------------------------------------------------------- inputs
def _models(case, seed):
    """The models of a case; everything random about them comes from the seed."""
    rng = np.random.default_rng(seed)
    f = case["family"]
    if f == "cube":   # one cube; its actuation starts at a phase of its own
        m = workloads.cube(case["n"], steps=0)
        m.phase = np.full(m.n_voxels, float(rng.random()))
        return [m]
    if f in ("robots", "big"):   # the bodies are the case's, their tissue the seed's
        body = np.random.default_rng(0)
        ms = [workloads.robot(body, grid=case["grid"], steps=0, name="robot_%04d" % i) for i in range(case["count"])]
        for m in ms:
            m.mat = rng.integers(0, 4, m.n_voxels).astype(np.int32)
            m.phase = np.array(workloads.ROBOT_PHASE)[m.mat]
            m.collisions_enabled = 1 if case.get("collide") else 0
        return ms
    if f == "slab":   # the checkerboard of phases shifted by the seed
        m = workloads.slab(case["nx"], case["ny"], case["nz"], steps=0, collisions=case["collide"])
        m.phase = (m.phase + float(rng.random())) % 1.0
        return [m]
    # the arena's footprint per ball is the 2,048-ball configuration's
    arena = int(round((9 * case["radius"] + 4) / 40.0 * 400 * math.sqrt(case["count"] / 2048.0))) + 2 * case["radius"] + 8
    if f == "arena":
        return [workloads.arena_balls(case["count"], radius=case["radius"], arena=arena, steps=0, seed=seed)]
    # swarm: one layer of bodies on the floor, each voxel's cilium pushing it sideways
    m = workloads.arena_balls(case["count"], radius=case["radius"], arena=int(arena * 1.8), gap=0.5, steps=0, seed=seed, z_layers=0)
    m.enable_cilia = 1
    push = rng.normal(0.0, 2e-4, (m.n_voxels, 3))
    push[:, 2] = 0.0
    m.base_cilia = push
    m.shift_cilia = rng.normal(0.0, 2e-5, (m.n_voxels, 3))
    m.enable_signals = 1
    m.materials = [workloads.base_material(cte=0.0, cilia=1.0, matid=1),
                   workloads.base_material(cte=0.0, cilia=1.0, matid=2, is_pacemaker=1, pacemaker_period=0.05)]
    m.mat = (rng.random(m.n_voxels) < 0.02).astype(np.int32)
    return [m]


def prepare(case, seed):
    precision = _abi.PREC_F64 if case["precision"] == "f64" else _abi.PREC_F32
    batch = engine.Batch(precision=precision, path=_abi.PATH_AUTO,
                         collision_rebuild_interval=8 if case["family"] == "arena" else 0)
    slots = [batch.admit(m) for m in _models(case, seed)]
    return {"batch": batch, "slots": slots, "steps": case["steps"]}


def run(state):
    batch, slots = state["batch"], state["slots"]
    batch.step(state["steps"])
    st = batch.poll()
    sims = [batch.read_state(s) for s in slots]
    out = {k: np.concatenate([x[k] for x in sims]) for k in ("pos", "orient", "lin_mom", "ang_mom", "flags", "tfac")}
    out["fitness"] = np.array([st[s].fitness for s in slots])
    out["com"] = np.array([list(st[s].current_com) for s in slots])
    out["time"] = np.array([st[s].current_time for s in slots])
    out["steps"] = np.array([st[s].steps for s in slots])
    out["state"] = np.array([st[s].state for s in slots])
    return out


# ---------------------------------------------------------------------------- work
# Floating-point operations of one beam element and of one voxel update (with the Poisson
# strain), counted over the ordinary branch.
LINK_FLOPS, VOXEL_FLOPS = 300, 260


def _sizes(case):
    """(voxels, links) of a case: exact for the regular bodies, expected for random ones."""
    f = case["family"]
    box = lambda x, y, z: (x * y * z, 3 * x * y * z - x * y - y * z - x * z)  # noqa: E731
    if f == "cube":
        return box(case["n"], case["n"], case["n"])
    if f == "slab":
        return box(case["nx"], case["ny"], case["nz"])
    if f in ("robots", "big"):   # 47.5% of the cells are the robot, 1.43 links a voxel
        v = 0.475 * case["grid"] ** 3 * case["count"]
        return v, 1.43 * v
    off = workloads.ball_offsets(case["radius"])
    cells = set(map(tuple, off.tolist()))
    links = sum((x + 1, y, z) in cells for x, y, z in cells) + sum((x, y + 1, z) in cells for x, y, z in cells) + \
        sum((x, y, z + 1) in cells for x, y, z in cells)
    return case["count"] * len(off), case["count"] * links


def work(case):
    """The state read once and written once (13 reals and three words a voxel, 9 reals and four
    words a link), and every step's arithmetic; what a step keeps on chip is not counted."""
    v, l = _sizes(case)
    r = 8 if case["precision"] == "f64" else 4
    return {"bytes": 2 * (v * (13 * r + 12) + l * (9 * r + 16)) + l * 12,
            "flops": case["steps"] * (VOXEL_FLOPS * v + LINK_FLOPS * l)}


# ---------------------------------------------------------------------------- exact values
# The physics in numpy with 64-bit state: beam elements between lattice neighbours, Poisson
# strain, floor contact with static and kinetic friction, actuation.  Material constants,
# strains, stresses, penetrations and thermal factors are single-precision quantities of the
# model (the reference holds them in float), and are rounded to it here too.
F = np.float32


def _qmul(a, b):
    w, x, y, z = a
    W, X, Y, Z = b
    return (w * W - x * X - y * Y - z * Z, w * X + x * W + y * Z - z * Y, w * Y - x * Z + y * W + z * X,
            w * Z + x * Y - y * X + z * W)


def _qrot(q, f):
    w, x, y, z = q
    a, b, c = f
    tw, tx, ty, tz = a * x + b * y + c * z, a * w - b * z + c * y, a * z + b * w - c * x, -a * y + b * x + c * w
    return (w * tx + x * tw + y * tz - z * ty, w * ty - x * tz + y * tw + z * tx, w * tz + x * ty - y * tx + z * tw)


def _conj(q):
    return (q[0], -q[1], -q[2], -q[3])


def _unrot(q, f):
    return _qrot(_conj(q), f)


def _rotvec(q):
    w, x, y, z = q
    sl = 1.0 - w * w
    near = sl < 2.4e-3
    with np.errstate(all="ignore"):
        k = np.where(near, np.sqrt((2 - 2 * w) / sl), np.arccos(np.clip(w, -1, 1)) / np.sqrt(sl)) * 2.0
    k = np.where((w >= 1) | (w <= -1), 0.0, k)
    return (k * x, k * y, k * z)


def _from_rotvec(v):
    h = tuple(c * 0.5 for c in v)
    m2 = h[0] * h[0] + h[1] * h[1] + h[2] * h[2]
    tiny = m2 * m2 < 5.328e-15
    m = np.sqrt(np.where(tiny, 1.0, m2))
    w = np.where(tiny, 1.0 - 0.5 * m2, np.cos(m))
    s = np.where(tiny, 1.0 - m2 / 6.0, np.sin(m) / m)
    return (w, h[0] * s, h[1] * s, h[2] * s)


def _to_x(a, v):
    return v if a == 0 else (v[1], -v[0], v[2]) if a == 1 else (v[2], v[1], -v[0])


def _from_x(a, v):
    return v if a == 0 else (-v[1], v[0], v[2]) if a == 1 else (-v[2], v[1], v[0])


def _angle_to_x(p):
    """The rotation that turns p onto +x."""
    with np.errstate(all="ignore"):
        yx, zx = p[1] / p[0], p[2] / p[0]
        near = (np.abs(yx) < 1.732e-2) & (np.abs(zx) < 1.732e-2)
        y0, z0 = 0.5 * zx, -0.5 * yx
        n = np.sqrt(p[0] * p[0] + p[1] * p[1] + p[2] * p[2])
        c, ny, nz = p[0] / n, p[1] / n, p[2] / n
        flip = np.arccos(np.clip(c, -1, 1)) > 3.14159265358979 - 1e-7
        s = np.sqrt((1 - c) * 0.5) / np.sqrt(ny * ny + nz * nz)
    w = np.where(near, 1 + 0.5 * (-y0 * y0 - z0 * z0), np.where(flip, 0.0, np.sqrt((1 + c) * 0.5)))
    return (w, np.zeros_like(w), np.where(near, y0, np.where(flip, 1.0, nz * s)), np.where(near, z0, np.where(flip, 0.0, -ny * s)))


def _exact_one(m, steps):
    """One simulation (linear materials, floor, no collisions) for `steps` steps."""
    nom = float(m.voxel_size)
    size = F(nom)
    mats = m.materials
    V = m.n_voxels
    E = np.array([a.elastic_mod for a in mats], F)
    nu = np.array([a.poissons_ratio if m.volume_effects else 0.0 for a in mats], F)
    mass = (nom ** 3 * np.array([a.density for a in mats], F).astype(np.float64)).astype(F)
    inertia = (mass.astype(np.float64) * nom * nom / 6.0).astype(F)
    c_lin = (2.0 * np.sqrt((mass * E).astype(np.float64) * nom)).astype(F)
    c_ang = (2.0 * np.sqrt((inertia * E).astype(np.float64) * nom * nom * nom)).astype(F)
    zi, zg, zc = (np.array([getattr(a, k) for a in mats], F) for k in ("zeta_internal", "zeta_global", "zeta_collision"))
    grav = -mass * F(9.80665) * F(m.gravity_mult)
    e_hat = (E / ((1 - 2 * nu) * (1 + nu))).astype(F)
    vm = np.asarray(m.mat)
    # links: lattice neighbours, the negative end first; the voxel added later leads the pair
    at = {tuple(c): i for i, c in enumerate(np.asarray(m.ijk).tolist())}
    links = []
    for a in range(3):
        step = [0, 0, 0]
        step[a] = 1
        pairs = [(i, at[(c[0] + step[0], c[1] + step[1], c[2] + step[2])]) for c, i in at.items()
                 if (c[0] + step[0], c[1] + step[1], c[2] + step[2]) in at]
        vn, vp = (np.array([p[k] for p in pairs], np.int64) for k in (0, 1))
        lead, other = np.maximum(vn, vp), np.minimum(vn, vp)
        # the first pair of two materials met in the structure's order makes their link material
        links.append([vn, vp, lead, other])
    first = {}
    met = sorted((int(x), a, int(o)) for a, (_, _, ld, ot) in enumerate(links) for x, o in zip(ld, ot))
    for x, _, o in met:
        first.setdefault(frozenset((int(vm[x]), int(vm[o]))), (int(vm[x]), int(vm[o])))
    made = {}
    for key, (a, b) in first.items():
        el = F(F(F(2.0) * E[a]) * E[b]) / F(E[a] + E[b])
        if nu[a] == 0 and nu[b] == 0:
            nl = F(0)
        else:
            eh = F(F(F(2) * e_hat[a]) * e_hat[b]) / F(e_hat[a] + e_hat[b])
            nl = F(np.sqrt(F(float(F(eh - el) / F(F(2) * eh)) + 0.0625)) - 0.25)
        hat = el / F(F(1 - F(2) * nl) * F(1 + nl))
        L = size
        a2 = F(F(F(el * L) * L) * L) / F(F(12.0) * F(1 + nl))
        b1, b2, b3 = F(el * L), F(F(el * L) * L) / F(2), F(F(F(el * L) * L) * L) / F(6)
        made[key] = [el, nl, hat, b1, a2, b1, b2, b3, F(np.sqrt(b1)), F(np.sqrt(F(F(F(a2 * L) * L) / F(6)))), F(np.sqrt(b1)),
                     F(np.sqrt(F(F(b2 * L) / F(2)))), F(np.sqrt(F(F(F(b3 * L) * L) / F(6))))]
    G = []
    for a, (vn, vp, _, _) in enumerate(links):
        rows = np.array([made[frozenset((int(vm[i]), int(vm[j])))] for i, j in zip(vn, vp)], F).reshape(-1, 13)
        n = len(vn)
        G.append({"a": a, "vn": vn, "vp": vp, "c": [rows[:, k] for k in range(13)], "ratio": E[vm[vp]] / E[vm[vn]],
                  "p2": tuple(np.zeros(n) for _ in range(3)), "a1": tuple(np.zeros(n) for _ in range(3)),
                  "a2": tuple(np.zeros(n) for _ in range(3)), "small": np.ones(n, bool), "valid": np.zeros(n, bool)})
    has = np.zeros((6, V), bool)
    for a, g in enumerate(G):
        has[2 * a][g["vn"]] = True
        has[2 * a + 1][g["vp"]] = True
    both = [has[2 * a] & has[2 * a + 1] for a in range(3)]
    pos = [np.asarray(m.ijk)[:, k] * nom for k in range(3)]
    lin, ang = ([np.zeros(V) for _ in range(3)] for _ in range(2))
    ori = (np.ones(V), np.zeros(V), np.zeros(V), np.zeros(V))
    phase = np.zeros(V) if m.phase is None else np.asarray(m.phase, np.float64)
    static = np.ones(V, bool)
    ps = [np.zeros(V, F) for _ in range(3)]
    vmass, vmi, vii = mass[vm], (F(1) / mass)[vm], (F(1) / inertia)[vm]
    sq_mass = np.sqrt(mass)[vm]
    cte = np.array([a.cte for a in mats], F)[vm]
    pen_k = (2 * E.astype(np.float64) * nom).astype(F)[vm]
    mu_s, mu_k = (np.array([getattr(a, k) for a in mats], F)[vm] for k in ("u_static", "u_dynamic"))
    vnu, vgrav = nu[vm], grav[vm].astype(np.float64)
    drag = (zg * c_lin)[vm].astype(np.float64)
    drag_r = (zg * c_ang)[vm].astype(np.float64)
    bounce = (zc * c_lin)[vm].astype(np.float64)

    def thermal(t):
        T = m.temp_amplitude * np.sin(float(F(2) * F(3.1415926)) * (t / m.temp_period + phase))
        return F(1) + np.where(T > 0, 0.0, T).astype(F) * cte

    def across(g, v):   # transverse area and strain sum of the voxels v across the link's axis
        o = [k for k in range(3) if k != g["a"]]
        s, u = ps[o[0]][v], ps[o[1]][v]
        ar = (float(size * size) * (1.0 + s.astype(np.float64)) * (1.0 + u.astype(np.float64))).astype(F)
        none = vnu[v] == 0
        return np.where(none, size * size, ar), np.where(none, F(0), s + u)

    tf = thermal(0.0)
    stiff = 0.0
    for g in G:   # the recommended step: the stiffest link over its lighter end
        vn, vp, c = g["vn"], g["vp"], g["c"]
        if not len(vn):
            continue
        an, ap = across(g, vn)[0], across(g, vp)[0]
        rl = 0.5 * (nom * tf[vn].astype(np.float64) + nom * tf[vp].astype(np.float64))
        k = np.where(c[1] == 0, c[3], ((c[2] * (F(0.5) * (an + ap))).astype(np.float64) / rl).astype(F))
        stiff = max(stiff, float(np.max(k.astype(np.float64) / np.minimum(vmass[vn], vmass[vp]).astype(np.float64))))
    dt = F(m.dt_frac * (1.0 / (float(F(6.283185)) * math.sqrt(stiff))))
    dtd, t = float(dt), 0.0
    damp = F(2) * sq_mass * zi[vm] / dt
    D = np.float64
    for _ in range(steps):
        f, mo = ([np.zeros(V) for _ in range(3)] for _ in range(2))
        es = [np.zeros(V, F) for _ in range(6)]
        for g in G:
            a, vn, vp = g["a"], g["vn"], g["vp"]
            el, nl, hat, _, A2, B1, B2, B3, qa1, qa2, qb1, qb2, qb3 = g["c"]
            rest = 0.5 * (nom * tf[vn].astype(D) + nom * tf[vp].astype(D))
            q1 = tuple(o[vn] for o in ori)
            q1 = (q1[0],) + _to_x(a, q1[1:])
            q2 = tuple(o[vp] for o in ori)
            q2 = (q2[0],) + _to_x(a, q2[1:])
            p = _qrot(_conj(q1), _to_x(a, tuple(x[vp] - x[vn] for x in pos)))
            q2 = _qmul(_conj(q1), q2)
            with np.errstate(all="ignore"):
                turn = ((np.abs(p[2]) + np.abs(p[1])) / p[0]).astype(F)
                ext = np.abs(1.0 - p[0] / rest).astype(F)
            was = g["small"]
            now = np.where(was, ~((turn > F(1.2) * F(0.05)) | (ext > F(1.2) * F(0.5))), (turn < F(0.05)) & (ext < F(0.5)))
            valid = g["valid"] & (now == was)
            g["small"], g["valid"] = now, np.ones_like(valid)
            turnq = _angle_to_x(p)
            one = (np.ones(len(vn)), np.zeros(len(vn)), np.zeros(len(vn)), np.zeros(len(vn)))
            r1 = tuple(np.where(now, i, j) for i, j in zip(one, turnq))
            q2 = tuple(np.where(now, i, j) for i, j in zip(q2, _qmul(turnq, q2)))
            length = np.sqrt(p[0] * p[0] + p[1] * p[1] + p[2] * p[2])
            p = (np.where(now, p[0], length) - rest, np.where(now, p[1], 0.0), np.where(now, p[2], 0.0))
            a1, a2 = _rotvec(r1), _rotvec(q2)
            dp, d1, d2 = (tuple((x - y) * 0.5 for x, y in zip(u, w)) for u, w in ((p, g["p2"]), (a1, g["a1"]), (a2, g["a2"])))
            g["p2"], g["a1"], g["a2"] = p, a1, a2
            e = (p[0] / rest).astype(F)
            an, sn = across(g, vn)
            ap, sp = across(g, vp)
            no = nl == 0
            area = F(0.5) * np.where(no, size * size + size * size, an + ap)
            tss = np.where(no, F(0), F(0.5) * (sn + sp))
            stress = np.where(no, el * e, hat * ((1 - nl) * e + nl * tss))
            A2, B1, B2, B3, qa1, qa2, qb1, qb2, qb3 = (x.astype(D) for x in (A2, B1, B2, B3, qa1, qa2, qb1, qb2, qb3))
            fn = [(stress * area).astype(D), B1 * p[1] - B2 * (a1[2] + a2[2]), B1 * p[2] + B2 * (a1[1] + a2[1])]
            fp = [-x for x in fn]
            mn = [A2 * (a2[0] - a1[0]), -B2 * p[2] - B3 * (2 * a1[1] + a2[1]), B2 * p[1] - B3 * (2 * a1[2] + a2[2])]
            mp = [A2 * (a1[0] - a2[0]), -B2 * p[2] - B3 * (a1[1] + 2 * a2[1]), B2 * p[1] - B3 * (a1[2] + 2 * a2[2])]
            kn, kp = np.where(valid, damp[vn].astype(D), 0.0), np.where(valid, damp[vp].astype(D), 0.0)
            v = (qa1 * dp[0], qb1 * dp[1] - qb2 * (d1[2] + d2[2]), qb1 * dp[2] + qb2 * (d1[1] + d2[1]))
            w1 = (-qa2 * (d2[0] - d1[0]), qb2 * dp[2] + qb3 * (2 * d1[1] + d2[1]), -qb2 * dp[1] + qb3 * (2 * d1[2] + d2[2]))
            w2 = (qa2 * (d2[0] - d1[0]), qb2 * dp[2] + qb3 * (d1[1] + 2 * d2[1]), -qb2 * dp[1] + qb3 * (d1[2] + 2 * d2[2]))
            fn, fp = [x + kn * y for x, y in zip(fn, v)], [x - kp * y for x, y in zip(fp, v)]
            mn, mp = [x - 0.5 * kn * y for x, y in zip(mn, w1)], [x - 0.5 * kp * y for x, y in zip(mp, w2)]
            fn = [np.where(now, x, y) for x, y in zip(fn, _unrot(r1, fn))]
            mn = [np.where(now, x, y) for x, y in zip(mn, _unrot(r1, mn))]
            for v_, fo, mm, s_, d in ((vn, fn, mn, F(2) * e / (F(1) + g["ratio"]), 2 * a),
                                      (vp, _unrot(q2, fp), _unrot(q2, mp), F(2) * e * g["ratio"] / (F(1) + g["ratio"]), 2 * a + 1)):
                for k, (x, y) in enumerate(zip(_from_x(a, tuple(fo)), _from_x(a, tuple(mm)))):
                    f[k][v_] += x
                    mo[k][v_] += y
                es[d][v_] = s_
        # voxels
        mi = vmi.astype(D)
        cf = list(_qrot(ori, f))
        cf = [c - (x * mi) * drag for c, x in zip(cf, lin)]
        cf[2] = cf[2] + vgrav
        bs = nom * tf.astype(D)
        pen = ((bs + bs + bs) / 3.0 / 2.0 - nom / 2.0 - pos[2]).astype(F)
        down = pen >= 0
        before = (cf[0], cf[1])
        nf = pen_k * pen
        vel = [x * mi for x in lin]
        cf[2] = np.where(down, cf[2] + (nf.astype(D) - bounce * vel[2]), cf[2])
        slips = (cf[0] * cf[0] + cf[1] * cf[1]).astype(F) > (mu_s * nf) * (mu_s * nf)
        h = np.sqrt(vel[0] * vel[0] + vel[1] * vel[1])
        with np.errstate(all="ignore"):
            u = [np.where(h > 0, (1.0 / h) * x, x) for x in vel[:2]]
        fr = (mu_k * nf).astype(D)
        held = static
        cf[0], cf[1] = (np.where(down & ~held, c - x * fr, c) for c, x in zip(cf[:2], u))
        static = held & down & ~(down & slips)
        df = (cf[0] - before[0], cf[1] - before[1])
        lin = [x + c * dtd for x, c in zip(lin, cf)]
        k = (dt * vmi).astype(D)
        tr = [x * k for x in lin]
        work_ = df[0] * tr[0] + df[1] * tr[1]
        ke = 0.5 * mi * (lin[0] * lin[0] + lin[1] * lin[1])
        static = np.where(down, static | (ke + work_ <= 0), False)
        for q in (0, 1):
            lin[q] = np.where(static, 0.0, lin[q])
            tr[q] = np.where(static, 0.0, tr[q])
        pos = [x + y for x, y in zip(pos, tr)]
        cm = [c - (x * vii.astype(D)) * drag_r for c, x in zip(_qrot(ori, mo), ang)]
        ang = [x + c * dtd for x, c in zip(ang, cm)]
        ori = _qmul(_from_rotvec(tuple(x * (dt * vii).astype(D) for x in ang)), ori)
        t = t + dtd
        tf = thermal(t)
        # Poisson strain of the next step
        st = [np.where(both[a], (es[2 * a] + es[2 * a + 1]) * F(0.5), es[2 * a] + es[2 * a + 1]) for a in range(3)]
        add = sum((np.where(both[a], st[a], F(0)) for a in range(3)), np.zeros(V, F)).astype(F)
        val = np.power((F(1) + add).astype(D), -vnu.astype(D)).astype(F) - F(1)
        ps = [np.where(both[a], st[a], val).astype(F) for a in range(3)]
    return {"pos": np.stack(pos, 1), "orient": np.stack(ori, 1), "lin_mom": np.stack(lin, 1), "ang_mom": np.stack(ang, 1),
            "tfac": tf.astype(D), "mass": vmass.astype(D), "time": t}


# voxel-steps that the numpy physics gets through in about 20 seconds
EXACT_VOXEL_STEPS = 4e6


def exact(case, seed):
    """What run() returns for the first pass.  None where contacts or extra forces act (every
    such case is one of large bodies, beyond what numpy does in the time), and beyond the
    voxel-steps it gets through in 20 seconds; flags, steps and states have no such value, nor
    have single-precision momenta (friction turns on the direction of velocities near zero,
    which rounding to 32 bits sets)."""
    if case["family"] not in ("cube", "robots") or case.get("collide") or _sizes(case)[0] * case["steps"] > EXACT_VOXEL_STEPS:
        return None
    models = _models(case, seed)
    sims = [_exact_one(m, case["steps"]) for m in models]
    out = {k: np.concatenate([x[k] for x in sims]) for k in ("pos", "orient", "tfac")}
    for k in ("lin_mom", "ang_mom"):
        out[k] = np.concatenate([x[k] for x in sims]) if case["precision"] == "f64" else None
    com, fit = [], []
    for m, x in zip(models, sims):
        w = x["mass"][:, None]
        com.append((x["pos"] * w).sum(0) / w.sum())
        d = com[-1] - (np.asarray(m.ijk) * float(m.voxel_size) * w).sum(0) / w.sum()
        fit.append(math.sqrt(float((d[:3 if case["family"] == "cube" else 2] ** 2).sum())))
    out["com"], out["time"] = np.array(com), np.array([x["time"] for x in sims])
    out["fitness"] = np.array(fit) if case["precision"] == "f64" else None
    out["flags"] = out["steps"] = out["state"] = None
    return out

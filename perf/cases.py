"""The work that a program built on this framework has it do, as cases that can be timed
and compared: whole steps of single scenes, of batches of worlds and of scenes with joints,
hulls and triangle meshes, batched scene queries and served requests, each through the
public entry points of physecs_amd.api.

A stepping case is a rollout: the program holds a scene that has been stepped for a while
and the bytes of its saved state; a pass loads the state, steps the scene `steps` times at
1/60 s and reads the poses and velocities back (an episode of a learner, a planner's
look-ahead, a rollback). The state is the same at the start of every pass, so every pass is
the same work.
"""
import math

import numpy as np
import torch

from physecs_amd import api, scenes

DT = 1.0 / 60.0

# (friction, restitution, damping) of every collider: damping other than 0 makes a contact
# soft, and restitution is then its frequency
MATERIALS = {"hard": (0.6, 0.0, 0.0), "bouncy": (0.6, 0.4, 0.0), "soft": (0.6, 8.0, 1.0)}


def listed():
    return [
        # one small stack, the smallest scene that is stepped in earnest: latency
        {"name": "pyramid_210", "kind": "pyramid", "rows": 20, "substeps": 4, "iterations": 2, "steps": 8},
        # a few jointed figures and chains: the joint rows, and few contacts
        {"name": "figures_24", "kind": "figures", "chains": 16, "ragdolls": 8, "substeps": 4, "iterations": 2,
         "steps": 8},
        # a game level's worth of loose bodies, with restitution, an odd count and more
        # substeps (the reference's default of 8)
        {"name": "pile_1331_bouncy", "kind": "pile", "bodies": 1331, "material": "bouncy", "substeps": 8,
         "iterations": 2, "steps": 8},
        # the same with soft contacts, larger
        {"name": "pile_6000_soft", "kind": "pile", "bodies": 6000, "material": "soft", "substeps": 4,
         "iterations": 2, "steps": 6},
        # the benchmark's scene: 32,768 mixed bodies in a container
        {"name": "pile_32768", "kind": "pile", "bodies": 32768, "material": "hard", "substeps": 4, "iterations": 2,
         "steps": 8},
        # a learner's worlds: many small ones, all stepped together
        {"name": "worlds_512_small", "kind": "worlds", "worlds": 512, "lo": 8, "hi": 48, "figures": 0.25,
         "substeps": 4, "iterations": 2, "steps": 8},
        # worlds of very uneven size, some with a figure: the largest case
        {"name": "worlds_1024", "kind": "worlds", "worlds": 1024, "lo": 8, "hi": 1024, "figures": 0.25,
         "substeps": 4, "iterations": 2, "steps": 12},
        # hulls and chains on a terrain of triangles
        {"name": "terrain_2048", "kind": "terrain", "hulls": 2048, "chains": 128, "quads": 128, "substeps": 4,
         "iterations": 2, "steps": 6},
        # rays into the benchmark's scene (a sensor's frame)
        {"name": "rays_262144", "kind": "rays", "rays": 262144, "bodies": 32768},
        # characters that walk on a terrain among hulls
        {"name": "characters_4096", "kind": "characters", "characters": 4096, "hulls": 512, "quads": 96},
        # a burst of requests through the server, to the end of the last
        {"name": "served_40", "kind": "served", "requests": 40, "lo": 16, "hi": 512, "horizon": 20},
    ]


def _log_int(rng, lo, hi):
    return int(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.99))))


def draw(rng):
    """One more case of the listed ones' kinds and ranges; sizes over their logarithm."""
    kind = rng.choice(["pyramid", "figures", "pile", "pile", "worlds", "worlds", "terrain", "rays", "characters",
                       "served"])
    sub = {"substeps": rng.choice([2, 3, 4, 4, 8]), "iterations": rng.choice([1, 2, 2, 3]),
           "steps": rng.randrange(3, 9)}
    if kind == "pyramid":
        return {"kind": kind, "rows": rng.randrange(3, 28), **sub}
    if kind == "figures":
        return {"kind": kind, "chains": rng.randrange(1, 40), "ragdolls": rng.randrange(0, 20), **sub}
    if kind == "pile":
        return {"kind": kind, "bodies": _log_int(rng, 60, 30000), "material": rng.choice(sorted(MATERIALS)), **sub}
    if kind == "worlds":
        hi = rng.choice([24, 100, 400, 1000])
        return {"kind": kind, "worlds": _log_int(rng, 8, 700), "lo": 8, "hi": hi, "figures": rng.choice([0.0, 0.25]),
                **sub}
    if kind == "terrain":
        return {"kind": kind, "hulls": _log_int(rng, 50, 2000), "chains": rng.randrange(0, 120),
                "quads": rng.randrange(24, 128), **sub}
    if kind == "rays":
        return {"kind": kind, "rays": _log_int(rng, 16, 260000), "bodies": _log_int(rng, 200, 30000)}
    if kind == "characters":
        return {"kind": kind, "characters": _log_int(rng, 1, 4000), "hulls": _log_int(rng, 20, 500),
                "quads": rng.randrange(24, 96)}
    return {"kind": kind, "requests": rng.randrange(2, 40), "lo": 16, "hi": rng.choice([64, 200, 500]),
            "horizon": rng.randrange(8, 24)}


# ---------------------------------------------------------------- scenes
def _shapes(rng, n):
    """Types and parameters of n bodies, a third each of spheres, capsules and boxes."""
    kinds = rng.permutation(np.arange(n) % 3)
    prm = np.zeros((n, 4))
    prm[:, :3] = rng.uniform(0.2, 0.6, (n, 3))                              # boxes: half extents
    ball, cap = kinds == scenes.SPHERE, kinds == scenes.CAPSULE
    prm[ball, 0], prm[ball, 1:] = rng.uniform(0.2, 0.5, int(ball.sum())), 0.0
    prm[cap, 1], prm[cap, 2:] = rng.uniform(0.15, 0.3, int(cap.sum())), 0.0   # half height, radius
    return kinds, prm


def _lattice(n, side):
    i = np.arange(n)
    off = (side - 1) * 1.5 / 2
    return np.stack([(i % side) * 1.5 - off, 1.0 + (i // (side * side)) * 1.5, ((i // side) % side) * 1.5 - off], 1)


def _pile(seed, n, material="hard"):
    """n spheres, capsules and boxes on a jittered lattice in an open container, the shapes
    and spacing of scenes.mixed_lattice, appended in bulk."""
    rng = np.random.default_rng(seed)
    side = math.ceil(n ** (1 / 3))
    s = scenes.Scene()
    scenes.container(s, half=max(25.0, (side - 1) * 1.5 / 2 + 1.75))
    kinds, prm = _shapes(rng, n)
    pos = _lattice(n, side) + rng.uniform(-0.05, 0.05, (n, 3))
    s.add_bodies_bulk(kinds, prm, pos, scenes.random_quats(rng, n), rng.normal(size=(n, 3)), np.zeros(n, int))
    s.col_material[:] = MATERIALS[material]
    return s


def _terrain(seed, hulls, chains, quads, drop=(0.3, 5.0)):
    """Convex hulls (bodies share 48 of them) and capsule chains dropped on a heightfield.
    Returns the scene and the heights."""
    rng = np.random.default_rng(seed)
    s = scenes.Scene()
    verts, tris, h = scenes.terrain_mesh(seed, quads=quads, amplitude=4.0)
    mesh = s.add_triangle_mesh(verts, tris)
    s.add_collider(s.add_actor([0, 0, 0]), scenes.TRIANGLE_MESH, [0, 0, 0, float(mesh)])
    shapes = []
    for _ in range(48):
        m = s.add_convex_mesh(*scenes.ellipsoid_hull(rng))
        v, faces, _, _ = s.convex[m]
        mass = 1000.0 * scenes.hull_volume(v, faces)
        com, inertia = scenes.convex_mass_props(v, faces, (1, 1, 1), mass)
        shapes.append((m, np.float32(1.0 / mass), com, inertia))
    half = quads / 2 - 4.0

    def ground(x, z):
        i, j = int(round(x + quads / 2)), int(round(z + quads / 2))
        return float(h[max(0, i - 1):i + 2, max(0, j - 1):j + 2].max())

    quats = scenes.random_quats(rng, max(hulls, 1))
    for k in range(hulls):
        m, inv_mass, com, inertia = shapes[int(rng.integers(0, 48))]
        x, z = rng.uniform(-half, half, 2)
        a = s.add_actor([x, ground(x, z) + 0.8 + rng.uniform(*drop), z], quats[k])
        s.add_dynamic(a, inv_mass, com, inertia)
        s.add_collider(a, scenes.CONVEX_MESH, [1.0, 1.0, 1.0, float(m)])
    for _ in range(chains):
        x, z = rng.uniform(-half, half - 7.0, 2)
        top = max(ground(x + k, z) for k in range(8)) + 0.3 + rng.uniform(*drop)
        scenes.capsule_chain(s, [x, top, z], n=8)
    return s, h


def _sizes(n, lo, hi):
    """n sizes log-uniform over [lo, hi], the same ones every time."""
    return np.exp(math.log(lo) + (np.arange(n) + 0.5) / n * math.log(hi / lo)).astype(int)


def _worlds(seed, n, lo, hi, figures):
    """n worlds as scenes.batched_worlds lays them out (bodies on a lattice above a ground
    box, in a share of them a jointed figure on a pad of its own); sizes in a seeded order."""
    rng = np.random.default_rng(seed)
    s = scenes.Scene()
    counts = rng.permutation(_sizes(n, lo, hi))
    with_figure = rng.permutation(np.arange(n) < int(figures * n))
    for w in range(n):
        m = int(counts[w])
        side = math.ceil(m ** (1 / 3))
        half = (side - 1) * 1.5 / 2 + 1.0
        s.add_static(scenes.BOX, [half + 2, 0.5, half + 2], [0, -0.5, 0], world=w)
        kinds, prm = _shapes(rng, m)
        s.add_bodies_bulk(kinds, prm, _lattice(m, side), scenes.random_quats(rng, m), rng.normal(size=(m, 3)),
                          np.full(m, w))
        if with_figure[w]:
            s.add_static(scenes.BOX, [2.0, 0.5, 2.0], [half + 20.0, -0.5, 0.0], world=w)
            scenes.ragdoll(s, [half + 20.0, 0.3, 0.0], world=w)
    return s


def _figures(seed, chains, ragdolls):
    """Capsule chains and jointed figures dropped on a ground box, each on a place of its own."""
    rng = np.random.default_rng(seed)
    s = scenes.Scene()
    rows = math.ceil((chains + ragdolls) / 4)
    s.add_static(scenes.BOX, [24, 0.5, 2.0 * rows + 4], [0, -0.5, 0])
    for k, place in enumerate(rng.permutation(chains + ragdolls)):
        x, z = 10.0 * (place % 4) - 19.0, 4.0 * (place // 4) - 2.0 * rows
        if k < chains:
            scenes.capsule_chain(s, [x, rng.uniform(1.0, 4.0), z + rng.uniform(-0.5, 0.5)], n=8)
        else:
            scenes.ragdoll(s, [x + 3.0, rng.uniform(0.2, 0.6), z + rng.uniform(-0.5, 0.5)])
    return s


def _settle(case):
    """Steps before the rollout starts: the bodies have fallen together."""
    if case["kind"] == "pile":
        return 60 + 5 * math.ceil(case["bodies"] ** (1 / 3))
    return {"pyramid": 30, "figures": 60, "worlds": 70, "terrain": 80}[case["kind"]]


def _rays(case, seed):
    rng = np.random.default_rng([seed, 1])
    n = case["rays"]
    side = math.ceil(case["bodies"] ** (1 / 3))
    half, top = (side - 1) * 1.5 / 2 + 1.0, side * 1.5 + 2.0
    origins = rng.uniform((-half - 4, 0.1, -half - 4), (half + 4, top + 8, half + 4), (n, 3)).astype(np.float32)
    d = rng.uniform((-half, 0, -half), (half, top, half), (n, 3)) - origins
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return origins, d.astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "rays":
        w = api.World(_pile(seed, case["bodies"]))
        return {"kind": kind, "world": w, "rays": _rays(case, seed)}
    if kind == "characters":
        s, h = _terrain(seed, case["hulls"], 0, case["quads"])
        w = api.World(s)
        for _ in range(80):
            w.step(DT)
        rng = np.random.default_rng([seed, 1])
        n, quads = case["characters"], case["quads"]
        xz = rng.uniform(-quads / 2 + 4, quads / 2 - 4, (n, 2))
        i, j = np.floor(xz[:, 0] + quads / 2).astype(int), np.floor(xz[:, 1] + quads / 2).astype(int)
        u, v = xz[:, 0] + quads / 2 - i, xz[:, 1] + quads / 2 - j
        a, b, c, d = h[i, j], h[i, j + 1], h[i + 1, j], h[i + 1, j + 1]
        ground = np.where(u + v <= 1, a + (c - a) * u + (b - a) * v, d + (b - d) * (1 - u) + (c - d) * (1 - v))
        pos = np.stack([xz[:, 0], ground - 0.05, xz[:, 1]], 1).astype(np.float32)
        yaw = rng.uniform(0, 2 * np.pi, n)
        quat = np.zeros((n, 4), np.float32)
        quat[:, 1], quat[:, 3] = np.sin(yaw / 2), np.cos(yaw / 2)
        walk = np.stack([np.cos(yaw), np.zeros(n), np.sin(yaw)], 1).astype(np.float32) * 0.1
        return {"kind": kind, "world": w, "pos": pos, "quat": quat, "walk": walk}
    if kind == "served":
        rng = np.random.default_rng([seed, 1])
        # every tenth request holds a chain; the sizes in a fixed, mixed order
        sizes = np.random.default_rng(7).permutation(_sizes(case["requests"], case["lo"], case["hi"]))
        requests = [scenes.served_request(int(rng.integers(1 << 30)), n_bodies=int(n), chain=k % 10 == 0)
                    for k, n in enumerate(sizes)]
        for r in requests:
            r.arrays()
        horizons = [int(x) for x in rng.integers(case["horizon"] // 2, case["horizon"] + 1, case["requests"])]
        return {"kind": kind, "server": api.Server(), "requests": requests, "horizons": horizons}
    if kind == "pyramid":
        s = scenes.box_pyramid(seed, rows=case["rows"])
    elif kind == "figures":
        s = _figures(seed, case["chains"], case["ragdolls"])
    elif kind == "pile":
        s = _pile(seed, case["bodies"], case["material"])
    elif kind == "worlds":
        s = _worlds(seed, case["worlds"], case["lo"], case["hi"], case["figures"])
    else:
        s, _ = _terrain(seed, case["hulls"], case["chains"], case["quads"])
    w = api.World(s, substeps=case["substeps"], iterations=case["iterations"])
    for _ in range(_settle(case)):
        w.step(DT)
    return {"kind": kind, "world": w, "saved": w.save_state(), "steps": case["steps"]}


def run(state):
    kind = state["kind"]
    if kind == "rays":
        o, d = state["rays"]
        collider, t, _ = state["world"].raycast(o, d, 200.0)
        return {"collider": collider, "distance": t}
    if kind == "characters":
        pos, flags = state["world"].character_move(state["pos"], state["quat"], state["walk"], 1.6, 0.35)
        return {"pos": pos, "flags": flags}
    if kind == "served":
        srv = state["server"]
        ids = [srv.submit(s, n) for s, n in zip(state["requests"], state["horizons"])]
        while not all(srv.done(r) for r in ids):
            srv.step(DT)
        results = [srv.take_result(r) for r in ids]
        return {k: np.concatenate([r[i] for r in results]) for i, k in enumerate(("pos", "quat", "vel", "angvel"))}
    w = state["world"]
    w.load_state(state["saved"])
    for _ in range(state["steps"]):
        w.step(DT)
    return dict(zip(("pos", "quat", "vel", "angvel"), w.state()))


# ---------------------------------------------------------------- what a pass cannot do without
def _bodies(case):
    kind = case["kind"]
    if kind == "pyramid":
        return case["rows"] * (case["rows"] + 1) // 2
    if kind == "figures":
        return 8 * case["chains"] + 15 * case["ragdolls"]
    if kind in ("pile", "rays"):
        return case["bodies"]
    lo, hi = case.get("lo", 0), case.get("hi", 0)
    mean = (hi - lo) / math.log(hi / lo) if hi > lo else lo          # of a log-uniform size
    if kind == "worlds":
        return int(case["worlds"] * (mean + 15 * case["figures"]))
    if kind == "served":
        return int(case["requests"] * mean)
    return case["hulls"] + 8 * case.get("chains", 0)


def work(case):
    """A step reads each body's pose and velocities (52 B), mass properties (52 B) and
    collider (64 B) and writes pose, velocities and bounds (76 B). Its arithmetic is the
    contact solve's: about 130 operations per point and pass, about 4 points per body in a
    settled pile, iterations + 1 passes per substep. A query reads its inputs and the
    bodies' colliders, bounds and poses (116 B) once and writes its results."""
    n = _bodies(case)
    if case["kind"] == "rays":
        return {"bytes": 116 * n + 36 * case["rays"], "flops": 300 * case["rays"]}
    if case["kind"] == "characters":
        return {"bytes": 116 * n + 24 * 2 * case["quads"] ** 2 + 53 * case["characters"],
                "flops": 4000 * case["characters"]}
    if case["kind"] == "served":
        steps, sub, it = 0.75 * case["horizon"], 4, 2
    else:
        steps, sub, it = case["steps"], case["substeps"], case["iterations"]
    return {"bytes": steps * n * 244, "flops": steps * sub * (it + 1) * n * 4 * 130}


def tolerance(case):
    """Every float of a step or a query is rounded in the reference's order, and the solve
    order is fixed, so two correct builds give the same bits; a step's velocities amplify
    any other rounding without bound."""
    return "exact"


# ---------------------------------------------------------------- 64-bit results
def exact(case, seed):
    """The hit distances of the rays, every ray against every collider with the reference's
    ray tests (sphere, capsule, box; directions are unit vectors). The steps have no such
    value within the time: two iterations do not converge, so their result is a chain of
    some hundred thousand contact solves per pass in one fixed order."""
    if case["kind"] != "rays":
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    arr = _pile(seed, case["bodies"]).arrays()
    origins, dirs = (torch.tensor(x, dtype=torch.float64, device=dev) for x in _rays(case, seed))

    def column(name):
        return torch.tensor(arr[name], dtype=torch.float64, device=dev)

    actor = torch.tensor(arr["col_actor"], dtype=torch.int64, device=dev)
    pos, quat, prm = column("pos")[actor], column("quat")[actor], column("col_params")
    kinds = torch.tensor(arr["col_type"], device=dev)
    x, y, z, w = quat.unbind(1)
    # rows of the inverse rotation: world to body
    rot = torch.stack([torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y + w * z), 2 * (x * z - w * y)], 1),
                       torch.stack([2 * (x * y - w * z), 1 - 2 * (x * x + z * z), 2 * (y * z + w * x)], 1),
                       torch.stack([2 * (x * z + w * y), 2 * (y * z - w * x), 1 - 2 * (x * x + y * y)], 1)], 1)
    best = torch.full((len(origins),), math.inf, dtype=torch.float64, device=dev)

    def closer(sel, hit, t):
        t = torch.where(hit & (t <= 200.0), t, math.inf)
        best[sel] = torch.minimum(best[sel], t.min(1).values)

    def ball(m, d, r2):
        """Entry distance into a sphere at -m from the origin (0 where that lies behind), and
        whether the line meets it and the ray does; m, d as 3 components."""
        b = m[0] * d[0] + m[1] * d[1] + m[2] * d[2]
        c = m[0] ** 2 + m[1] ** 2 + m[2] ** 2 - r2
        disc = b * b - c
        return disc >= 0, (disc >= 0) & ~((c > 0) & (b > 0)), (-b - disc.clamp(min=0).sqrt()).clamp(min=0)

    def slabs(m, d, half):
        """Entry distance into a box of these half extents, and whether there is one."""
        t0, t1 = torch.zeros_like(m[0]), torch.full_like(m[0], math.inf)
        for k in range(3):
            a, b = (-half[k] - m[k]) / d[k], (half[k] - m[k]) / d[k]
            t0, t1 = torch.maximum(t0, torch.minimum(a, b)), torch.minimum(t1, torch.maximum(a, b))
        return t0 <= t1, t0

    step = max(1, 24_000_000 // max(1, len(kinds)))
    for lo in range(0, len(origins), step):
        sel = slice(lo, min(lo + step, len(origins)))
        o, d = origins[sel], dirs[sel]
        for kind in (scenes.SPHERE, scenes.CAPSULE, scenes.BOX):
            c = kinds == kind
            if not bool(c.any()):
                continue
            p, r, R = pos[c], prm[c], rot[c]
            m = o[:, None, :] - p[None]
            if kind == scenes.SPHERE:
                _, hit, t = ball(m.unbind(2), d[:, None, :].expand_as(m).unbind(2), (r[:, 0] ** 2)[None])
                closer(sel, hit, t)
                continue
            lm = [(m * R[None, :, k]).sum(2) for k in range(3)]
            ld = [d @ R[:, k].T for k in range(3)]
            if kind == scenes.BOX:
                closer(sel, *slabs(lm, ld, r.unbind(1)))
                continue
            # a capsule is tested by the lines through its caps and its cylinder, a meeting
            # behind the origin counting as one at 0; its bounds keep those that lie behind out
            hh, r2 = r[:, 0][None], (r[:, 1] ** 2)[None]
            near, _ = slabs(m.unbind(2), [x[:, None] for x in d.unbind(1)],
                            (r[:, :1] * R[:, 1].abs() + r[:, 1:2]).unbind(1))
            for sign in (1.0, -1.0):
                line, _, t = ball([lm[0], lm[1] - sign * hh, lm[2]], ld, r2)
                closer(sel, near & line & (sign * (lm[1] + t * ld[1]) >= hh), t)
            a = ld[0] ** 2 + ld[2] ** 2
            b = lm[0] * ld[0] + lm[2] * ld[2]
            disc = b * b - a * (lm[0] ** 2 + lm[2] ** 2 - r2)
            t = ((-b - disc.clamp(min=0).sqrt()) / a).clamp(min=0)
            closer(sel, near & (disc >= 0) & ((lm[1] + t * ld[1]).abs() < hh), t)
    return {"collider": None, "distance": torch.where(best < math.inf, best, 0.0).cpu().numpy()}

"""Timed cases: what a program built on this library has it do, through its public entry points.

A case's "kind" names the use, the other values its sizes and options:

  frame    one interactive world, one World.step and its state per frame
  game     a world with sleep, contact events and interpolated stepping, several frames
  rollout  one world put back to a checkpoint and stepped on (planning, replays)
  batch    many box stacks / piles stepped together, every final state read
  chains   many jointed chains stepped together, every final state read
  terrain  worlds of spheres, boxes and hulls on heightfields, from a checkpoint
  large    one large sweep-and-prune world, from a checkpoint
  slots    a host-stepped World calling the Broadphase, Narrowphase and Solver slots of a frame
  solve    the Solver slot alone, over given contact and friction equations
  rays     a batch of closest-hit ray casts into a world
  serve    requests submitted, ticked until all are done, results read

Sizes follow the scenes of cannon_physics_amd.scenes: worlds of 8 to 512 bodies in batches,
chains of 4 to 64 links, terrains of 16 to 1024 bodies, a large world of thousands.
"""
import ctypes as C
import math
import random

import numpy as np

from cannon_physics_amd import _abi as A
from cannon_physics_amd import objects, scenes
from cannon_physics_amd.world import Context, World

DT = 1 / 60
FIELDS = ("position", "quaternion", "velocity", "angular_velocity")


def listed():
    return [
        # the smallest call: the demo scene's 216 spheres, a step and its state per frame
        {"name": "frame_spheres", "kind": "frame", "n": 216, "scene": "spheres"},
        # a game's frames: sleep, events to listeners, interpolated poses
        {"name": "game_pile", "kind": "game", "n": 180, "frames": 6},
        # planning in one mid-sized world: half a second from a checkpoint
        {"name": "rollout_pile", "kind": "rollout", "n": 300, "scene": "pile", "steps": 30, "sap": False, "split": False,
         "f64": False},
        # the same in the reference's own arithmetic, with sweep-and-prune
        {"name": "rollout_f64_sap", "kind": "rollout", "n": 157, "scene": "stack", "steps": 20, "sap": True,
         "split": False, "f64": True},
        # data generation: a large batch of uneven stacks and piles
        {"name": "batch_piles", "kind": "batch", "worlds": 2048, "lo": 8, "hi": 512, "steps": 60, "f64": False},
        # articulated bodies: every joint type, 4 to 64 links
        {"name": "batch_chains", "kind": "chains", "worlds": 1024, "lo": 4, "hi": 64, "steps": 30},
        # terrain: hulls and boxes against heightfield pillars
        {"name": "batch_terrain", "kind": "terrain", "worlds": 24, "lo": 16, "hi": 1024, "steps": 20},
        # the largest single world
        {"name": "large_sap", "kind": "large", "n": 16384, "steps": 3},
        # the drop-in slots of a World that steps on the host
        {"name": "slots_pile", "kind": "slots", "n": 450},
        # the solver slot over many equations
        {"name": "solve_lattice", "kind": "solve", "n": 1500},
        # a sensor's or a renderer's rays into a crowded scene
        {"name": "rays_scene", "kind": "rays", "n": 2000, "rays": 16384},
        # serving: requests of their own sizes and lengths through the queue
        {"name": "serve_piles", "kind": "serve", "requests": 48, "lo": 8, "hi": 256, "max_steps": 60},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "game", "rollout", "rollout", "batch", "batch", "chains", "terrain", "large", "slots",
                       "solve", "rays", "serve"])
    if kind == "frame":
        return {"kind": kind, "n": _log(rng, 8, 480), "scene": rng.choice(["pile", "stack"])}
    if kind == "game":
        return {"kind": kind, "n": _log(rng, 16, 400), "frames": rng.randint(2, 8)}
    if kind == "rollout":
        return {"kind": kind, "n": _log(rng, 8, 1000), "scene": rng.choice(["pile", "stack"]), "steps": rng.randint(5, 40),
                "sap": rng.random() < 0.4, "split": rng.random() < 0.25, "f64": rng.random() < 0.3}
    if kind == "batch":
        return {"kind": kind, "worlds": _log(rng, 2, 1500), "lo": 8, "hi": rng.choice([64, 200, 512]),
                "steps": rng.randint(8, 50), "f64": rng.random() < 0.2}
    if kind == "chains":
        lo = rng.randint(4, 20)
        return {"kind": kind, "worlds": _log(rng, 4, 900), "lo": lo, "hi": rng.randint(lo, 64), "steps": rng.randint(5, 30)}
    if kind == "terrain":
        return {"kind": kind, "worlds": rng.randint(1, 20), "lo": 16, "hi": rng.choice([100, 400, 1024]),
                "steps": rng.randint(4, 20)}
    if kind == "large":
        return {"kind": kind, "n": _log(rng, 600, 12000), "steps": rng.randint(1, 5)}
    if kind == "slots":
        return {"kind": kind, "n": _log(rng, 16, 900)}
    if kind == "solve":
        return {"kind": kind, "n": _log(rng, 20, 2000)}
    if kind == "rays":
        return {"kind": kind, "n": _log(rng, 16, 3000), "rays": _log(rng, 1, 16384)}
    lo = rng.randint(8, 40)
    return {"kind": kind, "requests": rng.randint(2, 48), "lo": lo, "hi": rng.randint(lo, 256), "max_steps": rng.randint(8, 60)}


# ---- scenes ------------------------------------------------------------------------------------

def _seeds(seed, k):
    r = random.Random(seed * 7919 + 13)
    return [r.randrange(1 << 30) for _ in range(k)]


def _solver(case):
    return objects.SplitSolver(objects.GSSolver(iterations=10)) if case.get("split") else objects.GSSolver(iterations=10)


def _pile(seed, n, kind, sap=False, solver=None, **kw):
    """scenes.c3_world, with the given broadphase and solver"""
    w = scenes.c3_world(seed, n=n, kind=kind, **kw)
    if solver is not None:
        w.solver = solver
    if sap:
        w.broadphase = objects.SAPBroadphase()
        w.broadphase.autoDetectAxis()
    return w


def _terrain(seed, n, hulls):
    """scenes.c5_terrain_world's layout over a pool of shared hulls: bodies dropped on a rotated
    64 x 64 value-noise heightfield"""
    rng = np.random.default_rng(seed)
    w = World(gravity=(0, -9.82, 0), broadphase=objects.NaiveBroadphase(), solver=objects.GSSolver(iterations=10))
    ground = objects.Body(mass=0)
    ground.addShape(objects.Heightfield(scenes.value_noise(64, 2.0, rng), elementSize=0.5))
    ground.quaternion.setFromEuler(-math.pi / 2, 0, 0)
    w.addBody(ground)
    side = int(math.ceil(math.sqrt(n)))
    for i in range(n):
        p = (2.0 + 27.0 * ((i % side) + rng.uniform(0.2, 0.8)) / side, 2.2 + rng.uniform(0, 0.8),
             -2.0 - 27.0 * ((i // side) + rng.uniform(0.2, 0.8)) / side)
        q = scenes.shoemake_quaternion(rng)
        k = int(rng.integers(0, 3))
        if k == 0:
            w.addBody(objects.Body(mass=1.0, position=p, shape=objects.Sphere(rng.uniform(0.2, 0.45))))
        elif k == 1:
            w.addBody(objects.Body(mass=1.0, position=p, quaternion=q, shape=objects.Box(rng.uniform(0.2, 0.45, size=3))))
        else:
            w.addBody(objects.Body(mass=1.0, position=p, quaternion=q, shape=hulls[int(rng.integers(0, len(hulls)))]))
    return w


def _ray_scene(case, seed):
    """spheres and rotated boxes over the ground plane, and rays from above all of them to below
    the plane, as arrays in the precision the scene is stored in"""
    rng = np.random.default_rng(seed * 31 + 5)
    n, m = case["n"], case["rays"]
    side = 2.0 * math.sqrt(n)
    f = np.float32
    pos = np.stack([rng.uniform(0, side, n), rng.uniform(0.5, 6.0, n), rng.uniform(0, side, n)], 1).astype(f)
    is_box = rng.random(n) < 0.5
    radius = rng.uniform(0.2, 0.6, n)
    half = rng.uniform(0.2, 0.6, (n, 3)).astype(f)
    u = rng.random((n, 3))
    a, b = np.sqrt(1 - u[:, 0]), np.sqrt(u[:, 0])
    quat = np.stack([a * np.sin(2 * np.pi * u[:, 1]), a * np.cos(2 * np.pi * u[:, 1]), b * np.sin(2 * np.pi * u[:, 2]),
                     b * np.cos(2 * np.pi * u[:, 2])], 1).astype(f)
    src = np.stack([rng.uniform(0, side, m), rng.uniform(8.0, 10.0, m), rng.uniform(0, side, m)], 1).astype(f)
    dst = (src + np.stack([rng.uniform(-6, 6, m), np.full(m, -12.0), rng.uniform(-6, 6, m)], 1)).astype(f)
    return pos, is_box, radius, half, quat, src, dst


def _lattice(case, seed):
    """touching unit spheres on a jittered lattice and the equations of their contacts: two
    friction equations per contact, then the contact equations"""
    rng = np.random.default_rng(seed * 17 + 3)
    n, f = case["n"], np.float32
    s = max(1, int(math.ceil(n ** (1 / 3))))
    cell = np.array([(i % s, i // (s * s), (i // s) % s) for i in range(n)])
    pos = (cell * 0.97 + 0.48 + rng.uniform(-0.02, 0.02, (n, 3))).astype(f)
    vel, avel = rng.normal(0, 0.4, (n, 3)).astype(f), rng.normal(0, 0.4, (n, 3)).astype(f)
    index = {tuple(c): i for i, c in enumerate(cell)}
    pairs = [(i, index[k]) for i, c in enumerate(cell) for k in ((c[0] - 1, c[1], c[2]), (c[0], c[1] - 1, c[2]),
                                                               (c[0], c[1], c[2] - 1)) if k in index]
    a = np.array([p[0] for p in pairs] + [i for i, c in enumerate(cell) if c[1] == 0], dtype=np.int64)
    b = np.array([p[1] for p in pairs] + [-1] * (len(a) - len(pairs)), dtype=np.int64)
    ground = b < 0
    to = np.where(ground[:, None], pos[a] * np.array([1, 0, 1]), pos[np.maximum(b, 0)]).astype(np.float64)
    nrm = to - pos[a]
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    t1 = np.cross(nrm, np.where(np.abs(nrm[:, :1]) < 0.9, [[1.0, 0, 0]], [[0, 1.0, 0]]))
    t1 /= np.linalg.norm(t1, axis=1, keepdims=True)
    t2 = np.cross(nrm, t1)
    nrm, t1, t2 = nrm.astype(f), t1.astype(f), t2.astype(f)
    ri = (nrm * f(0.5)).astype(f)
    rj = np.where(ground[:, None], pos[a] * np.array([1, 0, 1], f), -nrm * f(0.5)).astype(f)
    k = len(a)
    d, h = 3.0, DT
    e = {"kind": np.r_[np.full(2 * k, A.ROW_FRICTION), np.full(k, A.ROW_CONTACT)],
         "body_i": np.r_[np.repeat(a, 2), a] + 1, "body_j": np.r_[np.repeat(b, 2), b] + 1,
         "ri": np.r_[np.repeat(ri, 2, 0), ri], "rj": np.r_[np.repeat(rj, 2, 0), rj],
         "n": np.r_[np.stack([t1, t2], 1).reshape(-1, 3), nrm],
         "min_force": np.r_[np.full(2 * k, -0.3 * 9.82), np.zeros(k)],
         "max_force": np.r_[np.full(2 * k, 0.3 * 9.82), np.full(k, 1e6)],
         "a": np.full(3 * k, 4.0 / (h * (1 + 4 * d))), "b": np.full(3 * k, 4.0 * d / (1 + 4 * d)),
         "eps": np.full(3 * k, 4.0 / (h * h * 1e7 * (1 + 4 * d))), "restitution": np.full(3 * k, 0.3)}
    # body 0 is the ground plane
    return pos, vel, avel, e


# ---- states ------------------------------------------------------------------------------------

class _Worlds:
    """worlds of one context, with one host buffer for the state of all of them"""

    def __init__(self, f64=False):
        self.ctx = Context(precision=A.PRECISION_F64 if f64 else A.PRECISION_F32)
        self.ids, self.counts = [], []

    def add(self, recipe, copies=1):
        for _ in range(copies):
            w = self.ctx.create_world(recipe)
            self.ids.append(w)
            self.counts.append(self.ctx.num_bodies(w))

    def close_up(self):
        total = sum(self.counts)
        self.buf = (A.BodyState * total)()
        self.np = np.ctypeslib.as_array(self.buf)
        starts = np.cumsum([0] + self.counts[:-1])
        size = C.sizeof(A.BodyState)
        base = C.addressof(self.buf)
        self.parts = [(w, C.cast(base + int(s) * size, C.POINTER(A.BodyState)), n)
                      for w, s, n in zip(self.ids, starts, self.counts)]
        return self

    def download(self):
        lib, p = self.ctx.lib, self.ctx.ptr
        for w, at, n in self.parts:
            self.ctx.check(lib.chp_state_download(p, w, at, n))
        return self.np

    def upload(self):
        lib, p = self.ctx.lib, self.ctx.ptr
        for w, at, n in self.parts:
            self.ctx.check(lib.chp_state_upload(p, w, at, n))

    def state(self):
        s = self.download()
        return {k: s[k] for k in FIELDS}

    def checkpoint(self):
        self.saved = self.download().copy()

    def restore(self):
        self.np[:] = self.saved
        self.upload()

    def jitter(self, seed):
        """copies of one recipe part ways: a small velocity of its own for every dynamic body"""
        s = self.download()
        rng = np.random.default_rng(seed)
        kick = rng.normal(0, 0.05, (len(s), 3)).astype(np.float32)
        kick[np.cumsum([0] + self.counts[:-1])] = 0   # body 0 of a world is its ground
        s["velocity"] += kick
        self.upload()

    def __del__(self):
        self.ctx.close()


def _sizes(case, k):
    """k body counts spread evenly over the logarithm of the range"""
    return [int(round(case["lo"] * (case["hi"] / case["lo"]) ** ((j + 0.5) / k))) for j in range(k)]


def _padded(a, cap):
    """a fixed-size result buffer holding a's values, zero beyond them"""
    out = np.zeros((cap,) + a.shape[1:], a.dtype)
    out[: len(a)] = a
    return out


def prepare(case, seed):
    return {"frame": _p_frame, "game": _p_game, "rollout": _p_rollout, "batch": _p_batch, "chains": _p_chains,
            "terrain": _p_terrain, "large": _p_large, "slots": _p_slots, "solve": _p_solve, "rays": _p_rays,
            "serve": _p_serve}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _p_frame(case, seed):
    s = _seeds(seed, 1)[0]
    w = _Worlds()
    if case["scene"] == "spheres":
        scene = scenes.c1_spheres(s)
    else:
        scene = _pile(s, case["n"], case["scene"])
    w.add(scene.recipe())
    w.close_up()
    w.ctx.step(w.ids, DT, 90)   # the bodies have landed
    return {"run": _r_frame, "w": w}


def _r_frame(s):
    s["w"].ctx.step(s["w"].ids, DT, 1)
    return s["w"].state()


def _p_game(case, seed):
    w = _Worlds()
    w.add(_pile(_seeds(seed, 1)[0], case["n"], "pile", allowSleep=True).recipe())
    w.close_up()
    w.ctx.set_events(w.ids[0])
    w.ctx.step(w.ids, DT, 60)
    w.ctx.events(w.ids[0])
    w.checkpoint()
    return {"run": _r_game, "w": w, "frames": case["frames"], "cap": 32 * case["n"] + 256}


def _r_game(s):
    w, ctx, wid = s["w"], s["w"].ctx, s["w"].ids[0]
    w.restore()
    ctx.set_time(wid, 1.0)
    out = {}
    for k in range(s["frames"]):   # a 30 Hz display over a 60 Hz simulation
        ctx.step_interpolated(wid, DT, 2 * DT, 10)
        ev = _padded(ctx.events(wid), s["cap"])
        p, q = ctx.interpolated(wid)
        out["frame%d" % k] = {"kind": ev["kind"], "bodies": np.stack([ev["body_a"], ev["body_b"]]), "point": ev["ri"],
                              "normal": ev["ni"], "position": p, "quaternion": q}
    return out


def _p_rollout(case, seed):
    w = _Worlds(case["f64"])
    w.add(_pile(_seeds(seed, 1)[0], case["n"], case["scene"], case["sap"], _solver(case)).recipe())
    w.close_up()
    w.ctx.step(w.ids, DT, 60)
    w.checkpoint()
    return {"run": _r_rollout, "w": w, "steps": case["steps"]}


def _r_rollout(s):
    s["w"].restore()
    s["w"].ctx.step(s["w"].ids, DT, s["steps"])
    return s["w"].state()


def _r_batch(s):
    s["w"].ctx.step(s["w"].ids, DT, s["steps"])
    return s["w"].state()


def _p_batch(case, seed):
    # a few dozen scenes, each in several copies that part ways
    k = min(case["worlds"], 64)
    w = _Worlds(case["f64"])
    sizes = _sizes(case, k)
    for j, s in enumerate(_seeds(seed, k)):
        w.add(_pile(s, sizes[j], "stack" if j % 2 else "pile").recipe(), (case["worlds"] - j + k - 1) // k)
    w.close_up()
    w.jitter(seed)
    w.ctx.step(w.ids, DT, 150)   # the piles have formed
    return {"run": _r_batch, "w": w, "steps": case["steps"]}


def _p_chains(case, seed):
    k = min(case["worlds"], 64)
    w = _Worlds()
    for j, s in enumerate(_seeds(seed, k)):
        length = case["lo"] + (case["hi"] - case["lo"]) * j // max(1, k - 1)
        w.add(scenes.c4_chain_world(s, length=length).recipe(), (case["worlds"] - j + k - 1) // k)
    w.close_up()
    w.jitter(seed)
    w.ctx.step(w.ids, DT, 60)   # the columns are falling over
    return {"run": _r_batch, "w": w, "steps": case["steps"]}


def _p_terrain(case, seed):
    w = _Worlds()
    rng = np.random.default_rng(seed)
    hulls = [scenes.random_hull(rng, rng.uniform(0.2, 0.45)) for _ in range(6)]
    sizes = _sizes(case, case["worlds"])
    for j, s in enumerate(_seeds(seed, case["worlds"])):
        w.add(_terrain(s, sizes[j], hulls).recipe())
    w.close_up()
    w.ctx.step(w.ids, DT, 45)   # the bodies have landed
    w.checkpoint()
    return {"run": _r_rollout, "w": w, "steps": case["steps"]}


def _p_large(case, seed):
    # the large world's density (its 64 x 64 m ground scaled to the body count), close above the
    # ground, so that a pile has formed after the first steps
    side = max(4.0, 64.0 * math.sqrt(case["n"] / 32768.0))
    w = _Worlds()
    w.add(scenes.c2_large_world(seed, n=case["n"], extent=(side, 8.0, side)).recipe())
    w.close_up()
    w.ctx.step(w.ids, DT, 60)
    w.checkpoint()
    return {"run": _r_rollout, "w": w, "steps": case["steps"]}


def _p_slots(case, seed):
    w = _Worlds()
    w.add(_pile(_seeds(seed, 1)[0], case["n"], "pile").recipe())
    w.close_up()
    w.ctx.step(w.ids, DT, 60)
    s = w.download()
    info, _ = w.ctx.body_info(w.ids[0])
    mass = np.array([info[i].mass for i in range(len(s))])
    s["force"][:, 1] += (mass * -9.82).astype(np.float32)   # the World adds gravity before its slots
    w.saved = s.copy()
    return {"run": _r_slots, "w": w, "pair_cap": 48 * len(s) + 256, "eq_cap": 40 * len(s) + 800}


def _r_slots(s):
    w, ctx, wid = s["w"], s["w"].ctx, s["w"].ids[0]
    w.restore()
    pi, pj = ctx.broadphase(wid, s["pair_cap"])
    eqs, n, nf, nc = ctx.narrowphase(wid, pi, pj, DT, s["eq_cap"])
    it, mult = ctx.solve(wid, eqs, n, DT)
    e = np.ctypeslib.as_array(eqs)   # as long as its buffer, zero beyond n
    mult = _padded(mult, s["eq_cap"])
    return {"count": n, "pairs": _padded(np.stack([pi, pj], 1), s["pair_cap"]), "bodies": np.stack([e["body_i"], e["body_j"]]), "ri": e["ri"], "rj": e["rj"],
            "n": e["n"], "iterations": it, "multipliers": mult, "state": w.state()}


def _p_solve(case, seed):
    pos, vel, avel, e = _lattice(case, seed)
    scene = World(gravity=(0, -9.82, 0), broadphase=objects.NaiveBroadphase(), solver=objects.GSSolver(iterations=10))
    scene.addBody(scenes.ground_plane())
    ball = objects.Sphere(0.5)
    for p in pos:
        scene.addBody(objects.Body(mass=1, position=p.tolist(), shape=ball))
    w = _Worlds()
    w.add(scene.recipe())
    w.close_up()
    rows = len(e["kind"])
    w.ctx.set_capacity(w.ids[0], max_rows=rows + 64)
    s = w.download()
    s["velocity"][1:], s["angular_velocity"][1:] = vel, avel
    s["force"][1:, 1] = np.float32(-9.82)
    w.saved = s.copy()
    eqs = (A.Equation * rows)()
    arr = np.ctypeslib.as_array(eqs)
    for k, v in e.items():
        arr[k] = v
    return {"run": _r_solve, "w": w, "eqs": eqs, "rows": rows}


def _r_solve(s):
    w = s["w"]
    w.restore()
    it, mult = w.ctx.solve(w.ids[0], s["eqs"], s["rows"], DT)
    st = w.download()
    return {"iterations": it, "multipliers": mult, "velocity": st["velocity"], "angular_velocity": st["angular_velocity"]}


def _p_rays(case, seed):
    pos, is_box, radius, half, quat, src, dst = _ray_scene(case, seed)
    scene = World(gravity=(0, -9.82, 0), broadphase=objects.NaiveBroadphase(), solver=objects.GSSolver(iterations=10))
    scene.addBody(scenes.ground_plane())
    for k in range(case["n"]):
        shape = objects.Box(half[k].tolist()) if is_box[k] else objects.Sphere(float(radius[k]))
        scene.addBody(objects.Body(mass=1, position=pos[k].tolist(), shape=shape,
                                   quaternion=objects.Quaternion(*quat[k].tolist())))
    w = _Worlds()
    w.add(scene.recipe())
    w.close_up()
    m = case["rays"]
    rays, hits = (A.Ray * m)(), (A.RayHit * m)()
    r = np.ctypeslib.as_array(rays)
    r["from_" if "from_" in r.dtype.names else "from"], r["to"] = src, dst
    r["mode"] = A.RAY_CLOSEST
    r["skip_backfaces"] = 1
    r["check_collision_response"] = 1
    r["collision_filter_group"] = r["collision_filter_mask"] = -1
    return {"run": _r_rays, "w": w, "rays": rays, "hits": hits, "m": m}


def _r_rays(s):
    ctx, n = s["w"].ctx, C.c_uint32()
    ctx.check(ctx.lib.chp_raycast(ctx.ptr, s["w"].ids[0], s["rays"], s["m"], s["hits"], s["m"], C.byref(n)))
    h = np.ctypeslib.as_array(s["hits"])[: n.value]
    return {"ray": h["ray"], "body": h["body"], "shape": h["shape"], "distance": h["distance"], "point": h["point"],
            "normal": h["normal"]}


def _p_serve(case, seed):
    k = case["requests"]
    sizes = _sizes(case, k)
    recs = [(_pile(s, sizes[j], "pile" if j % 2 else "stack").recipe(), 4 + j * 7 % (case["max_steps"] - 3), sizes[j] + 1)
            for j, s in enumerate(_seeds(seed, k))]
    return {"run": _r_serve, "ctx": Context(), "recs": recs}


def _r_serve(s):
    ctx = s["ctx"]
    tickets = [ctx.serve_submit(rec, DT, steps) for rec, steps, _ in s["recs"]]
    while sum(ctx.serve_tick(8)):
        pass
    done = [np.ctypeslib.as_array(ctx.serve_result(t, n))[:n] for t, (_, _, n) in zip(tickets, s["recs"])]
    return {k: np.concatenate([d[k] for d in done]) for k in FIELDS}


# ---- what a pass cannot do without ---------------------------------------------------------------

BODY = 104 + 104 + 72        # state in, state out, constants
ROW_FLOPS = 60 + 160 / 10    # a row's sweep, and its set-up spread over 10 sweeps


def work(case):
    """bytes: every body's state and constants in and its state out once.  flops: the solver rows
    (about 9 per body of a pile: three contacts of three rows) over the iterations, and an
    integration per step."""
    k = case["kind"]
    mean = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"]) if case.get("hi", 0) > case.get("lo", 0) else case.get("lo", 0)
    if k == "rays":
        return {"bytes": 280 * case["n"] + case["rays"] * (C.sizeof(A.Ray) + C.sizeof(A.RayHit)), "flops": 300.0 * case["rays"]}
    if k == "solve":
        rows = 9 * case["n"]
        return {"bytes": BODY * case["n"] + rows * (C.sizeof(A.Equation) + 8), "flops": 10.0 * rows * ROW_FLOPS}
    if k == "chains":
        bodies, steps, rows, iters = case["worlds"] * (case["lo"] + case["hi"]) / 2, case["steps"], 4.0, 20
    elif k in ("batch", "terrain"):
        bodies, steps, rows, iters = case["worlds"] * mean, case["steps"], 9.0, 10
    elif k == "serve":
        bodies, steps, rows, iters = case["requests"] * mean, (4 + case["max_steps"]) / 2, 9.0, 10
    else:
        bodies, rows, iters = case["n"], 9.0, 10
        steps = case.get("steps", 2 * case["frames"] if k == "game" else 1)
    return {"bytes": float(BODY * bodies), "flops": bodies * steps * (rows * iters * ROW_FLOPS + 100.0)}


# ---- 64-bit values -------------------------------------------------------------------------------

def exact(case, seed):
    """The solver slot and the ray casts have values of their own; a trajectory of contacts has
    none (which contacts there are, and which friction rows clamp, is decided in the step's own
    arithmetic)."""
    if case["kind"] == "solve":
        return _exact_solve(case, seed)
    if case["kind"] == "rays":
        return _exact_rays(case, seed)
    return None


def _exact_solve(case, seed):
    pos, vel, avel, e = _lattice(case, seed)
    z = np.zeros((1, 3))
    p, v, w = (np.concatenate([z, x.astype(np.float64)]) for x in (pos, vel, avel))
    f = np.zeros_like(p)
    f[1:, 1] = np.float32(-9.82)
    im = np.ones(len(p))
    im[0] = 0
    # a sphere's inertia here is that of its bounding cube: m / 12 * ((2r)^2 + (2r)^2)
    ii = im * 6.0
    a, b = e["body_i"], e["body_j"]
    ri, rj, n = (e[k].astype(np.float64) for k in ("ri", "rj", "n"))
    # stored in the solver's input records in 64 bits, used as they are
    contact = e["kind"] == A.ROW_CONTACT
    ra, rb = np.cross(ri, n), np.cross(rj, n)
    rest = np.where(contact, e["restitution"], 0.0) + 1
    dot = lambda x, y: np.einsum("ij,ij->i", x, y)  # noqa: E731
    gw = rest * (dot(v[b], n) - dot(v[a], n)) + dot(w[b], rb) - dot(w[a], ra)
    gm = dot(f[b], n) * im[b] - dot(f[a], n) * im[a]
    g = np.where(contact, dot(n, p[b] + rj - p[a] - ri), 0.0)
    rhs = -g * e["a"] - gw * e["b"] - DT * gm
    inv_c = 1 / (im[a] + im[b] + ii[a] * dot(ra, ra) + ii[b] * dot(rb, rb) + e["eps"])
    lam = [0.0] * len(a)
    dv, dw = np.zeros_like(p), np.zeros_like(p)
    # per row: J over (va, wa, vb, wb) and what an impulse adds to them
    J = np.concatenate([-n, -ra, n, rb], 1)
    M = np.concatenate([-n * im[a][:, None], -ra * ii[a][:, None], n * im[b][:, None], rb * ii[b][:, None]], 1)
    x = np.concatenate([dv, dw], 1)   # (body, 6)
    ja, jb, ma, mb = J[:, :6].copy(), J[:, 6:].copy(), M[:, :6].copy(), M[:, 6:].copy()
    al, bl, rl, cl, el = a.tolist(), b.tolist(), rhs.tolist(), inv_c.tolist(), e["eps"].tolist()
    lo, hi = e["min_force"].tolist(), e["max_force"].tolist()
    it = 0
    for it in range(1, 11):
        tot = 0.0
        for k in range(len(al)):
            xa, xb, lk = x[al[k]], x[bl[k]], lam[k]
            d = cl[k] * (rl[k] - float(ja[k] @ xa + jb[k] @ xb) - el[k] * lk)
            d = min(max(lk + d, lo[k]), hi[k]) - lk
            lam[k] = lk + d
            tot += abs(d)
            xa += d * ma[k]
            xb += d * mb[k]
        if tot * tot < 1e-14:
            break
    return {"iterations": None, "multipliers": np.array(lam) / DT, "velocity": v + x[:, :3], "angular_velocity": w + x[:, 3:]}


def _exact_rays(case, seed):
    pos, is_box, radius, half, quat, src, dst = (x.astype(np.float64) if x.dtype.kind == "f" else x
                                                 for x in _ray_scene(case, seed))
    radius = radius.astype(np.float64)
    q = quat
    x, y, z, w = q.T
    rot = np.stack([np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)], 1),
                    np.stack([2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)], 1),
                    np.stack([2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], 1)], 1)
    m = len(src)
    dist, point, normal = np.zeros(m), np.zeros((m, 3)), np.zeros((m, 3))
    ib, isph = np.nonzero(is_box)[0], np.nonzero(~is_box)[0]
    for k in range(m):
        d = dst[k] - src[k]
        best, nrm = src[k][1] / -d[1], np.array([0.0, 1.0, 0.0])
        o = src[k] - pos[isph]
        A2, B2, C2 = d @ d, o @ d, np.einsum("ij,ij->i", o, o) - radius[isph] ** 2
        disc = B2 * B2 - A2 * C2
        hit = np.nonzero(disc > 0)[0]
        if len(hit):
            t = (-B2[hit] - np.sqrt(disc[hit])) / A2
            j = int(np.argmin(t))
            if t[j] < best:
                best = t[j]
                nrm = (src[k] + best * d - pos[isph[hit[j]]]) / radius[isph[hit[j]]]
        if len(ib):
            near = np.nonzero(np.linalg.norm(np.cross(pos[ib] - src[k], d), axis=1) <= 1.1 * math.sqrt(d @ d))[0]
            for i in ib[near]:
                lo_, ld = rot[i].T @ (src[k] - pos[i]), rot[i].T @ d
                t1, t2 = (-half[i] - lo_) / ld, (half[i] - lo_) / ld
                tin, tout = np.minimum(t1, t2), np.maximum(t1, t2)
                ax = int(np.argmax(tin))
                if tin[ax] <= tout.min() and tin[ax] < best:
                    best = tin[ax]
                    nrm = rot[i][:, ax] * (-1.0 if ld[ax] > 0 else 1.0)
        point[k], normal[k], dist[k] = src[k] + best * d, nrm, best * math.sqrt(d @ d)
    return {"ray": None, "body": None, "shape": None, "distance": dist, "point": point, "normal": normal}

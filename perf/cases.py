"""The work a program has this framework do, as measurable cases.

A case is one pass of a program's loop through the public entry points (``reactphysics3d_amd.lib``):

  world    one PhysicsWorld: update() once (an interactive program, eager) or a few times (a captured step
           graph), then read the body states back
  batch    many worlds at once: apply forces, step, read back (reinforcement learning, design sweeps, a
           server's game rooms); fixed iterations or to a residual; with or without sleeping and events
  rollout  put a world back into a snapshot and step it forward (sampling-based planning)
  rays     a closest-hit ray cast against every collider of a world (sensors, picking, line of sight)
  train    train the learned warm start's network on logged samples

Worlds are stepped until they have landed before they are timed, so that the work of a pass does not
drift while a state is run again and again.  Steps are bit-exact against the reference engine for a given
solve order, and two runs of the same calls give the same bits: their outputs compare exactly.
"""
import ctypes
import math

import numpy as np
import torch

from reactphysics3d_amd import lib
from reactphysics3d_amd import scene as S
from reactphysics3d_amd.lib import Batch, Mlp

DT = 1.0 / 60.0


def listed():
    return [
        # a small interactive scene (27 boxes on a ground): one update() and its read-back, where launches
        # and latency are all there is
        {"name": "pile_27_update", "kind": "world", "scene": "pile", "n": 27, "graph": False, "steps": 1, "settle": 150},
        # machines: cone-limited chains, slider and hinge rigs with limits and motors, rolled forward from
        # one state as a planner does
        {"name": "rigs_rollout_8_steps", "kind": "rollout", "scene": "rigs", "n": 97, "graph": True, "steps": 8, "settle": 60},
        # the 1000-box pile, one interactive update()
        {"name": "pile_1000_update", "kind": "world", "scene": "pile", "n": 1000, "graph": False, "steps": 1, "settle": 150},
        # a heap of spheres, boxes and capsules that one workgroup per world still takes, captured steps
        {"name": "heap_3001_steps", "kind": "world", "scene": "heap", "n": 3001, "graph": True, "steps": 2, "settle": 120},
        # the largest single world: 65,536 spheres, boxes and capsules landed in a walled container
        {"name": "heap_65536_update", "kind": "world", "scene": "heap", "n": 65536, "graph": False, "steps": 1, "settle": 120},
        # convex meshes and chains of spheres on ball-and-socket joints
        {"name": "hulls_6000_update", "kind": "world", "scene": "hulls", "n": 6000, "graph": False, "steps": 1, "settle": 120},
        # every convex shape on a triangle-mesh terrain (the middle phase and triangle tests)
        {"name": "terrain_600_update", "kind": "world", "scene": "mesh", "n": 600, "graph": False, "steps": 1, "settle": 120},
        # a server's game rooms: sleeping islands, contact events, a few bodies pushed every frame
        {"name": "rooms_200_events", "kind": "batch", "worlds": 200, "levels": 50, "min_bodies": 8, "max_bodies": 96,
         "residual": False, "sleeping": True, "events": True, "push": 0.02, "graph": False, "steps": 1, "settle": 150},
        # reinforcement learning: every body driven, four substeps a frame, observations read back
        {"name": "envs_1024_control", "kind": "batch", "worlds": 1024, "levels": 64, "min_bodies": 8, "max_bodies": 128,
         "residual": False, "sleeping": False, "events": False, "push": 1.0, "graph": True, "steps": 4, "settle": 150},
        # the headline workload: 4096 worlds of 8 to 512 bodies, every world to the residual 1e-4
        {"name": "worlds_4096_residual", "kind": "batch", "worlds": 4096, "levels": 64, "min_bodies": 8, "max_bodies": 512,
         "residual": True, "sleeping": False, "events": False, "push": 0.0, "graph": True, "steps": 4, "settle": 60},
        # sensors: 100,000 rays from above into a crowded container
        {"name": "rays_100000", "kind": "rays", "bodies": 2000, "rays": 100000},
        # two passes over the logged samples of the learned warm start, 4096 a minibatch
        {"name": "train_65536", "kind": "train", "samples": 65536, "minibatch": 4096, "epochs": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["world", "world", "world", "rollout", "batch", "batch", "rays", "train"])
    if kind in ("world", "rollout"):
        scene = rng.choice(["pile", "heap", "hulls", "mesh", "field", "rigs"]) if kind == "world" else \
            rng.choice(["pile", "rigs", "heap"])
        most = {"pile": 2000, "heap": 40000, "hulls": 6000, "mesh": 800, "field": 800, "rigs": 600}[scene]
        n = _log_int(rng, 9, most if kind == "world" else 600)
        graph = kind == "rollout" or (n <= 3000 and rng.random() < 0.5)   # captured steps take up to 4096 bodies a world
        return {"kind": kind, "scene": scene, "n": n, "graph": graph,
                "steps": rng.randint(4, 16) if kind == "rollout" else (rng.randint(1, 4) if graph else 1), "settle": 100}
    if kind == "batch":
        residual = rng.random() < 0.4
        sleeping = not residual and rng.random() < 0.4
        lo = _log_int(rng, 5, 24)
        hi = min(512, lo * rng.randint(2, 16))
        worlds = _log_int(rng, 16, max(17, min(3000, 160000 // hi)))
        return {"kind": "batch", "worlds": worlds, "levels": min(worlds, rng.randint(8, 40)), "min_bodies": lo,
                "max_bodies": hi, "residual": residual, "sleeping": sleeping, "events": sleeping or rng.random() < 0.2,
                "push": rng.choice([0.0, 0.02, 1.0]), "graph": rng.random() < 0.7, "steps": rng.randint(1, 4), "settle": 60}
    if kind == "rays":
        bodies = _log_int(rng, 30, 3000)
        return {"kind": "rays", "bodies": bodies, "rays": _log_int(rng, 100, 100000)}
    minibatch = rng.choice([1000, 1024, 2048, 4096, 5000])
    return {"kind": "train", "samples": _log_int(rng, 2000, 65536), "minibatch": minibatch, "epochs": rng.randint(1, 2)}


# ---------------------------------------------------------------------------------------------
# scenes
# ---------------------------------------------------------------------------------------------

def _unit_quats(rng, n):
    q = rng.normal(size=(n, 4))
    return (q / np.linalg.norm(q, axis=1, keepdims=True)).astype(np.float32)


def _heap(n, seed, gravity=True, hulls=0, density=0.19, depth=12.0):
    """n bodies at random in a walled box of `depth` metres with the given share of its volume filled:
    spheres, boxes and capsules by turns (the sizes of scene.mixed_container), or convex meshes of a
    shared set of `hulls`."""
    rng = np.random.default_rng(seed)
    sc = S.Scene(f"heap_{n}", S.make_settings(gravity=(0.0, 0.0, -9.81 if gravity else 0.0)))
    volume = 1.36 if not hulls else 1.6
    half = 0.5 * max(6.0, math.sqrt(n * volume / (density * depth)))
    walls = [((0.0, 0.0, -0.5), (half + 1.0, half + 1.0, 0.5))]
    for s in (1.0, -1.0):
        walls.append(((s * (half + 0.5), 0.0, depth), (0.5, half + 1.0, depth)))
        walls.append(((0.0, s * (half + 0.5), depth), (half, 0.5, depth)))
    for pos, he in walls:
        sc.add_collider(sc.add_body(S.STATIC, pos), S.BOX, he)
    shapes = []
    for _ in range(hulls):
        axes = rng.uniform(0.3, 1.2, 3)
        d = rng.normal(size=(24, 3))
        shapes.append(sc.add_hull_from_points((axes * d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)))
    inner = half - 1.0
    pos = np.column_stack([rng.uniform(-inner, inner, n), rng.uniform(-inner, inner, n),
                           rng.uniform(1.0, depth, n)]).astype(np.float32).tolist()
    quat = _unit_quats(rng, n).tolist()
    lin = rng.normal(size=(n, 3)).astype(np.float32).tolist()
    size = rng.uniform(0.0, 1.0, (n, 3)).tolist()
    for i in range(n):
        b = sc.add_body(S.DYNAMIC, pos[i], quat[i], lin=lin[i])
        u = size[i]
        if hulls:
            sc.add_collider(b, S.HULL, (float(shapes[int(u[0] * hulls) % hulls]),), density=1000.0)
        elif i % 3 == 0:
            sc.add_collider(b, S.SPHERE, (0.25 + 0.75 * u[0],), density=1000.0)
        elif i % 3 == 1:
            sc.add_collider(b, S.BOX, tuple(0.25 + 0.75 * x for x in u), density=1000.0)
        else:
            sc.add_collider(b, S.CAPSULE, (0.2 + 0.3 * u[0], 0.5 + 1.5 * u[1]), density=1000.0)
    return sc


def _pile(n, seed):
    """n unit boxes in the grid of scene.box_pile (a cube of them, the last layer cut off)."""
    side = max(1, round(n ** (1.0 / 3.0)))
    levels = -(-n // (side * side))
    sc = S.box_pile(side, levels, seed=seed)
    del sc.bodies[1 + n:], sc.colliders[1 + n:]
    return sc


def _rigs(n, seed):
    """About n bodies: chains with cone limits, slider and hinge rigs, all with 10 / 5 iterations."""
    chains, rigs = max(1, n // 12), max(1, n // 12)
    sc = S.Scene(f"rigs_{n}", S.make_settings(gravity=(0.0, 0.0, -9.81), vel_iters=10, pos_iters=5))
    S.cone_chains(chains, 4, seed=seed, sc=sc)
    S.slider_rigs(rigs, seed=seed + 1, sc=sc)
    S.hinge_rigs(rigs, seed=seed + 2, sc=sc)
    return sc


def _scene(case, seed):
    kind, n = case["scene"], case["n"]
    if kind == "pile":
        return _pile(n, seed)
    if kind == "heap":
        return _heap(n, seed)
    if kind == "rigs":
        return _rigs(n, seed)
    if kind == "hulls":
        sc = _heap(n, seed, hulls=48)
        return S.sphere_chains(max(1, n // 100), 16, seed=seed + 1, sc=sc)
    cells = max(10, int(1.6 * math.sqrt(n)))
    return S.concave_scene("mesh" if kind == "mesh" else "heightfield", n_bodies=n, nx=cells, seed=seed)


class _Copies(Batch):
    """A batch of `count` worlds that repeat a list of built worlds (the levels of a game, the variants of a
    training environment) through rp3dg_batch_create."""

    def __init__(self, scenes, count):
        self.h = None
        self.worlds = [lib.world_from_scene(sc) for sc in scenes]
        self.scenes = [scenes[w % len(scenes)] for w in range(count)]
        handles = (ctypes.c_void_p * count)(*[self.worlds[w % len(scenes)] for w in range(count)])
        self.h = lib.load().rp3dg_batch_create(handles, count)
        if not self.h:
            raise RuntimeError("rp3dg_batch_create failed: " + lib.last_error())
        sizes = [[f(sc) for sc in self.scenes] for f in (lambda s: s.nb_bodies, lambda s: len(s.colliders),
                                                         lambda s: len(s.joints))]
        self.body_base, self.collider_base, self.joint_base = (np.cumsum([0] + s) for s in sizes)
        self.nb = int(self.body_base[-1])


def _step(batch, case):
    if case["graph"]:
        batch.step_graph(DT, case["steps"])
    else:
        batch.step(DT, case["steps"])


# ---------------------------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("world", "rollout"):
        batch = Batch(_scene(case, seed))
        batch.step(DT, case["settle"])
        _step(batch, case)
        state = {"case": case, "batch": batch}
        if kind == "rollout":
            state["snapshot"] = batch.snapshot()
        return state
    if kind == "batch":
        rng = np.random.default_rng(seed)
        # the levels are the program's; what differs from run to run is how their copies start
        scenes = [S.batched_world(i, min_bodies=case["min_bodies"], max_bodies=case["max_bodies"])
                  for i in range(case["levels"])]
        for sc in scenes:
            sc.settings["sleeping"] = int(case["sleeping"])
        batch = _Copies(scenes, case["worlds"])
        dynamic = np.concatenate([np.array([b[0] == S.DYNAMIC for b in sc.bodies]) for sc in batch.scenes])
        lin = rng.normal(0.0, 0.2, (batch.nb, 3)).astype(np.float32)
        lin[~dynamic] = 0.0
        batch.set_bodies(lin=lin)
        if case["events"]:
            batch.set_contact_events(True)
        batch.step(DT, case["settle"])
        if case["residual"]:
            batch.set_residual_mode(1e-4, 100)
        pushes = []
        if case["push"] > 0.0:
            for _ in range(4):   # the controls of four frames, given by turns
                f = rng.normal(0.0, 3.0 if case["push"] == 1.0 else 15.0, (batch.nb, 3)).astype(np.float32)
                f[~dynamic | (rng.random(batch.nb) >= case["push"])] = 0.0
                pushes.append(f)
        _step(batch, case)
        return {"case": case, "batch": batch, "pushes": pushes, "pass": 0}
    if kind == "rays":
        rng = np.random.default_rng(seed)
        scene = _heap(case["bodies"], seed)
        n, half = case["rays"], max(-b[1][0] for b in scene.bodies[:5]) - 1.0
        p1 = np.column_stack([rng.uniform(-half, half, n), rng.uniform(-half, half, n), rng.uniform(16.0, 20.0, n)])
        p2 = np.column_stack([rng.uniform(-half, half, n), rng.uniform(-half, half, n), rng.uniform(-3.0, 6.0, n)])
        return {"case": case, "batch": Batch(scene), "scene": scene, "p1": p1.astype(np.float32), "p2": p2.astype(np.float32)}
    x, t, p0 = _samples(case, seed)
    net = Mlp(seed=7)
    net.set_normalization(x.mean(0), 1.0 / (x.std(0) + 1e-6), t.std(0) + 1e-6)
    return {"case": case, "net": net, "x": x, "t": t, "p0": p0}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "rays":
        collider, point, normal, fraction = state["batch"].raycast(state["p1"], state["p2"])
        return {"collider": collider, "point": point, "normal": normal, "fraction": fraction}
    if kind == "train":
        net = state["net"]
        net.set_params(state["p0"])
        loss = net.train(state["x"], state["t"], epochs=case["epochs"], minibatch=case["minibatch"], lr=2e-3, seed=11)
        return {"params": net.params(), "loss": loss}
    batch = state["batch"]
    if kind == "rollout":
        batch.restore(state["snapshot"])
    if kind == "batch" and state["pushes"]:
        batch.apply_forces(state["pushes"][state["pass"] % 4])
        state["pass"] += 1
    _step(batch, case)
    out = dict(zip(("position", "orientation", "linear", "angular"), batch.bodies()))
    if kind == "batch" and case["sleeping"]:
        out["sleeping"] = batch.sleeping()
    if kind == "batch" and case["events"]:
        events = batch.contact_events()
        out["events"] = np.full((max(8 * batch.nb, len(events)), 4), -1, np.int32)   # a fixed-size record of the frame
        out["events"][:len(events)] = events
    return out


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without, and how far another correct implementation may be
# ---------------------------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "rays":
        # 32 B in, 32 B out a ray; every collider of the world once; the box test against each is the
        # reference's tree walk at its least (log2 of the colliders), the shape test a few times a ray
        n, c = case["rays"], case["bodies"] + 5
        return {"bytes": 64.0 * n + 120.0 * c, "flops": n * (24.0 * math.log2(c) + 200.0)}
    if kind == "train":
        n, e = case["samples"], case["epochs"]
        return {"bytes": e * (108.0 * n + 4.0 * 20099 * 6 * math.ceil(n / case["minibatch"])), "flops": 3.0 * 39680 * n * e}
    if kind == "batch":
        lo, hi = case["min_bodies"], case["max_bodies"]
        mean = (hi - lo) / math.log(hi / lo) if hi > lo else lo   # body counts are log-uniform
        n, iters = case["worlds"] * mean, 60 if case["residual"] else 10
    else:
        n, iters = case["n"], 10 if case["scene"] in ("pile", "rigs") else 6
    # per body and step: its state read and written once (16 vectors of 16 B), its collider's box, and about one
    # contact manifold of 2.5 points with its cache read and written; per point and iteration the normal and the
    # split row, per manifold two friction rows and the twist
    return {"bytes": case["steps"] * n * (256.0 + 112.0 + 2.0 * (2.5 * 48.0 + 64.0)),
            "flops": case["steps"] * n * iters * (2.5 * 180.0 + 330.0)}


def tolerance(case):
    if case["kind"] == "rays":
        # 32-bit ray tests: the hit moves by rounding (1e-6 of its size), and a ray that grazes an edge may
        # hit its neighbour instead
        return {"rel": 1e-3, "max": 0.5, "differ": 1e-4}
    if case["kind"] == "train":
        # bf16 products; Adam divides by the root of the running square, so small gradients carry their
        # rounding into the weights at full size
        return {"rel": 2e-2, "max": 0.5}
    return "exact"


# ---------------------------------------------------------------------------------------------
# 64-bit answers
# ---------------------------------------------------------------------------------------------

def exact(case, seed):
    """Rays and training in 64 bits.  A step has none: it is thousands of ordered corrections, each with
    branches on the one before (which contacts exist, which are clamped), defined only together with the
    solve order; its outputs are compared bit for bit instead."""
    if case["kind"] == "rays":
        return _exact_rays(case, seed)
    if case["kind"] == "train":
        return _exact_train(case, seed)
    return None


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _samples(case, seed):
    """Samples like the log's (unit normals, lever arms, velocities, masses, impulses that follow from them) and
    the weights the training starts from."""
    rng = np.random.default_rng(seed)
    n = case["samples"]
    x = rng.normal(size=(n, 24)).astype(np.float32)
    x[:, :3] /= np.linalg.norm(x[:, :3], axis=1, keepdims=True)
    x[:, 12:14] = rng.uniform(0.2, 2.0, (n, 2))
    x[:, 16] = rng.integers(0, 5, n)
    x[:, 18:20] = rng.integers(0, 9, (n, 2))
    x[:, 20] = np.abs(x[:, 20]) * 0.01
    x[:, 21] = rng.uniform(0.1, 0.9, n)
    x[:, 22] = rng.uniform(0.2, 2.0, n)
    x[:, 23] = 1.0 / rng.integers(1, 5, n)
    w = rng.normal(size=(24, 3)).astype(np.float32) / 5.0
    t = np.tanh(x @ w) * x[:, 22:23] + 0.05 * rng.normal(size=(n, 3)).astype(np.float32)
    limit = [(24, 128), (128, 128), (128, 3)]
    p = [np.concatenate([(rng.uniform(-1, 1, i * o) * math.sqrt(6.0 / (i + o))), np.zeros(o)]) for i, o in limit]
    return x, t.astype(np.float32), np.concatenate(p).astype(np.float32)


def _exact_train(case, seed):
    x, t, p0 = _samples(case, seed)
    mu, inv, scale = (a.astype(np.float32) for a in (x.mean(0), 1.0 / (x.std(0) + 1e-6), t.std(0) + 1e-6))
    dev = _device()
    put = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.float64)).to(dev)  # noqa: E731
    xd, td = (put(x) - put(mu)) * put(inv), put(t) / put(scale)
    sizes, weights, o = [(24, 128), (128,), (128, 128), (128,), (128, 3), (3,)], [], 0
    for s in sizes:
        k = int(np.prod(s))
        weights.append(put(p0[o:o + k]).reshape(s).requires_grad_())
        o += k
    m, v = [torch.zeros_like(w) for w in weights], [torch.zeros_like(w) for w in weights]
    n, mask, st, step, loss = case["samples"], (1 << 64) - 1, 11, 0, 0.0
    for _ in range(case["epochs"]):
        perm = list(range(n))
        for i in range(n - 1, 0, -1):   # splitmix64, Fisher-Yates
            st = (st + 0x9E3779B97F4A7C15) & mask
            z = ((st ^ (st >> 30)) * 0xBF58476D1CE4E5B9) & mask
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
            j = (z ^ (z >> 31)) % (i + 1)
            perm[i], perm[j] = perm[j], perm[i]
        perm = torch.tensor(perm, device=dev)
        for b in range(0, n, case["minibatch"]):
            idx = perm[b:b + case["minibatch"]]
            w1, b1, w2, b2, w3, b3 = weights
            h = torch.nn.functional.silu(xd[idx] @ w1 + b1)
            h = torch.nn.functional.silu(h @ w2 + b2)
            loss = 0.5 * ((h @ w3 + b3 - td[idx]) ** 2).sum() / len(idx)
            grads = torch.autograd.grad(loss, weights)
            step += 1
            with torch.no_grad():
                for w, g, mm, vv in zip(weights, grads, m, v):
                    mm.mul_(0.9).add_(g, alpha=0.1)
                    vv.mul_(0.999).addcmul_(g, g, value=0.001)
                    w -= 2e-3 * (mm / (1.0 - 0.9 ** step)) / ((vv / (1.0 - 0.999 ** step)).sqrt() + 1e-8)
    params = torch.cat([w.detach().reshape(-1) for w in weights]).cpu().numpy()
    return {"params": params, "loss": float(loss.detach())}


def _rotate(q, v):
    """v turned by the unit quaternion q (x, y, z, w), row by row."""
    u, w = q[..., :3], q[..., 3:4]
    c = torch.linalg.cross(u.expand_as(v), v)
    return v + 2.0 * (w * c + torch.linalg.cross(u.expand_as(v), c))


def _exact_rays(case, seed):
    scene = _heap(case["bodies"], seed)
    dev = _device()
    n = case["rays"]
    if dev == "cpu" and n * case["bodies"] > 2e7:
        return None
    rng = np.random.default_rng(seed)
    half = max(-b[1][0] for b in scene.bodies[:5]) - 1.0
    p1 = np.column_stack([rng.uniform(-half, half, n), rng.uniform(-half, half, n), rng.uniform(16.0, 20.0, n)])
    p2 = np.column_stack([rng.uniform(-half, half, n), rng.uniform(-half, half, n), rng.uniform(-3.0, 6.0, n)])
    a, b = (torch.from_numpy(p.astype(np.float32).astype(np.float64)).to(dev) for p in (p1, p2))
    d = b - a
    best = torch.full((n,), 2.0, dtype=torch.float64, device=dev)
    normal = torch.zeros((n, 3), dtype=torch.float64, device=dev)
    for body, col in zip(scene.bodies, scene.colliders):
        f64 = lambda x: torch.tensor(np.asarray(x, np.float32).astype(np.float64), device=dev)  # noqa: E731
        pos, quat, par = f64(body[1]), f64(body[2]), f64(col[2])
        back = torch.cat([-quat[:3], quat[3:]])
        o, r = _rotate(back, a - pos), _rotate(back, d)
        if col[1] == S.BOX:
            t1, t2 = (-par[:3] - o) / r, (par[:3] - o) / r
            enter, axis = torch.minimum(t1, t2).max(1)
            hit = (enter <= torch.maximum(t1, t2).min(1)[0]) & (enter >= 0.0)
            nrm = torch.zeros_like(o).scatter_(1, axis[:, None], -torch.sign(r.gather(1, axis[:, None])))
            t = torch.where(hit, enter, torch.full_like(enter, 3.0))
        else:
            rad = par[0]
            hh = 0.5 * par[1] if col[1] == S.CAPSULE else torch.zeros_like(rad)
            t, nrm = torch.full_like(best, 3.0), torch.zeros_like(o)
            for s in ((-1.0, 1.0) if col[1] == S.CAPSULE else (0.0,)):
                m = o - torch.stack([torch.zeros_like(hh), s * hh, torch.zeros_like(hh)])
                rr, mr, mm = (r * r).sum(1), (m * r).sum(1), (m * m).sum(1) - rad * rad
                disc = mr * mr - rr * mm
                ts = (-mr - disc.clamp(min=0.0).sqrt()) / rr
                take = (disc >= 0.0) & (ts >= 0.0) & (ts < t)
                t = torch.where(take, ts, t)
                nrm = torch.where(take[:, None], m + ts[:, None] * r, nrm)
            if col[1] == S.CAPSULE:
                rr = r[:, 0] ** 2 + r[:, 2] ** 2
                mr = o[:, 0] * r[:, 0] + o[:, 2] * r[:, 2]
                mm = o[:, 0] ** 2 + o[:, 2] ** 2 - rad * rad
                disc = mr * mr - rr * mm
                ts = (-mr - disc.clamp(min=0.0).sqrt()) / rr
                y = o[:, 1] + ts * r[:, 1]
                take = (disc >= 0.0) & (ts >= 0.0) & (y.abs() <= hh) & (ts < t)
                side = o + ts[:, None] * r
                side[:, 1] = 0.0
                t = torch.where(take, ts, t)
                nrm = torch.where(take[:, None], side, nrm)
        closer = (t <= 1.0) & (t < best)
        best = torch.where(closer, t, best)
        world = _rotate(quat, nrm)
        world = world / world.norm(dim=1, keepdim=True).clamp(min=1e-30)
        normal = torch.where(closer[:, None], world, normal)
    hit = best <= 1.0
    fraction = torch.where(hit, best, torch.zeros_like(best))
    point = torch.where(hit[:, None], a + fraction[:, None] * d, torch.zeros_like(a))
    return {"collider": None, "point": point.cpu().numpy(), "normal": normal.cpu().numpy(), "fraction": fraction.cpu().numpy()}

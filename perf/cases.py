"""The work that is measured: what programs have this framework do, through
its Python handle (adaptivemerging_amd.context.Context) and the C ABI under it.

Most programs step scenes.  So most cases are steps, from six bodies to twenty
thousand, at the reference's default of 30 sweeps, at the 50 of the merging and
batched configurations and at the headline's cap of 1000, with merging and
sleeping at their defaults where a program leaves them on.  Beside them stand a
collision query without a solve, and the learned warm start: a step that uses
it, its network's forward and backward passes, and its training.

A step case is one of two kinds.  An episode uploads its scene and runs it from
the start, so collections form and dissolve alike in every pass.  The others
put the bodies back where they were before each pass (push_state), as a
controller does that tries several actions from one state, except the dominoes,
whose platforms keep them moving and which simply go on.

exact() has a value for the collision query and for the network.  A solve has
none: its result after a given number of Gauss-Seidel sweeps depends on the
order of the contacts, which the framework chooses and a plain computation
cannot know.  Those cases are held to the same bits instead: all of a step is
64-bit arithmetic in an order that the framework fixes.
"""
import ctypes as C
import math

import numpy as np

from adaptivemerging_amd import _lib, workloads
from adaptivemerging_amd.context import Context, ContactArrays
from adaptivemerging_amd.scene import Scene, random_rotation

DT = 0.01


def listed():
    return [
        # the shortest calls: a stack of four boards and a cube, a demo scene or a unit test; all launches and waits
        {"name": "stack_episode", "kind": "stack", "layers": 4, "sweeps": 30, "steps": 30},
        # the jenga tower of the first configuration (100 blocks) with everything at the reference's defaults
        {"name": "jenga_episode", "kind": "jenga", "layers": 33, "sweeps": 30, "steps": 30},
        # 2,000 dominoes on ten moving platforms, merging on, before the push: the second configuration
        {"name": "dominoes", "kind": "dominoes", "platforms": 10, "rows": 2, "per_row": 100, "sweeps": 50, "steps": 4},
        # sphere trees (585 nodes each) dropped into a box: the third configuration, where detection walks trees
        {"name": "trees", "kind": "trees", "n": 96, "sweeps": 50, "steps": 2},
        # many scenes in one context, merging on, from a settled state: the batched configuration
        {"name": "batch_episode", "kind": "batch", "scenes": 48, "most": 600, "sweeps": 50, "steps": 15},
        # a small pile in a bin, four steps of a control loop at the default sweeps
        {"name": "pile_777", "kind": "pile", "n": 777, "sweeps": 30, "steps": 4, "tolerance": 1e-5},
        # an ordinary pile
        {"name": "pile_5003", "kind": "pile", "n": 5003, "sweeps": 50, "steps": 2, "tolerance": 1e-5},
        # the headline: 20,000 boxes towards residual 1e-6 under the cap of 1000 sweeps
        {"name": "pile_20000_capped", "kind": "pile", "n": 20000, "sweeps": 1000, "steps": 1, "tolerance": 1e-6},
        # a collision query on new poses: spheres in a bin, contacts read back and nothing solved
        {"name": "query_spheres", "kind": "query", "n": 4001},
        # a step that starts from the network's prediction
        {"name": "learned_step", "kind": "learned", "n": 2000, "sweeps": 50, "steps": 2},
        # the network on a caller's own rows, both directions
        {"name": "network_rows", "kind": "network", "rows": 20001},
        # one epoch of the warm start's training, at the batch that the benchmark uses
        {"name": "training_epoch", "kind": "training", "n": 300, "solves": 8, "batch": 256},
    ]


def draw(rng):
    """Another case of the listed ones' ranges, none of them dearer than the capped pile."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["stack", "jenga", "dominoes", "trees", "batch", "pile", "pile", "pile", "query", "learned",
                       "network", "training"])
    if kind == "stack":
        return {"kind": kind, "layers": rng.randint(1, 12), "sweeps": rng.randint(5, 60), "steps": rng.randint(12, 40)}
    if kind == "jenga":
        return {"kind": kind, "layers": rng.randint(5, 40), "sweeps": rng.randint(10, 60), "steps": rng.randint(12, 40)}
    if kind == "dominoes":
        return {"kind": kind, "platforms": rng.randint(1, 12), "rows": rng.randint(1, 3), "per_row": rng.randint(20, 110),
                "sweeps": rng.randint(20, 80), "steps": rng.randint(1, 6)}
    if kind == "trees":
        return {"kind": kind, "n": log_int(8, 128), "sweeps": rng.randint(20, 60), "steps": rng.randint(1, 4)}
    if kind == "batch":
        return {"kind": kind, "scenes": log_int(4, 64), "most": log_int(60, 700), "sweeps": rng.randint(20, 60),
                "steps": rng.randint(11, 18)}
    if kind == "pile":
        n = log_int(50, 18000)
        return {"kind": kind, "n": n, "sweeps": min(log_int(10, 1000), int(9e6 / n)), "steps": 1 if n > 6000 else rng.randint(1, 4),
                "tolerance": rng.choice([1e-6, 1e-5, 1e-3])}
    if kind == "query":
        return {"kind": kind, "n": log_int(100, 9000)}
    if kind == "learned":
        return {"kind": kind, "n": log_int(100, 4000), "sweeps": rng.randint(20, 100), "steps": rng.randint(1, 3)}
    if kind == "network":
        return {"kind": kind, "rows": log_int(200, 60000)}
    return {"kind": "training", "n": log_int(60, 400), "solves": rng.randint(3, 10), "batch": rng.choice([256, 512, 1024])}


# ---------------------------------------------------------------------------
# scenes

class Laid:
    """A scene laid out once, as a program keeps it that uploads it again and again."""

    def __init__(self, scene, state=None):
        b, nd, x, R, v, w = scene.arrays()
        if state is not None:
            x, R, v, w = state
        self._a = (b, nd, x, R, v, w)

    def arrays(self):
        return self._a


def _tree_scene(n, seed):
    """n sphere trees of four shapes in layers over the floor of an open box."""
    rng = np.random.default_rng(seed)
    s = Scene()
    for p, nrm in (([0, 0, 0], [0, 1, 0]), ([-1, 0, 0], [1, 0, 0]), ([1, 0, 0], [-1, 0, 0]), ([0, 0, -1], [0, 0, 1]),
                   ([0, 0, 1], [0, 0, -1])):
        s.add_plane(p, nrm, friction=0.4)
    shapes = [workloads.sphere_tree_body_shape(rng) for _ in range(4)]
    for k in range(n):
        centres, radii, children, mass, inertia = shapes[k % 4]
        x = np.array([(k % 4 - 1.5) * 0.44, 0.25 + (k // 16) * 0.4, (k // 4 % 4 - 1.5) * 0.44]) + rng.uniform(-0.02, 0.02, 3)
        s.add_tree(centres, radii, children, x, random_rotation(rng), mass=mass, inertia=inertia, friction=0.4)
    return s


def _sphere_radii(n, seed):
    return np.random.default_rng(seed).uniform(0.05, 0.12, n)


def _sphere_half(n):
    """Half the bin's width, for about a dozen layers of spheres at most."""
    return 0.11 * max(2.0, (n / 1.5) ** (1 / 3))


def _sphere_poses(n, seed):
    """Centres on a jittered lattice with neighbours overlapping by a few millimetres here and there."""
    rng = np.random.default_rng(seed + 1)
    half = _sphere_half(n)
    side = max(1, int(2 * half / 0.165))
    k = np.arange(n)
    x = np.stack([(k % side + 0.5) * 2 * half / side - half, 0.08 + (k // (side * side)) * 0.15,
                  (k // side % side + 0.5) * 2 * half / side - half], axis=1)
    return x + rng.uniform(-0.02, 0.02, (n, 3))


SPHERE_PLANES = 5


def _sphere_scene(n, seed):
    s = Scene()
    h = _sphere_half(n)
    for p, nrm in (([0, 0, 0], [0, 1, 0]), ([-h, 0, 0], [1, 0, 0]), ([h, 0, 0], [-1, 0, 0]), ([0, 0, -h], [0, 0, 1]),
                   ([0, 0, h], [0, 0, -1])):
        s.add_plane(p, nrm)
    for r, x in zip(_sphere_radii(n, seed), _sphere_poses(n, seed)):
        s.add_sphere(float(r), x, density=1000.0)
    return s


def _contact_buffers(n):
    """What a query reads of its contacts, with room for four of each sphere (overlaps this shallow give two)."""
    m = 4 * n + 16
    return {"body1": np.zeros(m, np.int32), "body2": np.zeros(m, np.int32), "point": np.zeros((m, 3)),
            "normal": np.zeros((m, 3)), "violation": np.zeros(m)}


def _counts(case):
    """Bodies of each scene of a batch, 50 to case["most"], spread over their logarithm."""
    n = case["scenes"]
    return [int(50 * (case["most"] / 50) ** ((k + 0.5) / n)) for k in range(n)]


def _settled(ctx, steps):
    for _ in range(steps):
        ctx.step(DT)
    return ctx.pull_state()


PLAIN = dict(gravity_amount=9.81, enable_merging=0, enable_unmerging=0, enable_sleeping=0)


def _pile(case, seed, **params):
    """A shelf-packed pile, fallen together (the taller, the longer that takes)."""
    ctx = Context()
    ctx.upload(workloads.box_pile(seed=seed, n=case["n"], bin_size=_bin(case["n"])))
    ctx.set_params(**{**PLAIN, "iterations": 30})
    state = _settled(ctx, 60 + case["n"] // 70)
    ctx.set_params(**params)
    return {"ctx": ctx, "state": state, "n": case.get("steps", 1)}


def _bin(n):
    return 4.0 if n >= 4000 else 2.5 if n >= 400 else 1.6


# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind, sweeps = case["kind"], case.get("sweeps", 30)
    if kind in ("stack", "jenga"):
        scene = workloads.merge_stack(seed=seed, layers=case["layers"]) if kind == "stack" else workloads.jenga_tower(
            seed=seed, layers=case["layers"], overlap=0.001)
        ctx = Context()
        ctx.set_params(gravity_amount=9.81, iterations=sweeps)
        return {"kind": "episode", "ctx": ctx, "scene": Laid(scene), "n": case["steps"]}
    if kind == "batch":
        scene = workloads.batch([workloads.batched_pile_scenes(seed=seed + k, n_scenes=1, bodies=(n + 0.5, n + 0.5))[0]
                                 for k, n in enumerate(_counts(case))])
        ctx = Context()
        ctx.upload(scene)
        ctx.set_params(**{**PLAIN, "iterations": 20})
        laid = Laid(scene, _settled(ctx, 80))
        ctx.set_params(gravity_amount=9.81, iterations=sweeps, enable_merging=1, enable_unmerging=1)
        return {"kind": "episode", "ctx": ctx, "scene": laid, "n": case["steps"]}
    if kind == "dominoes":
        ctx = Context()
        ctx.upload(workloads.domino_platforms(seed=seed, platforms=case["platforms"], rows_per_platform=case["rows"],
                                              per_row=case["per_row"]))
        ctx.set_params(gravity_amount=9.81, iterations=sweeps)
        _settled(ctx, 60)
        return {"kind": "going", "ctx": ctx, "n": case["steps"]}
    if kind == "trees":
        ctx = Context()
        ctx.upload(_tree_scene(case["n"], seed))
        ctx.set_params(**PLAIN, iterations=sweeps)
        return {"kind": "steps", "ctx": ctx, "state": _settled(ctx, 40), "n": case["steps"]}
    if kind == "pile":
        return {"kind": "steps", **_pile(case, seed, iterations=sweeps, tolerance=case["tolerance"])}
    if kind == "query":
        ctx = Context()
        ctx.upload(_sphere_scene(case["n"], seed))
        return {"kind": kind, "ctx": ctx, "state": ctx.pull_state(), "out": _contact_buffers(case["n"])}
    if kind == "learned":
        # uploaded anew each time, so that every contact of the first step is a new one, whose start is predicted
        scene = workloads.box_pile(seed=seed, n=case["n"], bin_size=_bin(case["n"]))
        s = _pile(case, seed, iterations=sweeps, learned_warm_start=1)
        s.update(kind="episode", scene=Laid(scene, s["state"]))
        # a network that expects a new contact to carry about half a body's weight
        weights = _weights(seed)
        weights[-195:] *= 0.1
        weights[-3:] = (0.5, 0.0, 0.0)
        s["ctx"].set_mlp_params(weights)
        return s
    if kind == "network":
        ctx = Context()
        ctx.set_mlp_params(_weights(seed))
        X, T = _rows(case["rows"], seed)
        return {"kind": kind, "ctx": ctx, "X": X, "T": T, "Y": np.zeros_like(T), "G": np.zeros(_lib.MLP_PARAMS, np.float32)}
    if kind == "training":
        # pairs from solves that reach a loose tolerance, so that a few steps give many
        s = _pile(case, seed, iterations=400, tolerance=0.05, collect_training=1)
        ctx = s["ctx"]
        ctx.mlp_init(seed)
        for _ in range(case["solves"]):
            ctx.step(DT)
        return {"kind": kind, "ctx": ctx, "weights": ctx.mlp_params(), "batch": case["batch"], "seed": seed}
    raise ValueError(kind)


def run(state):
    ctx, kind = state["ctx"], state["kind"]
    if kind in ("episode", "going", "steps"):
        if kind == "episode":
            ctx.upload(state["scene"])
        elif kind == "steps":
            ctx.push_state(*state["state"])
        for _ in range(state["n"]):
            st = ctx.step(DT)
        x, R, v, w = ctx.pull_state()
        return {"x": x, "R": R, "v": v, "w": w, "dv": ctx.pull_deltav(ctx.n), "residual": st["last_change"],
                "counts": np.array([st["n_contacts"], st["n_groups"], st["n_colours"], st["iterations_used"],
                                    st["n_collections"], st["n_internal_contacts"]])}
    if kind == "query":
        ctx.push_state(*state["state"])
        n = ctx.detect(DT)
        out = state["out"]
        want = ContactArrays()
        want.body1, want.body2 = _lib.iptr(out["body1"]), _lib.iptr(out["body2"])
        want.point_b1, want.normal_b1, want.violation = (_lib.dptr(out[k]) for k in ("point", "normal", "violation"))
        got = C.c_int32()
        _call(ctx, "am_contacts_pull", C.byref(want), len(out["body1"]), C.byref(got))
        return {**out, "contacts": n}
    if kind == "network":
        n, loss = len(state["X"]), C.c_float()
        _call(ctx, "am_mlp_forward", _lib.ptr(state["X"]), n, _lib.ptr(state["Y"]))
        _call(ctx, "am_mlp_gradients", _lib.ptr(state["X"]), _lib.ptr(state["T"]), n, _lib.ptr(state["G"]), C.byref(loss))
        return {"y": state["Y"], "gradients": state["G"], "loss": loss.value}
    ctx.set_mlp_params(state["weights"])
    loss = ctx.train_epochs(1, batch=state["batch"], lr=1e-3, seed=state["seed"])
    return {"weights": ctx.mlp_params(), "loss": loss}


def _call(ctx, name, *args):
    rc = getattr(ctx.lib, name)(ctx.h, *args)
    if rc != 0:
        raise _lib.AMError(rc, ctx.lib.am_last_error(ctx.h).decode())


# ---------------------------------------------------------------------------
# the network's rows: features are of order one (directions, ratios, logs), targets bounded by 2
LAYERS = [(24, 64), (64, 64), (64, 64), (64, 3)]


def _weights(seed):
    """He-scaled weights, flat as am_mlp_set_params takes them."""
    rng = np.random.default_rng(seed)
    parts = []
    for fan_in, fan_out in LAYERS:
        parts += [rng.normal(size=fan_in * fan_out) * math.sqrt(2.0 / fan_in), rng.normal(size=fan_out) * 0.1]
    return np.concatenate(parts).astype(np.float32)


def _rows(n, seed):
    rng = np.random.default_rng(seed + 1)
    return (rng.normal(size=(n, 24)).astype(np.float32),
            np.clip(rng.normal(size=(n, 3)), -2.0, 2.0).astype(np.float32))


# ---------------------------------------------------------------------------
# contacts per body of each kind, as measured
CONTACTS = {"stack": 2.4, "jenga": 11.5, "dominoes": 4.0, "trees": 6.3, "batch": 2.6, "pile": 7.0, "learned": 7.4,
            "query": 1.8, "training": 6.7}
TALL_PILE = 14.7  # from 10,000 bodies on


def work(case):
    """Bytes: each step reads and writes every body's state (18 doubles) and
    writes its contacts once (points, frames, Jacobians, multipliers: 650
    bytes).  Operations: 45 per row of a contact and sweep, three rows.  Rows
    of the network: each direction reads its inputs and writes its results."""
    kind = case["kind"]
    if kind == "network":
        macs = sum(a * b for a, b in LAYERS)
        # forward alone, then forward, its backward and the weights' gradients
        return {"bytes": case["rows"] * (24 + 3) * 4 * 2 + 3 * 4 * _lib.MLP_PARAMS, "flops": case["rows"] * macs * 2 * 4}
    bodies = _bodies(case)
    contacts = (TALL_PILE if kind == "pile" and bodies >= 10000 else CONTACTS[kind]) * bodies
    if kind == "training":
        rows, macs = contacts * case["solves"], sum(a * b for a, b in LAYERS)
        return {"bytes": rows * 27 * 4 + 2 * 4 * _lib.MLP_PARAMS, "flops": rows * macs * 2 * 3}
    if kind == "query":
        return {"bytes": bodies * 2 * 144 + contacts * 64, "flops": contacts * 200}
    steps = case["steps"]
    return {"bytes": steps * (bodies * 2 * 144 + contacts * 650), "flops": steps * contacts * case["sweeps"] * 135}


def _bodies(case):
    kind = case["kind"]
    if kind == "stack":
        return case["layers"] + 1
    if kind == "jenga":
        return 3 * case["layers"] + 1
    if kind == "dominoes":
        return case["platforms"] * case["rows"] * case["per_row"]
    if kind == "batch":
        return sum(_counts(case))
    return case["n"]


def tolerance(case):
    if case["kind"] in ("network", "training", "learned"):
        return TOLERANCES[case["kind"]]
    return "exact"


# About four times what weights moved by 1e-7 to 1e-6 of themselves change: a
# sum in another order flips the BF16 rounding of a few hidden units.  One
# epoch of training carries such a flip through all the steps that follow.
TOLERANCES = {
    "network": {"rel": 2.5e-3, "max": 0.04},
    "training": {"rel": 1e-2, "max": 0.25},
    "learned": {"rel": 1e-5, "max": 5e-4},
}


def exact(case, seed):
    if case["kind"] == "network":
        return _exact_network(case["rows"], seed)
    if case["kind"] == "query":
        return _exact_query(case["n"], seed)
    return None


def _exact_network(rows, seed):
    p, q = _weights(seed).astype(np.float64), 0
    layers = []
    for a, b in LAYERS:
        layers.append((p[q:q + a * b].reshape(a, b), p[q + a * b:q + a * b + b]))
        q += a * b + b
    X, T = (t.astype(np.float64) for t in _rows(rows, seed))
    acts = [X]
    for k, (W, b) in enumerate(layers):
        z = acts[-1] @ W + b
        acts.append(np.maximum(z, 0.0) if k < 3 else z)
    y = acts.pop()
    d = 2.0 * (y - T) / rows
    grads = []
    for k in range(3, -1, -1):
        W, _ = layers[k]
        grads[:0] = [(acts[k].T @ d).reshape(-1), d.sum(0)]
        if k:
            d = np.where(acts[k] > 0, d @ W.T, 0.0)
    return {"y": y, "gradients": np.concatenate(grads), "loss": float(((y - T) ** 2).sum() / rows)}


def _exact_query(n, seed):
    """Sphere-plane contacts plane by plane, then sphere pairs i < j; the
    spheres are not rotated, so body-1 coordinates are world ones less its centre."""
    r, x = _sphere_radii(n, seed), _sphere_poses(n, seed)
    h = _sphere_half(n)
    b1, b2, pts, nrm, vio = [], [], [], [], []
    planes = [((0, 0, 0), (0, 1, 0)), ((-h, 0, 0), (1, 0, 0)), ((h, 0, 0), (-1, 0, 0)), ((0, 0, -h), (0, 0, 1)),
              ((0, 0, h), (0, 0, -1))]
    for k, (p, u) in enumerate(planes):
        p, u = np.array(p, float), np.array(u, float)
        along = (x - p) @ u
        hit = np.nonzero(along - r < 0)[0]
        b1.append(hit + SPHERE_PLANES)
        b2.append(np.full(len(hit), k))
        pts.append(-along[hit, None] * u)
        nrm.append(np.broadcast_to(-u, (len(hit), 3)))
        vio.append(along[hit] - r[hit])
    for i0 in range(0, n, 256):
        i1 = min(i0 + 256, n)
        d2 = ((x[i0:i1, None, :] - x[None, i0:, :]) ** 2).sum(2)
        reach = r[i0:i1, None] + r[None, i0:]
        i, j = np.nonzero(np.triu(d2 < reach * reach, 1))
        i, j = i + i0, j + i0
        d = x[j] - x[i]
        dist = np.sqrt((d * d).sum(1))
        alpha = (r[i] - r[j] + dist) / (2 * dist)
        b1.append(i + SPHERE_PLANES)
        b2.append(j + SPHERE_PLANES)
        pts.append(alpha[:, None] * d)
        nrm.append(d / dist[:, None])
        vio.append(dist - r[i] - r[j])
    out, m = _contact_buffers(n), sum(len(v) for v in vio)
    for key, parts in (("body1", b1), ("body2", b2), ("point", pts), ("normal", nrm), ("violation", vio)):
        out[key][:m] = np.concatenate(parts)
    return {**out, "contacts": m}

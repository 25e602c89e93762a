"""libam (HIP, gfx950) against the CPU oracle on identical inputs.

Bar: integer, index and floating-point contact fields bit-exact; lambdas and
deltaV bit-exact against the oracle's sequential sweep in the GPU's sweep
order; integration bit-exact (both sides take the Rodrigues update's sine and
cosine from fdlibm's algorithm, not from their math libraries).
"""
import numpy as np
import pytest

from adaptivemerging_amd import workloads
from tests.helpers import assert_bits_equal, assert_contacts_equal, oracle_step_like_gpu, twin

pytestmark = pytest.mark.gpu


def test_detect_jenga(gpu_lib):
    scene = workloads.jenga_tower(seed=1, layers=12, overlap=0.002)
    ctx, orc = twin(scene)
    n_g = ctx.detect(0.01)
    n_o = orc.detect()
    print("contacts", n_g, n_o, flush=True)
    assert n_g == n_o and n_g > 0
    assert_contacts_equal(ctx.contacts(), orc.contacts())


def test_detect_cluster_boxes_spheres(gpu_lib):
    scene = workloads.box_cluster(seed=3, n=125, spheres=20)
    ctx, orc = twin(scene)
    n_g = ctx.detect(0.01)
    n_o = orc.detect()
    print("contacts", n_g, n_o, flush=True)
    assert n_g == n_o and n_g > 50
    assert_contacts_equal(ctx.contacts(), orc.contacts())


def test_detect_sphere_trees(gpu_lib):
    scene = workloads.sphere_tree_drop(seed=5, n=16, heights=(0.15, 0.9), box=(1.2, 1.0, 1.2))
    ctx, orc = twin(scene)
    n_g = ctx.detect(0.01)
    n_o = orc.detect()
    print("contacts", n_g, n_o, flush=True)
    assert n_g == n_o and n_g > 0
    assert_contacts_equal(ctx.contacts(), orc.contacts())


@pytest.mark.parametrize("n", [1, 2, 13, 14, 65, 130])
def test_detect_pairs_beyond_the_room_for_them(gpu_lib, n):
    """n spheres all in one cell: every pair of them is one, more than the twelve a
    thread keeps and than the four a body there is room for at first; twice, the
    second time with the room made by the first."""
    from adaptivemerging_amd.scene import Scene

    rng = np.random.default_rng(n)
    s = Scene()
    s.add_plane([0, 0, 0], [0, 1, 0])
    for _ in range(n):
        s.add_sphere(0.5, rng.uniform(0.0, 0.3, 3) + [0, 0.3, 0])
    ctx, orc = twin(s)
    n_o = orc.detect()
    for _ in range(2):
        n_g = ctx.detect(0.01)
        print("contacts", n_g, n_o, flush=True)
        assert n_g == n_o and n_g >= n * (n - 1) // 2
        assert_contacts_equal(ctx.contacts(), orc.contacts())
    ctx.close()


def _tree(rng, fanouts, radius=0.05, size=0.4):
    """A sphere tree with fanouts[k] children for every node of level k."""
    centres, radii, children = [], [], []

    def build(level):
        node = len(centres)
        centres.append(rng.uniform(-size / 2, size / 2, 3).tolist())
        radii.append(radius)
        children.append([])
        if level < len(fanouts):
            children[node] = [build(level + 1) for _ in range(fanouts[level])]
            radii[node] = 0.9  # encloses everything below it
        return node

    build(0)
    return centres, radii, children


@pytest.mark.parametrize("fanouts", [[], [6], [7], [8], [1] * 60, [64], [65], [127], [128], [8, 8], [16, 3, 5], [2] * 8])
def test_detect_trees_walked_by_waves(gpu_lib, fanouts):
    """Overlapping trees of every shape a wave's stack meets, each against the
    others, boxes, spheres and a plane: no more nodes than a thread takes (8),
    long chains, 64 and 65 children, as many as a thread's stack holds.  Same
    contacts, in the same order, as the oracle's recursion."""
    from adaptivemerging_amd.scene import Scene

    rng = np.random.default_rng(len(fanouts) + sum(fanouts))
    s = Scene()
    s.add_plane([0, 0, 0], [0, 1, 0])
    for i in range(4 if max(fanouts, default=0) <= 64 else 1):  # two trees of 65 children are refused (below)
        c, r, ch = _tree(rng, fanouts)
        s.add_tree(c, r, ch, rng.uniform(-0.1, 0.1, 3) + [0, 0.1, 0])
    s.add_box([0.3, 0.2, 0.3], [0.1, 0.1, 0.0])
    s.add_sphere(0.15, [0.0, 0.2, 0.1])
    s.add_tree([[0, 0, 0], [0.1, 0, 0]], [0.3, 0.1], [[1], []], [0.0, 0.1, 0.0])
    ctx, orc = twin(s)
    n_g = ctx.detect(0.01)
    n_o = orc.detect()
    print("contacts", n_g, n_o, flush=True)
    assert n_g == n_o and n_g > 0
    assert_contacts_equal(ctx.contacts(), orc.contacts())
    ctx.close()


@pytest.mark.parametrize("fanouts,trees", [([2, 128], 1), ([65], 2)])
def test_detect_refuses_trees_too_wide_for_a_walk(gpu_lib, fanouts, trees):
    """A thread's stack holds 128 entries: one sibling and 128
    children, or 64 siblings and the 65 children of the other tree, do not fit."""
    from adaptivemerging_amd import _lib
    from adaptivemerging_amd.context import Context
    from adaptivemerging_amd.scene import Scene

    s = Scene()
    s.add_plane([0, 0, 0], [0, 1, 0])
    for _ in range(trees):
        c, r, ch = _tree(np.random.default_rng(1), fanouts)
        s.add_tree(c, r, ch, [0.0, 0.1, 0.0])
    ctx = Context()
    ctx.upload(s)
    with pytest.raises(_lib.AMError) as e:
        ctx.detect(0.01)
    assert e.value.code == _lib.AM_ERR_CAPACITY
    ctx.close()


@pytest.mark.parametrize("schedule", [0, 1])
@pytest.mark.parametrize("iterations", [1, 7, 100])
def test_pgs_jenga_bit_exact(gpu_lib, iterations, schedule):
    scene = workloads.jenga_tower(seed=2, layers=10, overlap=0.002)
    ctx, orc = twin(scene, iterations=iterations, tolerance=1e-9, friction_override=1, friction=0.6,
                    pgs_schedule=schedule)
    ctx.apply_gravity(); orc.apply_gravity()
    ctx.detect(0.01); orc.detect()
    it_g, last_g = ctx.solve(0.01)
    order = ctx.solve_order()
    assert sorted(order.tolist()) == list(range(len(order)))
    it_o, last_o, ch_o = orc.solve(order, 0.01)
    print("iterations", it_g, it_o, last_g, last_o, flush=True)
    assert it_g == it_o
    assert_bits_equal("last_change", np.array([last_g]), np.array([last_o]))
    g, o = ctx.contacts(), orc.contacts()
    assert_contacts_equal(g, o)
    assert_bits_equal("deltaV", ctx.pull_deltav(), orc.pull_deltav())
    np.testing.assert_allclose(ctx.changes(), ch_o, rtol=1e-14, atol=0)


def test_pgs_cluster_warm_started(gpu_lib):
    scene = workloads.box_cluster(seed=4, n=200, spheres=30)
    ctx, orc = twin(scene, iterations=40)
    ctx.apply_gravity(); orc.apply_gravity()
    n = ctx.detect(0.01); orc.detect()
    lam = np.random.default_rng(0).uniform(0, 1, size=(n, 3))
    ctx.push_lambdas(lam); orc.push_lambdas(lam)
    ctx.solve(0.01)
    order = ctx.solve_order()
    orc.solve(order, 0.01)
    assert_contacts_equal(ctx.contacts(), orc.contacts())
    assert_bits_equal("deltaV", ctx.pull_deltav(), orc.pull_deltav())


def test_colouring_valid(gpu_lib):
    scene = workloads.box_cluster(seed=6, n=343, spheres=40)
    ctx, _ = twin(scene)
    ctx.detect(0.01)
    col, ncol = ctx.colours()
    c = ctx.contacts()
    b, _, _, _, _, _ = scene.arrays()
    pinned = (b["flags"] & 1) != 0
    order = ctx.solve_order()
    # order is colour-major and contacts of one body pair stay in list order
    assert np.all(np.diff(col[order]) >= 0)
    seen = {}
    for k in order:
        for body in (c["body1"][k], c["body2"][k]):
            if pinned[body] or col[k] == 64:
                continue
            key = (col[k], body)
            pair = (min(c["body1"][k], c["body2"][k]), max(c["body1"][k], c["body2"][k]))
            assert seen.setdefault(key, pair) == pair, "two body pairs of one colour share a dynamic body"
    print("colours", ncol, flush=True)


def _priority(g):
    h = (g * 0x9E3779B1) & 0xFFFFFFFF
    h ^= h >> 16
    h = (h * 0x85EBCA6B) & 0xFFFFFFFF
    h ^= h >> 13
    return h


@pytest.mark.parametrize("pairs,on_platform", [(1, 0), (64, 1), (1025, 63), (500, 200), (4025, 70),
                                                 (4026, 70), (4096, 0), (4097, 0), (20000, 300)])
def test_sweep_order_is_the_greedy_colouring(gpu_lib, pairs, on_platform):
    """The exported order against a plain greedy colouring: groups in order of
    priority take the smallest colour free at their dynamic bodies (64: the
    sequential tail), then order by colour, larger groups first, index.
    `pairs` body pairs of spheres (a chain on a plane, then some alone) and a
    platform under on_platform boxes (more than 64 of them fill the tail),
    below, at and above the 4,096 groups that one workgroup lays out."""
    from adaptivemerging_amd.context import Context
    from adaptivemerging_amd.scene import Scene

    s = Scene()
    s.add_plane([0, 0, 0], [0, 1, 0])
    chain = max(1, pairs // 3)
    for i in range(chain):  # each touches the plane and the one before it
        s.add_sphere(0.101, [0.2 * i, 0.1, -30.0])
    for i in range(pairs - (2 * chain - 1)):
        s.add_sphere(0.101, [0.5 * (i % 200), 0.1, -40.0 - 0.5 * (i // 200)])
    if on_platform:
        s.add_box([40.0, 0.5, 40.0], [100.0, 0.249, 0.0])
        for i in range(on_platform):
            s.add_box([0.2, 0.2, 0.2], [100.0 - 10 + (i % 30) * 0.5, 0.598, (i // 30) * 0.5])
    ctx = Context()
    ctx.upload(s)
    ctx.set_params()
    ctx.detect(0.01)
    c = ctx.contacts()
    b, _, _, _, _, _ = s.arrays()
    pinned = (b["flags"] & 1) != 0
    key = np.sort(np.stack([c["body1"], c["body2"]], axis=1), axis=1)
    start = np.concatenate([[0], 1 + np.flatnonzero(np.any(np.diff(key, axis=0) != 0, axis=1)), [len(key)]])
    n = len(start) - 1
    assert n == pairs + (on_platform + 1 if on_platform else 0)
    used, colour = {}, np.zeros(n, int)
    for g in sorted(range(n), key=lambda g: (_priority(g), g), reverse=True):
        mine = [used.setdefault(int(e), set()) for e in key[start[g]] if not pinned[e]]
        col = next(k for k in range(65) if k == 64 or not any(k in u for u in mine))
        colour[g] = col
        for u in mine:
            u.add(col)
    size = np.minimum(np.diff(start), 15)
    order = sorted(range(n), key=lambda g: (colour[g], 15 - size[g] if colour[g] < 64 else 0, g))
    expect = np.concatenate([np.arange(start[g], start[g + 1]) for g in order])
    print("groups", n, "colours", colour.max() + 1, flush=True)
    assert np.array_equal(ctx.solve_order(), expect)
    got, ncol = ctx.colours()
    assert np.array_equal(got, np.repeat(colour, np.diff(start)))
    assert ncol == len(set(colour))
    ctx.close()


def test_steps_jenga(gpu_lib):
    scene = workloads.jenga_tower(seed=7, layers=8, overlap=0.001)
    ctx, orc = twin(scene, iterations=50, gravity_amount=9.81, friction_override=1, friction=0.6)
    dt = 0.01
    for step in range(5):
        it_g, it_o = oracle_step_like_gpu(ctx, orc, dt)
        assert it_g == it_o
        for name, a, b in zip("xRvw", ctx.pull_state(), orc.pull_state()):
            assert_bits_equal(f"step {step} {name}", a, b)


def test_rotation_update_over_angles(gpu_lib):
    """advancePositions' Rodrigues update for rotation angles |w| dt from
    1e-9 to 60 rad, and next to multiples of pi/2, bit for bit."""
    scene = workloads.box_cluster(seed=9, n=512, spheres=64)
    ctx, orc = twin(scene)
    rng = np.random.default_rng(3)
    n = scene.n
    dt = 0.01
    ang = np.exp(rng.uniform(np.log(1e-9), np.log(60.0), n))
    ang[:96] = [k * np.pi / 2 * (1 + e) for k in range(1, 33) for e in (0.0, 1e-16, -3e-12)]
    axis = rng.normal(size=(n, 3))
    axis /= np.linalg.norm(axis, axis=1, keepdims=True)
    w = axis * (ang / dt)[:, None]
    v = rng.normal(size=(n, 3))
    ctx.push_state(v=v, w=w); orc.set_state(v=v, w=w)
    for rep in range(3):
        ctx.advance_positions(dt); orc.advance_positions(dt)
        for name, a, b in zip("xR", ctx.pull_state()[:2], orc.pull_state()[:2]):
            assert_bits_equal(f"update {rep} {name}", a, b)


def test_motion_metric(gpu_lib):
    scene = workloads.box_cluster(seed=8, n=27, spheres=5)
    ctx, orc = twin(scene)
    rng = np.random.default_rng(1)
    v = rng.normal(size=(scene.n, 3)); w = rng.normal(size=(scene.n, 3))
    ctx.push_state(v=v, w=w); orc.set_state(v=v, w=w)
    pairs = np.array([[1, 2], [3, 4], [5, -1], [10, 20], [0, 7]], dtype=np.int32)
    g = ctx.motion_metric(pairs)
    o = np.array([orc.motion_metric(int(a), int(b)) for a, b in pairs])
    assert_bits_equal("metric", g, o)


@pytest.mark.parametrize("grid,block", [(2, 64), (8, 64), (32, 128), (64, 64), (128, 256)])
def test_pgs_multiblock_bit_exact(gpu_lib, grid, block):
    """The cooperative (grid-barrier) path of the coloured sweep kernel."""
    scene = workloads.box_cluster(seed=9, n=729, spheres=60)
    ctx, orc = twin(scene, iterations=25, pgs_grid=grid, pgs_block=block, pgs_schedule=1)
    ctx.apply_gravity(); orc.apply_gravity()
    n = ctx.detect(0.01); orc.detect()
    lam = np.random.default_rng(2).uniform(0, 0.5, size=(n, 3))
    ctx.push_lambdas(lam); orc.push_lambdas(lam)
    it_g, _ = ctx.solve(0.01)
    order = ctx.solve_order()
    it_o, _, _ = orc.solve(order, 0.01)
    print("contacts", n, "iterations", it_g, it_o, flush=True)
    assert it_g == it_o
    assert_contacts_equal(ctx.contacts(), orc.contacts())
    assert_bits_equal("deltaV", ctx.pull_deltav(), orc.pull_deltav())


@pytest.mark.parametrize("n", [1, 63, 64, 65, 300])
def test_warm_start_takes_each_old_contact_once(gpu_lib, n):
    """n contacts of one pair of boxes; a third of them carry one of 9 infos, so
    several look for the same old contact: the first in the list takes its lambda,
    the later ones get zero, as in the oracle's list order.  Some moved (bad ones
    search the other infos), some are too far, and a pair with a sphere shares its
    old contact among all."""
    from adaptivemerging_amd.scene import Scene

    rng = np.random.default_rng(n)
    s = Scene()
    s.add_box([1, 1, 1], [0, 0, 0])
    s.add_box([1, 1, 1], [0, 0.99, 0])
    s.add_sphere(0.5, [0.9, 0, 0])
    ctx, orc = twin(s)
    for step in range(2):
        m = n + 7 * step
        b1 = np.zeros(2 * m, np.int32)
        b2 = np.repeat([1, 2], m).astype(np.int32)
        info = np.where(rng.random(2 * m) < 0.35, rng.integers(0, 9, 2 * m), np.arange(2 * m) % 40).astype(np.int32)
        p = np.tile([0.1, 0.5, 0.1], (2 * m, 1)) + rng.uniform(-0.04, 0.04, (2 * m, 3))
        nrm = np.tile([0.0, 1.0, 0.0], (2 * m, 1))
        for o in (ctx, orc):
            if step:
                o.update_contacts_map()
            o.push_contacts(b1, b2, p, nrm, np.full(2 * m, -1e-3), info=info)
        if step == 0:
            lam = rng.uniform(0.1, 1.0, (2 * m, 3))
            ctx.push_lambdas(lam); orc.push_lambdas(lam)
    for _ in range(2):  # again: what was taken stays zero
        got, want = ctx.warm_start(), orc.warm_start()
        print("bad, repaired", got, flush=True)
        assert tuple(got) == tuple(want)
        assert_contacts_equal(ctx.contacts(), orc.contacts(), keys=["lambda", "lambda_warm", "new_this_step",
                                                                    "prev_violation"])
    ctx.close()

"""Adaptive merging on the GPU (single sweep inside collections, body-pair
histories, merge and unmerge, collection physics) against the CPU
restatement in oracle/merging.py, phase by phase and bit for bit."""
import numpy as np
import pytest

from adaptivemerging_amd import workloads
from adaptivemerging_amd.context import Context
from oracle.merging import MergingOracle
from tests.helpers import assert_bits_equal, assert_contacts_equal

pytestmark = pytest.mark.gpu

PARAMS = dict(gravity_amount=9.81, iterations=100, tolerance=1e-10)


def make(scene, **extra):
    ctx = Context()
    ctx.upload(scene)
    ctx.set_params(**{**PARAMS, **extra})
    mo = MergingOracle(scene, type(ctx.params)())
    for k, _ in type(ctx.params)._fields_:
        setattr(mo.params, k, getattr(ctx.params, k))
    mo.set_params()
    return ctx, mo


def kick(obj, body, fy):
    f, t = obj.pull_forces()
    f[body][1] += fy
    obj.push_forces(f, t)


# distinct breadth-first layers seen by check_organized (a run can assert it saw some)
ORGANIZED_SEEN = set()


def check_organized(ctx, mo):
    """The single sweep's exported order visits the body pairs of every
    dynamic body in non-decreasing breadth-first layer, the layers of
    getOrganizedContacts as the merging oracle restates them."""
    ls = getattr(mo, "last_sweep", None)
    if not mo.members or ls is None or ls["layers"] is None:
        return
    order = ctx.solve_order()
    b1, b2, layers = ls["body1"], ls["body2"], ls["layers"]
    assert len(order) == len(layers)
    last = {}
    for k in order:
        for b in {int(b1[k]), int(b2[k])}:
            if mo.pinned(b):
                continue
            assert layers[k] >= last.get(b, -1), f"body {b}: layer {layers[k]} after {last[b]}"
            last[b] = layers[k]
        ORGANIZED_SEEN.add(layers[k])


def step_both(ctx, mo, dt, step, kick_body=None):
    mo.total_steps += 1
    ctx.clear_bodies(); mo.clear_bodies()
    ctx.apply_gravity(); mo.o.apply_gravity()
    ctx.apply_spring_forces(); mo.o.apply_springs()
    if kick_body is not None:
        kick(ctx, kick_body, 2000.0)
        kick(mo.o, kick_body, 2000.0)
    ctx.update_contacts_map(); mo.o.update_contacts_map()
    ctx.detect(dt); mo.o.detect()
    ctx.warm_start(); mo.o.warm_start()
    ctx.update_in_collections(dt)
    mo.update_in_collections(dt, ctx.solve_order)
    check_organized(ctx, mo)
    assert_contacts_equal(ctx.internal_contacts(), mo.internal_contacts())
    ctx.accumulate_for_unmerging(dt); mo.accumulate_for_unmerging(dt)
    cut_g = ctx.unmerge(dt)
    cut_o = mo.unmerge(dt)
    assert cut_g == cut_o, f"step {step}: unmerge {cut_g} vs {cut_o}"
    if mo.merging_event:
        ctx.clear_top_level(); mo.clear_top_level()
    ctx.redo_warm_start(); mo.o.redo_warm_start()
    it_g, _ = ctx.solve(dt)
    it_o, _, _ = mo.o.solve(ctx.solve_order(), dt)
    assert it_g == it_o
    ctx.clear_body_pair_contacts(); mo.clear_body_pair_contacts()
    ctx.advance_velocities(dt); mo.advance_velocities(dt)
    ctx.accumulate_for_merging(dt); mo.accumulate_for_merging(dt)
    ctx.advance_positions(dt); mo.advance_positions(dt)
    ext, _ = ctx.body_pairs()
    assert [(p["body1"], p["body2"], p["flag"], p["hist_n"]) for p in ext] == \
        [(r["b1"], r["b2"], int(r["flag"]), len(r["hist"])) for r in mo.bpc]
    for p, r in zip(ext, mo.bpc):
        assert_bits_equal(f"step {step} metric history", np.array(p["hist"]), np.array(r["hist"]))
    merged = 0
    if step % 10 == 0:
        merged = ctx.merge()
        assert merged == mo.merge()
    return merged, cut_g


def compare_world(ctx, mo, step):
    parent, top = ctx.structure()
    assert list(top) == mo.top, f"step {step}: top list"
    assert list(parent[:mo.n_phys]) == mo.parent[:mo.n_phys], f"step {step}: parents"
    n = len(parent)
    assert n == mo.n_entities
    g = ctx.pull_state(n)
    o = mo.o.pull_state(n)
    for name, a, b in zip("xRvw", g, o):
        assert_bits_equal(f"step {step} {name}", a, b)
    assert_bits_equal(f"step {step} jinv", ctx.pull_jinv(n), mo.o.pull_jinv())
    ge = ctx.entities()
    for e in top:
        if ge[e]["geom"] == 3:
            oe = mo.desc(int(e))
            for key in ("mass", "minv", "jinv0", "inertia0", "bbox", "flags"):
                assert_bits_equal(f"step {step} collection {e} {key}", ge[e][key], oe[key])
    assert_contacts_equal(ctx.contacts(), mo.o.contacts())
    assert_contacts_equal(ctx.internal_contacts(), mo.internal_contacts())


@pytest.mark.parametrize("position_level", [0, 1])
def test_merge_and_unmerge_match_oracle(gpu_lib, position_level):
    """Boards settle and merge (with the ground plane: a pinned collection),
    an upward force on a member breaks its contacts inside the collection and
    it unmerges, then it merges again; with the velocity-level metric and
    with the position-level one (Merging.metricPositionLevel)."""
    scene = workloads.merge_stack(seed=3)
    ctx, mo = make(scene, metric_position_level=position_level)
    dt = 0.01
    merges = cuts = 0
    for step in range(1, 41):
        m, c = step_both(ctx, mo, dt, step, kick_body=4 if step == 31 else None)
        merges += m
        cuts += c
        compare_world(ctx, mo, step)
        print("step", step, "top", list(ctx.structure()[1]), "merged", m, "cut", c, flush=True)
    assert merges >= 2 and cuts >= 1
    assert len(ORGANIZED_SEEN) >= 2, ORGANIZED_SEEN


@pytest.mark.parametrize("position_level", [0, 1])
def test_step_equals_phases(gpu_lib, position_level):
    """am_step with merging (and sleeping) on runs exactly the phases above."""
    scene = workloads.merge_stack(seed=4)
    a = Context(); a.upload(scene); a.set_params(**PARAMS, metric_position_level=position_level)
    b = Context(); b.upload(scene); b.set_params(**PARAMS, metric_position_level=position_level)
    dt = 0.01
    for step in range(1, 26):
        st = a.step(dt)
        b.clear_bodies(); b.apply_gravity(); b.apply_spring_forces()
        b.update_contacts_map(); b.detect(dt); b.warm_start(); b.wake()
        b.update_in_collections(dt); b.accumulate_for_unmerging(dt); b.unmerge(dt)
        if b.merging_event:
            b.clear_top_level()
        b.redo_warm_start(); b.solve(dt); b.clear_body_pair_contacts(); b.advance_velocities(dt)
        b.accumulate_for_merging(dt); b.advance_positions(dt)
        if step % 10 == 0:
            b.merge()
        b.sleep()
        pa, ta = a.structure()
        pb, tb = b.structure()
        assert list(ta) == list(tb) and list(pa) == list(pb)
        n = len(pa)
        for name, x, y in zip("xRvw", a.pull_state(n), b.pull_state(n)):
            assert_bits_equal(f"step {step} {name}", x, y)
    assert st["n_collections"] >= 1


def test_unmerge_all_matches_oracle(gpu_lib):
    """The "unmerge all" request (Merging.unmergeAll) between two steps, then
    the run goes on; the GPU matches the oracle before and after."""
    scene = workloads.merge_stack(seed=3)
    ctx, mo = make(scene)
    ctx.set_params(enable_sleeping=0)
    mo.set_params(enable_sleeping=0)
    dt = 0.01
    for step in range(1, 13):
        step_both(ctx, mo, dt, step)
    n_g = ctx.unmerge_all()
    n_o = mo.unmerge_all()
    assert n_g == n_o >= 1
    compare_world(ctx, mo, 12)
    for step in range(13, 31):
        step_both(ctx, mo, dt, step)
        compare_world(ctx, mo, step)


def test_layout_of_contacts_inside_one_collection(gpu_lib):
    """Contacts given between two members of one collection have the same solve
    body on both sides: the group counts once among that body's groups, so the
    layout ends, with every contact in the order once."""
    ctx = Context()
    ctx.upload(workloads.merge_stack(seed=4))
    ctx.set_params(**PARAMS)
    for _ in range(25):
        st = ctx.step(0.01)
    assert st["n_collections"] >= 1
    parent, _ = ctx.structure()
    coll = max(parent)
    a, b = [i for i, p in enumerate(parent) if p == coll][:2]
    free = next(i for i, p in enumerate(parent) if p != coll and i not in (a, b, coll))
    b1, b2 = [a, a, a, b], [b, b, free, free]
    p = np.zeros((4, 3))
    ctx.push_contacts(b1, b2, p, np.tile([0.0, 1.0, 0.0], (4, 1)), np.full(4, -1e-3), info=[0, 1, 0, 0])
    print("collection", coll, "members", a, b, "other", free, flush=True)
    assert sorted(ctx.solve_order().tolist()) == [0, 1, 2, 3]
    ctx.close()


@pytest.mark.parametrize("iterations", [0, 1, 2, 7])
def test_solve_of_contacts_inside_one_collection(gpu_lib, iterations):
    """A group with the same solve body on both sides: both halves of its updates
    act on that body's one deltaV, under every schedule and launch shape, as in the
    oracle's sequential sweep (bit for bit).  Such groups alone, before and behind
    groups with another body, listed either way round, with lambdas to start from."""
    ctx, mo = make(workloads.merge_stack(seed=4), enable_merge_pinned=0)
    dt = 0.01
    for step in range(1, 26):
        step_both(ctx, mo, dt, step)
    mo.set_params(iterations=iterations, tolerance=0.0)
    parent, _ = ctx.structure()
    coll = max(parent)
    inside = [i for i, p in enumerate(parent) if p == coll]
    assert coll >= 0 and len(inside) >= 2 and not mo.pinned(coll)
    a, b = inside[:2]
    free = next(i for i, p in enumerate(parent[:mo.n_phys]) if p != coll and not mo.pinned(i))
    x = ctx.pull_state(mo.n_phys)[0]
    rng = np.random.default_rng(iterations)
    f = rng.normal(size=(mo.n_entities, 3))
    for pairs in ([(a, b)] * 3, [(a, b), (b, a), (a, free), (b, free), (b, free)], [(a, free), (a, b), (b, a)]):
        n = len(pairs)
        b1, b2 = np.array(pairs, np.int32).T.copy()
        p = (x[b1] + x[b2]) / 2 + rng.uniform(-0.1, 0.1, (n, 3))
        nrm = rng.normal(size=(n, 3))
        nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
        lam = np.abs(rng.normal(size=(n, 3)))
        for shape in (dict(), dict(pgs_grid=64), dict(pgs_schedule=1), dict(pgs_plain_launch=1)):
            ctx.set_params(**{**dict(iterations=iterations, tolerance=0.0, pgs_schedule=0, pgs_grid=0,
                                     pgs_plain_launch=0), **shape})
            for o in (ctx, mo.o):
                o.clear_bodies()
                o.push_forces(f, f[::-1].copy())
                o.push_contacts(b1, b2, p, nrm, np.full(n, -1e-3), info=np.arange(n))
                o.push_lambdas(lam)
            it_g, _ = ctx.solve(dt)
            it_o, _, _ = mo.o.solve(ctx.solve_order(), dt)
            print(pairs, shape, "shape", ctx.launch_shape(), "sweeps", it_g, flush=True)
            assert it_g == it_o == iterations
            assert_contacts_equal(ctx.contacts(), mo.o.contacts())
            dv = ctx.pull_deltav(mo.n_entities)
            assert_bits_equal("deltaV", dv, mo.o.pull_deltav())
            # the halves of a group inside the collection cancel, the other groups' do not
            assert np.any(dv[coll] != 0) == any(free in q for q in pairs)
        ctx.set_params(pgs_schedule=0, pgs_grid=0, pgs_plain_launch=0)
    if iterations:
        ctx.autotune(dt, sweeps=3, reps=1, apply=False)  # raises on a shape that changes the bits
    ctx.close()

"""The sweep layout against a plain restatement of its rules: the colouring when
its kernels give up polling and go on in another launch, and the single sweep's
layered colouring, below and above the 4,096 groups that one workgroup lays out."""
import numpy as np
import pytest

from adaptivemerging_amd.context import Context
from adaptivemerging_amd.scene import Scene
from oracle.merging import organized_layers
from tests.helpers import assert_bits_equal, assert_contacts_equal
from tests.test_gpu_parity import _priority

pytestmark = pytest.mark.gpu


def _scene(pairs, on_platform, stack=0):
    """A chain of spheres on a plane, then some alone (together `pairs` touching
    pairs), a platform under on_platform boxes, and a stack of boxes."""
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
    for i in range(stack):
        s.add_box([1.0, 0.2, 1.0], [0.0, 0.099 + 0.199 * i, 30.0])
    return s


@pytest.mark.parametrize("polls", [1, 6])
@pytest.mark.parametrize("pairs,on_platform", [(1, 0), (64, 3), (500, 200), (4026, 69), (4097, 0), (20000, 300)])
def test_colouring_in_several_launches(gpu_lib, pairs, on_platform, polls):
    """With a bound of a few polls the workgroup that lays out a small set gives up
    where a group waits for longer, the launches take over, and those need several
    rounds.  Same order, colours and solve as without a bound."""
    ctxs = []
    for bound in (0, polls):
        ctx = Context()
        ctx.upload(_scene(pairs, on_platform))
        ctx.set_params(iterations=3, tolerance=0.0)
        ctx.set_colour_polls(bound)
        ctx.apply_gravity()
        ctx.detect(0.01)
        ctxs.append(ctx)
    a, b = ctxs
    print("contacts", a.n_contacts(), "colours", a.colours()[1], flush=True)
    assert np.array_equal(a.solve_order(), b.solve_order())
    assert np.array_equal(a.colours()[0], b.colours()[0])
    a.solve(0.01); b.solve(0.01)
    assert_contacts_equal(a.contacts(), b.contacts())
    assert_bits_equal("deltaV", a.pull_deltav(), b.pull_deltav())
    a.close(); b.close()


def _layered_order(body1, body2, layers, pinned):
    """Groups (runs of one body pair) by layer, then priority, each take the
    smallest colour that no group of its layer has at its dynamic bodies, above
    every colour that lower layers have there (at most 64 above; past those the
    next); then order by colour, larger groups first below 64, index."""
    key = np.sort(np.stack([body1, body2], axis=1), axis=1)
    start = np.concatenate([[0], 1 + np.flatnonzero(np.any(np.diff(key, axis=0) != 0, axis=1)), [len(key)]])
    n = len(start) - 1
    layer = [layers[k] for k in start[:-1]]
    taken, colour = {}, np.zeros(n, int)  # per body: its groups' (layer, colour)
    for g in sorted(range(n), key=lambda g: (layer[g], -_priority(g), -g)):
        mine = [taken.setdefault(int(e), []) for e in key[start[g]] if not pinned[e]]
        lo = max([c + 1 for t in mine for l, c in t if l < layer[g]], default=0)
        used = {c for t in mine for l, c in t if l == layer[g]}
        colour[g] = next(c for c in range(lo, lo + 65) if c == lo + 64 or c not in used)
        for t in mine:
            t.append((layer[g], colour[g]))
    size = np.minimum(np.diff(start), 15)
    order = sorted(range(n), key=lambda g: (colour[g], 15 - size[g] if colour[g] < 64 else 0, g))
    return np.concatenate([np.arange(start[g], start[g + 1]) for g in order]), n, colour


@pytest.mark.parametrize("polls", [0, 2])
@pytest.mark.parametrize("pairs,on_platform", [(40, 6), (500, 200), (6600, 200)])
def test_single_sweep_order_is_the_layered_colouring(gpu_lib, pairs, on_platform, polls):
    """The single sweep inside collections, whose colours follow the breadth-first
    layers; more than 64 boxes on the platform put groups of several colours past
    the parallel ones."""
    s = _scene(pairs, on_platform, stack=4)
    # one more box falls on the platform's first: the new contacts of the step that counts
    s.add_box([0.2, 0.2, 0.2], [90.0, 0.86, 0.0])
    pinned = (s.arrays()[0]["flags"] & 1) != 0
    ctx = Context()
    ctx.upload(s)
    ctx.set_params(gravity_amount=9.81, iterations=30, enable_sleeping=0, enable_merge_pinned=0)
    ctx.set_colour_polls(polls)
    dt, seen, most = 0.01, 0, 0
    for step in range(1, 60):
        ctx.clear_bodies(); ctx.apply_gravity(); ctx.update_contacts_map(); ctx.detect(dt); ctx.warm_start()
        new = ctx.contacts()["new_this_step"]
        ctx.update_in_collections(dt)
        inner = ctx.internal_contacts()
        if len(inner["body1"]) and new.any() and step > 10:
            ext = ctx.contacts()
            b1, b2 = (np.concatenate([ext[k], inner[k]]) for k in ("body1", "body2"))
            layers = organized_layers(b1, b2, np.concatenate([new, inner["new_this_step"]]), len(new))
            expect, n, colour = _layered_order(b1, b2, layers, pinned)
            print("step", step, "groups", n, "layers", max(layers) + 1, "colours", colour.max() + 1, flush=True)
            assert np.array_equal(ctx.solve_order(), expect)
            seen, most = seen + 1, max(most, n)
            if on_platform > 64:
                assert len(set(colour[colour >= 64])) > 1
            if seen == 3:
                break
        ctx.accumulate_for_unmerging(dt); ctx.unmerge(dt); ctx.redo_warm_start()
        ctx.solve(dt)
        ctx.clear_body_pair_contacts(); ctx.advance_velocities(dt)
        ctx.accumulate_for_merging(dt); ctx.advance_positions(dt)
        if step % 10 == 0:
            ctx.merge()
    assert seen and (most > 4096) == (pairs > 4096)
    ctx.close()


def test_one_body_groups_among_many(gpu_lib):
    """A contact between two members of one collection among more than 4,096
    groups: the launches' layout reports it too, and the coloured kernel runs."""
    s = _scene(13000, 0, stack=4)  # the chain merges too; 4,335 spheres stay alone
    ctx = Context()
    ctx.upload(s)
    ctx.set_params(gravity_amount=9.81, iterations=30, enable_sleeping=0, enable_merge_pinned=0)
    for _ in range(60):
        if ctx.step(0.01)["n_collections"]:
            break
    parent, _ = ctx.structure()
    coll = max(parent)
    a, b = [i for i, p in enumerate(parent) if p == coll][:2]
    free = [i for i, p in enumerate(parent[:s.n]) if p < 0 and i > 0]
    for inside in (False, True):
        b1 = np.array(([a] if inside else []) + free)
        b2 = np.array(([b] if inside else []) + [0] * len(free))
        n = len(b1)
        assert n > 4096
        ctx.push_contacts(b1, b2, np.zeros((n, 3)), np.tile([0.0, -1.0, 0.0], (n, 1)), np.full(n, -1e-3))
        assert sorted(ctx.solve_order().tolist()) == list(range(n))
        ctx.solve(0.01)
        print("contacts", n, "shape", ctx.launch_shape(), flush=True)
        assert ctx.launch_shape()[1] == (256 if inside else 320)
    ctx.close()

"""The sweep layout below and above the 4,096 groups that one workgroup lays out:
the colouring when its kernels give up polling and go on in another launch."""
import numpy as np
import pytest

from adaptivemerging_amd.context import Context
from adaptivemerging_amd.scene import Scene
from tests.helpers import assert_bits_equal, assert_contacts_equal

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

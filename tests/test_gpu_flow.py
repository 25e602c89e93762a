"""The dataflow schedule of the PGS sweeps (per-body update counters instead
of grid barriers) against the CPU oracle's sequential sweep in the exported
order: lambdas, deltaV, contact states and the per-sweep max |dl| bit-exact.

The schedule double-buffers lambda and deltaV by sweep parity and may run one
sweep past the one that converges, so the cases cover an early exit on odd and
even sweeps, an exit one sweep before the cap and on the cap itself, no exit,
and lanes that own several groups (small grids)."""
import numpy as np
import pytest

from adaptivemerging_amd import workloads
from tests.helpers import assert_bits_equal, assert_contacts_equal, twin

pytestmark = pytest.mark.gpu


def _solve_pair(scene, lam_seed, **params):
    ctx, orc = twin(scene, **params)
    ctx.apply_gravity(); orc.apply_gravity()
    n = ctx.detect(0.01); orc.detect()
    if lam_seed is not None:
        lam = np.random.default_rng(lam_seed).uniform(0, 0.5, size=(n, 3))
        ctx.push_lambdas(lam); orc.push_lambdas(lam)
    it_g, last_g = ctx.solve(0.01)
    order = ctx.solve_order()
    it_o, last_o, ch_o = orc.solve(order, 0.01)
    print("contacts", n, "sweeps", it_g, it_o, "params", params, flush=True)
    assert it_g == it_o
    assert_bits_equal("last_change", np.array([last_g]), np.array([last_o]))
    assert_contacts_equal(ctx.contacts(), orc.contacts())
    assert_bits_equal("deltaV", ctx.pull_deltav(), orc.pull_deltav())
    np.testing.assert_allclose(ctx.changes(), ch_o, rtol=1e-14, atol=0)
    ctx.close()
    return it_g


@pytest.mark.parametrize("grid", [0, 1, 3])
@pytest.mark.parametrize("iterations", [1, 2, 3, 8])
def test_flow_fixed_sweeps(gpu_lib, grid, iterations):
    scene = workloads.box_cluster(seed=11, n=512, spheres=40)
    _solve_pair(scene, 3, iterations=iterations, tolerance=0.0, pgs_grid=grid, pgs_schedule=0)


def test_flow_early_exit_around_the_cap(gpu_lib):
    scene = workloads.jenga_tower(seed=12, layers=8, overlap=0.002)
    kw = dict(tolerance=3e-3, friction_override=1, friction=0.6, pgs_schedule=0)
    t = _solve_pair(scene, None, iterations=1000, **kw)
    assert 4 < t < 1000, f"expected an early exit, got {t} sweeps"
    for cap in (t - 2, t - 1, t, t + 1, t + 4):
        got = _solve_pair(scene, None, iterations=cap, **kw)
        assert got == min(cap, t)


@pytest.mark.parametrize("tolerance", [0.5, 0.3, 0.2, 0.12])
def test_flow_early_exit_odd_and_even(gpu_lib, tolerance):
    scene = workloads.box_cluster(seed=13, n=343, spheres=30)
    _solve_pair(scene, 5, iterations=500, tolerance=tolerance, pgs_schedule=0, pgs_grid=2)


def test_flow_equals_coloured_schedule(gpu_lib):
    from adaptivemerging_amd.context import Context

    scene = workloads.box_cluster(seed=14, n=729, spheres=60)
    out = []
    for schedule in (0, 1):
        ctx = Context()
        ctx.upload(scene)
        ctx.set_params(iterations=30, tolerance=1e-6, gravity_amount=9.81, pgs_schedule=schedule)
        for _ in range(3):
            ctx.step(0.01)
        out.append((ctx.pull_state(), ctx.contacts()["lambda"]))
        ctx.close()
    for a, b in zip(out[0][0], out[1][0]):
        assert_bits_equal("state", a, b)
    assert_bits_equal("lambda", out[0][1], out[1][1])


def test_flow_groups_beyond_the_lds_slots(gpu_lib):
    """Sphere trees resting on planes give body pairs with hundreds of
    contacts: the records past the kernel's LDS slots come from global memory."""
    import collections

    scene = workloads.sphere_tree_drop(seed=5, n=16, heights=(0.15, 0.9), box=(1.2, 1.0, 1.2))
    ctx, orc = twin(scene, iterations=12, tolerance=0.0, gravity_amount=9.81, pgs_schedule=0)
    ctx.apply_gravity(); orc.apply_gravity()
    n = ctx.detect(0.01); orc.detect()
    c = ctx.contacts()
    sizes = collections.Counter(zip(np.minimum(c["body1"], c["body2"]), np.maximum(c["body1"], c["body2"])))
    print("contacts", n, "largest group", max(sizes.values()), flush=True)
    assert max(sizes.values()) > 8
    it_g, _ = ctx.solve(0.01)
    order = ctx.solve_order()
    it_o, _, _ = orc.solve(order, 0.01)
    assert it_g == it_o
    assert_contacts_equal(ctx.contacts(), orc.contacts())
    assert_bits_equal("deltaV", ctx.pull_deltav(), orc.pull_deltav())


@pytest.mark.parametrize("schedule", [0, 1])
def test_flow_unclamped_contacts_take_the_general_update(gpu_lib, schedule):
    """Contacts of magnet-active bodies are not clamped (PGS.java:119-120).
    The dataflow kernel's fast update covers clamped contacts only, so every
    step holding one runs again with the general update; results stay
    bit-exact against the oracle's sequential sweep, at every sweep."""
    from adaptivemerging_amd._lib import AM_BODY_MAGNET_ACTIVE

    scene = workloads.jenga_tower(seed=3, layers=8, overlap=0.002)
    dyn = [i for i in range(scene.n) if not int(scene.bodies[i]["flags"]) & 1]
    for i in dyn[::5]:
        scene.bodies[i]["flags"] = int(scene.bodies[i]["flags"]) | AM_BODY_MAGNET_ACTIVE
    for iterations in (1, 2, 9):
        _solve_pair(scene, 7, iterations=iterations, tolerance=0.0, gravity_amount=9.81, pgs_schedule=schedule)


@pytest.mark.parametrize("spheres,boxes", [(1, 0), (5, 1), (1024, 0), (1025, 0), (0, 1030), (16384, 0), (16385, 3),
                                           (40000, 0), (56000, 0)])
def test_resident_steps_at_their_edges(gpu_lib, spheres, boxes):
    """Bodies of one contact (spheres) and of four (boxes), each alone on a
    plane: one colour, whose groups go to the resident kernel's waves (1024 of
    them, steps of at most 16 groups).  Below and past a group a wave, a full
    step each, a second step for some waves, and more than the LDS of the card
    holds, where k_pgs_flow runs instead.  Against the oracle, bit for bit."""
    from adaptivemerging_amd.scene import Scene

    s = Scene()
    s.add_plane([0, 0, 0], [0, 1, 0], friction=0.6)
    for i in range(spheres + boxes):
        x, z = (i % 200) * 0.5, (i // 200) * 0.5
        v = [0.3, -0.5, 0.1 * (i % 7)]
        if i < spheres:
            s.add_sphere(0.1, [x, 0.099, z], v=v, density=300.0 + i % 11)
        else:
            s.add_box([0.2, 0.1, 0.2], [x, 0.049, z], v=v, density=300.0 + i % 11)
    for iterations in (1, 4):
        ctx, orc = twin(s, iterations=iterations, tolerance=0.0, gravity_amount=9.81)
        ctx.apply_gravity(); orc.apply_gravity()
        n = ctx.detect(0.01); orc.detect()
        ctx.solve(0.01)
        shape = ctx.launch_shape()
        print("contacts", n, "shape", shape, flush=True)
        assert n == spheres + 4 * boxes
        assert shape[1] == (64 if spheres == 56000 else 320)
        orc.solve(ctx.solve_order(), 0.01)
        assert_contacts_equal(ctx.contacts(), orc.contacts())
        assert_bits_equal("deltaV", ctx.pull_deltav(), orc.pull_deltav())
        ctx.close()


def test_the_kernel_follows_the_sweeps_that_run(gpu_lib):
    """The resident kernel takes up to 65,536 sweeps, with 1 KiB of arrival words
    for each: those of the solve at hand, not of the other kind of solve nor of the
    parameters that a tuning run replaces."""
    import ctypes as C

    from adaptivemerging_amd.context import Context

    def free_bytes():
        path = next(ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64" in ln)
        free, total = C.c_size_t(), C.c_size_t()
        assert C.CDLL(path).hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    ctx = Context()
    ctx.upload(workloads.merge_stack(seed=4))
    # the boards merge with each other but not with the ground: contacts for both solves
    ctx.set_params(gravity_amount=9.81, iterations=100, tolerance=1e-10, enable_sleeping=0, enable_merge_pinned=0)
    for _ in range(25):
        st = ctx.step(0.01)
    assert st["n_collections"] >= 1 and ctx.launch_shape()[1] == 320
    # a bound of sweeps for the main solve: a tuning run of 2 sweeps lists what runs them
    ctx.set_params(iterations=70000, tolerance=1e-3)
    ctx.detect(0.01)
    trials, _ = ctx.autotune(0.01, sweeps=2, reps=1, apply=False)
    print("first trial", trials[0], flush=True)
    assert trials[0]["block_used"] == 320
    # many sweeps of the single sweep's solve: k_pgs_flow's words are 64 bytes a sweep
    ctx.set_params(iterations=30)
    ctx.update_in_collections(0.01)
    before = free_bytes()
    ctx.set_params(iterations_in_collection=100000)
    ctx.detect(0.01)
    ctx.update_in_collections(0.01)
    taken = before - free_bytes()
    print("bytes taken", taken, flush=True)
    assert taken < 32 << 20
    ctx.close()


def test_ordinary_launches_of_two_contexts_at_once(gpu_lib):
    """With pgs_plain_launch nothing keeps two contexts' kernels apart: the small
    workgroups of k_pgs_flow run, at any size, which leave room for each other.
    Two threads step a wall of boxes each (2,300 groups: 256 workgroups of the
    resident kernel); both end where one alone does, bit for bit."""
    import threading

    from adaptivemerging_amd.context import Context
    from adaptivemerging_amd.scene import Scene

    scene = Scene()
    scene.add_plane([0, 0, 0], [0, 1, 0], friction=0.8)
    for j in range(30):
        for i in range(40):
            scene.add_box([0.4, 0.2, 0.3], [0.41 * i + 0.2 * (j % 2), 0.0999 + 0.1999 * j, 0])

    def run(out, k):
        ctx = Context()
        ctx.upload(scene)
        ctx.set_params(iterations=60, tolerance=0.0, gravity_amount=9.81, pgs_plain_launch=1, enable_merging=0,
                       enable_sleeping=0)
        for _ in range(20):
            ctx.step(0.005)
        out[k] = (ctx.launch_shape(), ctx.pull_state())
        ctx.close()

    alone, out = {}, {}
    run(alone, 0)
    print("shape", alone[0][0], flush=True)
    assert alone[0][0] == (512, 64)
    ctx = Context()
    ctx.upload(scene)
    ctx.set_params(iterations=60, tolerance=0.0, gravity_amount=9.81, pgs_plain_launch=2, enable_merging=0,
                   enable_sleeping=0)
    for _ in range(20):  # one context at a time: the resident kernel
        ctx.step(0.005)
    assert ctx.launch_shape() == (256, 320)
    for name, a, b in zip("xRvw", alone[0][1], ctx.pull_state()):
        assert_bits_equal(f"resident {name}", b, a)
    ctx.close()
    threads = [threading.Thread(target=run, args=(out, k)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(2):
        for name, a, b in zip("xRvw", alone[0][1], out[k][1]):
            assert_bits_equal(f"context {k} {name}", b, a)

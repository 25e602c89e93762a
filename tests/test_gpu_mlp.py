"""Learned warm start on the GPU: BF16 MFMA forward and backward kernels
against an FP64 NumPy reference with the same BF16 rounding points, Adam
training reduces the loss, and a solve from the predicted start is bit-exact
against the oracle's sweep from the same start."""
import ctypes as C

import numpy as np
import pytest

from adaptivemerging_amd import _lib, workloads
from adaptivemerging_amd.context import Context
from tests import mlp_ref
from tests.helpers import assert_bits_equal, assert_contacts_equal, twin

pytestmark = pytest.mark.gpu


def mlp_call(ctx, name, *args):
    rc = getattr(ctx.lib, name)(ctx.h, *args)
    if rc != 0:
        raise _lib.AMError(rc, ctx.lib.am_last_error(ctx.h).decode())


def init_params(ctx, seed=1):
    mlp_call(ctx, "am_mlp_init", C.c_uint64(seed))
    p = np.zeros(_lib.MLP_PARAMS, np.float32)
    mlp_call(ctx, "am_mlp_get_params", _lib.ptr(p), len(p))
    return p


def test_mlp_forward_matches_fp64_reference(gpu_lib):
    ctx = Context()
    rng = np.random.default_rng(0)
    p = (rng.normal(size=_lib.MLP_PARAMS) * 0.2).astype(np.float32)
    mlp_call(ctx, "am_mlp_set_params", _lib.ptr(p), len(p))
    for n in (1, 15, 16, 17, 200, 1000):
        X = rng.normal(size=(n, 24)).astype(np.float32)
        Y = np.zeros((n, 3), np.float32)
        mlp_call(ctx, "am_mlp_forward", _lib.ptr(X), n, _lib.ptr(Y))
        ref, _ = mlp_ref.forward(p, X)
        # FP32 accumulation vs FP64 can flip a BF16 rounding of a hidden unit
        np.testing.assert_allclose(Y, ref, rtol=5e-3, atol=5e-3)
    q = np.zeros_like(p)
    mlp_call(ctx, "am_mlp_get_params", _lib.ptr(q), len(q))
    assert np.array_equal(p, q)


def test_mlp_gradients_match_fp64_reference(gpu_lib):
    ctx = Context()
    rng = np.random.default_rng(1)
    p = (rng.normal(size=_lib.MLP_PARAMS) * 0.2).astype(np.float32)
    mlp_call(ctx, "am_mlp_set_params", _lib.ptr(p), len(p))
    n = 333
    X = rng.normal(size=(n, 24)).astype(np.float32)
    T = rng.normal(size=(n, 3)).astype(np.float32)
    G = np.zeros(_lib.MLP_PARAMS, np.float32)
    loss = C.c_float()
    mlp_call(ctx, "am_mlp_gradients", _lib.ptr(X), _lib.ptr(T), n, _lib.ptr(G), C.byref(loss))
    Gr, lr = mlp_ref.gradients(p, X, T)
    assert abs(loss.value - lr) < 1e-4 * max(1.0, lr)
    scale = np.max(np.abs(Gr))
    np.testing.assert_allclose(G, Gr, rtol=2e-3, atol=2e-4 * scale)


# tiles of 16 rows, four a workgroup, 512 at once: around one tile, one
# workgroup and one pass of all waves.  Tolerances as above: FP32 sums against
# FP64 ones differ by about 1e-6, and a sum that crosses a BF16 rounding point
# moves one of a row's 195 units by 2^-9 of itself.
@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 8192, 8193])
def test_mlp_gradients_at_tile_edges(gpu_lib, n):
    ctx = Context()
    rng = np.random.default_rng(n)
    p = (rng.normal(size=_lib.MLP_PARAMS) * 0.2).astype(np.float32)
    mlp_call(ctx, "am_mlp_set_params", _lib.ptr(p), len(p))
    X = rng.normal(size=(n, 24)).astype(np.float32)
    T = rng.normal(size=(n, 3)).astype(np.float32)
    Y = np.zeros((n, 3), np.float32)
    mlp_call(ctx, "am_mlp_forward", _lib.ptr(X), n, _lib.ptr(Y))
    np.testing.assert_allclose(Y, mlp_ref.forward(p, X)[0], rtol=5e-3, atol=5e-3)
    loss = C.c_float()
    G = np.zeros(_lib.MLP_PARAMS, np.float32)
    for _ in range(2):  # the workspace is kept: a second call must not add to the first
        mlp_call(ctx, "am_mlp_gradients", _lib.ptr(X), _lib.ptr(T), n, _lib.ptr(G), C.byref(loss))
    Gr, lr = mlp_ref.gradients(p, X, T)
    assert abs(loss.value - lr) < 1e-4 * max(1.0, lr)
    np.testing.assert_allclose(G, Gr, rtol=2e-3, atol=2e-4 * np.max(np.abs(Gr)))


def test_training_reduces_loss(gpu_lib):
    """Pairs come only from solves that reach the tolerance: a shallow pile of
    100 boxes, whose solves reach 1e-6 within the cap."""
    scene = workloads.box_pile(seed=1100, n=100, bin_size=4.0)
    ctx = Context()
    ctx.upload(scene)
    ctx.set_params(iterations=3000, tolerance=1e-6, gravity_amount=9.81, collect_training=0, enable_merging=0,
                   enable_unmerging=0, enable_sleeping=0)
    init_params(ctx)
    for _ in range(60):
        ctx.step(0.01)
    ctx.set_params(collect_training=1)
    converged = 0
    for _ in range(12):
        converged += ctx.step(0.01)["last_change"] < 1e-6
    assert converged >= 3
    n = C.c_int32()
    mlp_call(ctx, "am_train_size", C.byref(n))
    assert n.value > 500
    losses = []
    for _ in range(4):
        l = C.c_float()
        mlp_call(ctx, "am_train_epochs", 5, 256, C.c_float(3e-3), C.c_uint64(7), C.byref(l))
        losses.append(l.value)
    print("losses", losses, flush=True)
    assert losses[-1] < 0.75 * losses[0]


def test_learned_start_solve_bit_exact(gpu_lib):
    scene = workloads.box_cluster(seed=12, n=125, spheres=10)
    ctx, orc = twin(scene, iterations=30, gravity_amount=9.81, learned_warm_start=1)
    init_params(ctx, seed=5)
    ctx.apply_gravity(); orc.apply_gravity()
    n = ctx.detect(0.01); orc.detect()
    lam = np.random.default_rng(4).uniform(0, 0.2, size=(n, 3))
    ctx.push_lambdas(lam)
    ctx.solve(0.01)
    start = np.zeros((n, 3))
    m = C.c_int32()
    mlp_call(ctx, "am_start_lambdas_pull", _lib.ptr(start), n, C.byref(m))
    orc.push_lambdas(start)
    order = ctx.solve_order()
    orc.solve(order, 0.01)
    assert_contacts_equal(ctx.contacts(), orc.contacts(), keys=["lambda", "state", "b", "diag"])
    assert_bits_equal("deltaV", ctx.pull_deltav(), orc.pull_deltav())


def test_learned_start_gain_on_held_out_pile(gpu_lib):
    """What the trained network gains: trained on pairs from converged solves
    of two 100-box piles, it starts the new contacts of a held-out pile while
    the boxes land; sweeps to 1e-6 are counted with and without it from the
    same states.  The learned start is taken only when its start residual is
    below the plain one's.  Measured: no gain to speak of (the sweep count is
    set by the pile's slow modes, not by the start of its new contacts), so
    this asserts only that it costs at most 5 % more sweeps, and prints the
    ratio."""
    params = dict(iterations=3000, tolerance=1e-6, gravity_amount=9.81, enable_merging=0, enable_unmerging=0,
                  enable_sleeping=0)
    tr = Context()
    for seed in (1101, 1102):
        tr.upload(workloads.box_pile(seed=seed, n=100, bin_size=4.0))
        tr.set_params(**params, collect_training=0)
        for _ in range(60):
            tr.step(0.01)
        tr.set_params(collect_training=1)
        for _ in range(15):
            tr.step(0.01)
    assert tr.train_size() > 2000
    tr.mlp_init(3)
    for e in range(8):
        tr.train_epochs(1, 256, 1e-3, 3 + e)
    mlp = tr.mlp_params()
    tr.close()
    held_out = workloads.box_pile(seed=1201, n=100, bin_size=4.0)
    sweeps = {}
    for learned in (0, 1):
        c = Context()
        c.upload(held_out)
        c.set_params(**params)
        for _ in range(10):
            c.step(0.01)
        if learned:
            c.set_mlp_params(mlp)
            c.set_params(learned_warm_start=1)
        total = 0
        for _ in range(20):
            st = c.step(0.01)
            total += st["iterations_used"]
            if learned and st["used_learned"]:
                assert st["start_residual_learned"] < st["start_residual_plain"]
        sweeps[learned] = total
        c.close()
    ratio = sweeps[0] / sweeps[1]
    print(f"sweeps to 1e-6 over 20 steps: plain {sweeps[0]}, learned {sweeps[1]}, ratio {ratio:.3f}", flush=True)
    assert ratio >= 0.95


def test_learned_start_fallback_on_full_pile(gpu_lib):
    """The learned leg of the 20,000-box pile configuration with an untrained
    network: after the pile has settled, each step evaluates the prediction's
    start residual against the plain start's and keeps the plain start unless
    the prediction is better.  Steps that keep it equal a plain context's
    steps bit for bit (positions, rotations, velocities); at least one step
    must keep it, and every state stays finite."""
    scene = workloads.box_pile(seed=0, n=20000)
    kw = dict(iterations=100, tolerance=1e-6, gravity_amount=9.81, enable_merging=0, enable_unmerging=0,
              enable_sleeping=0)
    plain, lrn = Context(), Context()
    for c in (plain, lrn):
        c.upload(scene)
        c.set_params(**kw)
        for _ in range(300):
            c.step(0.01)
    lrn.mlp_init(11)
    lrn.set_params(learned_warm_start=1)
    kept = 0
    for step in range(4):
        sp = plain.step(0.01)
        sl = lrn.step(0.01)
        print(f"step {step}: contacts {sl['n_contacts']} used_learned {sl['used_learned']} start residual plain "
              f"{sl['start_residual_plain']:.4g} learned {sl['start_residual_learned']:.4g}", flush=True)
        for name, a, b in zip("xRvw", plain.pull_state(), lrn.pull_state()):
            assert np.all(np.isfinite(b)), name
        if sl["used_learned"]:
            assert sl["start_residual_learned"] < sl["start_residual_plain"]
            break
        kept += 1
        assert sl["iterations_used"] == sp["iterations_used"]
        for name, a, b in zip("xRvw", plain.pull_state(), lrn.pull_state()):
            assert_bits_equal(f"step {step} {name}", a, b)
    assert kept >= 1
    plain.close()
    lrn.close()

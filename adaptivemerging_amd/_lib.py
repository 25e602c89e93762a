"""ctypes binding of libam.so (include/am.h).

The library is loaded from this package directory.  There is no fallback: if
libam.so is missing or a call fails, an AMError is raised.
"""
from __future__ import annotations

import ctypes as C
import os

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libam.so")

AM_OK = 0
AM_ERR_INVALID = -1
AM_ERR_HIP = -2
AM_ERR_CAPACITY = -3
AM_ERR_STATE = -4
AM_ERR_NUMERIC = -5
AM_ERR_MISMATCH = -6

AM_GEOM_BOX = 0
AM_GEOM_TREE = 1
AM_GEOM_PLANE = 2
AM_GEOM_COLLECTION = 3

AM_BODY_PINNED = 1
AM_BODY_MAGNET_ACTIVE = 2
AM_BODY_SLEEPING = 4
AM_BODY_KINEMATIC = 8
AM_GEOM_COMPOSITE = 4


def AM_BV_SUB(s: int, bv: int) -> int:
    """The bv id of a contact on sub-body s of a composite (include/am.h)."""
    return -3 - (s << 16) - (bv + 1)
AM_SLEEP_HIST_STRIDE = 201

AM_STATE_BROKEN = 0
AM_STATE_ONEDGE = 1
AM_STATE_CLEAR = 2

AM_BV_NONE = -1
AM_BV_PLANE = -2

# numpy views of the C structs (no padding in either layout)
BODY_DTYPE = np.dtype(
    [
        ("geom", "<i4"), ("flags", "<i4"), ("tree_first", "<i4"), ("tree_count", "<i4"),
        ("scene", "<i4"), ("reserved", "<i4"),
        ("size", "<f8", 3), ("radius", "<f8"), ("mass", "<f8"), ("minv", "<f8"),
        ("jinv0", "<f8", 9), ("friction", "<f8"), ("restitution", "<f8"),
        ("plane_n", "<f8", 3), ("plane_p", "<f8", 3), ("plane_d", "<f8"), ("bbox", "<f8", 24),
        ("inertia0", "<f8", 9),
    ]
)
NODE_DTYPE = np.dtype([("c", "<f8", 3), ("r", "<f8"), ("first_child", "<i4"), ("n_children", "<i4")])
AM_SPRING_ZERO, AM_SPRING_WORLD, AM_SPRING_BODYBODY = 0, 1, 2
SPRING_DTYPE = np.dtype([("type", "<i4"), ("body1", "<i4"), ("body2", "<i4"), ("pad", "<i4"), ("pb1", "<f8", 3),
                         ("pb2", "<f8", 3), ("pw", "<f8", 3), ("l0", "<f8"), ("k", "<f8"), ("d", "<f8"),
                         ("ls", "<f8")])
KINEMATIC_DTYPE = np.dtype([("body", "<i4"), ("pad", "<i4"), ("x0", "<f8", 3), ("dir", "<f8", 3),
                            ("amplitude", "<f8"), ("omega", "<f8"), ("phase", "<f8")])
assert BODY_DTYPE.itemsize == 480 and NODE_DTYPE.itemsize == 40 and KINEMATIC_DTYPE.itemsize == 80


class Params(C.Structure):
    _fields_ = [
        ("iterations", C.c_int32), ("iterations_in_collection", C.c_int32),
        ("tolerance", C.c_double), ("omega", C.c_double), ("feedback_stiffness", C.c_double),
        ("enable_post_stabilization", C.c_int32), ("enable_compliance", C.c_int32),
        ("compliance", C.c_double),
        ("restitution_override", C.c_int32), ("friction_override", C.c_int32),
        ("restitution", C.c_double), ("friction", C.c_double), ("sliding_threshold", C.c_double),
        ("warm_start", C.c_int32), ("use_gravity", C.c_int32),
        ("gravity_amount", C.c_double), ("gravity_angle_deg", C.c_double),
        ("viscous_linear_decay", C.c_double), ("viscous_angular_decay", C.c_double),
        ("spring_stiffness_mod", C.c_double), ("spring_damping_mod", C.c_double),
        ("enable_sleeping", C.c_int32), ("sleep_step_accum", C.c_int32), ("sleep_threshold", C.c_double),
        ("enable_merging", C.c_int32), ("enable_merge_pinned", C.c_int32),
        ("enable_merge_stable_contact", C.c_int32), ("enable_merge_let_it_breathe", C.c_int32),
        ("enable_unmerging", C.c_int32), ("enable_unmerge_friction", C.c_int32),
        ("enable_unmerge_normal", C.c_int32), ("enable_unmerge_relative_motion", C.c_int32),
        ("update_contacts_in_collections", C.c_int32), ("step_accum_merging", C.c_int32),
        ("step_accum_unmerging", C.c_int32), ("steps_between_merge_events", C.c_int32),
        ("metric_position_level", C.c_int32),
        ("threshold_merge", C.c_double), ("threshold_unmerge", C.c_double), ("threshold_breath", C.c_double),
        ("pgs_block", C.c_int32), ("pgs_grid", C.c_int32), ("pgs_plain_launch", C.c_int32),
        ("pgs_schedule", C.c_int32),
        ("learned_warm_start", C.c_int32), ("collect_training", C.c_int32),
        ("organize_contacts", C.c_int32), ("host_threads", C.c_int32),
    ]


_DP = C.POINTER(C.c_double)
_IP = C.POINTER(C.c_int32)


class ContactArrays(C.Structure):
    _fields_ = [
        ("body1", _IP), ("body2", _IP), ("bv1", _IP), ("bv2", _IP), ("info", _IP),
        ("point_b1", _DP), ("normal_b1", _DP), ("tangent1_b1", _DP), ("tangent2_b1", _DP),
        ("violation", _DP), ("prev_violation", _DP), ("jacobian", _DP),
        ("lambda_", _DP), ("lambda_warm", _DP), ("b", _DP), ("diag", _DP),
        ("state", _IP), ("new_this_step", _IP),
    ]


class StepStats(C.Structure):
    _fields_ = [
        ("n_contacts", C.c_int32), ("n_pairs", C.c_int32), ("n_groups", C.c_int32), ("n_colours", C.c_int32),
        ("iterations_used", C.c_int32), ("bad_warm_starts", C.c_int32),
        ("bad_warm_starts_repaired", C.c_int32), ("reserved", C.c_int32),
        ("last_change", C.c_double), ("ms_detect", C.c_double), ("ms_warm_start", C.c_double),
        ("ms_solve", C.c_double), ("ms_integrate", C.c_double), ("ms_total", C.c_double),
        ("ms_pgs_kernel", C.c_double), ("ms_setup_kernel", C.c_double), ("ms_learned", C.c_double),
        ("start_residual_plain", C.c_double), ("start_residual_learned", C.c_double),
        ("used_learned", C.c_int32), ("n_collections", C.c_int32), ("n_merged", C.c_int32),
        ("n_unmerged", C.c_int32), ("n_internal_contacts", C.c_int32), ("n_sleeping", C.c_int32),
        ("ms_merging", C.c_double),
    ]

    def as_dict(self) -> dict:
        return {k: getattr(self, k) for k, _ in self._fields_ if not k.startswith("reserved")}


class TuneTrial(C.Structure):
    _fields_ = [
        ("pgs_schedule", C.c_int32), ("pgs_grid", C.c_int32), ("pgs_block", C.c_int32),
        ("grid_used", C.c_int32), ("block_used", C.c_int32), ("reserved", C.c_int32),
        ("ms_per_sweep", C.c_double),
    ]

    def as_dict(self) -> dict:
        return {k: getattr(self, k) for k, _ in self._fields_ if not k.startswith("reserved")}


class BodyPair(C.Structure):
    _fields_ = [
        ("body1", C.c_int32), ("body2", C.c_int32), ("in_collection", C.c_int32), ("n_contacts", C.c_int32),
        ("hist_n", C.c_int32), ("state_n", C.c_int32), ("flag", C.c_int32), ("collection", C.c_int32),
        ("hist", C.c_double * 8), ("states", C.c_int32 * 8),
    ]


# Exported symbols of include/am.h; the test suite checks this list against
# the header and the shared object.
SYMBOLS = [
    "am_version", "am_ctx_create", "am_ctx_destroy", "am_last_error", "am_params_default", "am_params_set",
    "am_scene_upload", "am_scene_upload_ex", "am_structure_pull", "am_entities_pull", "am_jinv_pull", "am_state_push",
    "am_state_pull", "am_forces_push", "am_forces_pull", "am_clear_bodies", "am_apply_gravity", "am_deltav_pull",
    "am_springs_set", "am_apply_spring_forces", "am_wake", "am_sleep", "am_wake_all", "am_sleep_state_pull", "am_unmerge_all",
    "am_update_contacts_map", "am_detect", "am_contacts_push", "am_contacts_pull", "am_lambdas_push",
    "am_warm_start", "am_redo_warm_start", "am_no_warm_start", "am_solve", "am_solve_order_pull",
    "am_colours_pull", "am_colour_polls_set", "am_update_in_collections", "am_changes_pull", "am_advance_velocities",
    "am_advance_positions", "am_accumulate_for_unmerging", "am_unmerge", "am_clear_top_level",
    "am_clear_body_pair_contacts", "am_accumulate_for_merging", "am_merge", "am_body_pairs_pull",
    "am_internal_contacts_pull",
    "am_step", "am_motion_metric", "am_mlp_init", "am_mlp_set_params", "am_mlp_get_params", "am_mlp_forward",
    "am_mlp_gradients", "am_features_pull", "am_train_size", "am_train_clear", "am_train_epochs",
    "am_start_lambdas_pull", "am_autotune", "am_advance_positions_post", "am_impulse_add", "am_kinematic_set",
    "am_kinematic_update", "am_sim_time_get", "am_sim_time_set", "am_apply_impulses", "am_apply_viscous_decay",
    "am_scene_iterations_pull", "am_motion_metric_noalloc", "am_launch_shape_pull",
]
AM_METRIC_NOALLOC_MAX = 65536
MLP_PARAMS = 10115
MLP_FEATURES = 24


class AMError(RuntimeError):
    def __init__(self, code: int, msg: str):
        super().__init__(f"libam error {code}: {msg}")
        self.code = code


_lib = None


def load(path: str = LIB_PATH) -> C.CDLL:
    """Loads libam.so from the package directory (raises if it is missing)."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(path):
        raise AMError(AM_ERR_STATE, f"{path} is not built; run adaptivemerging_amd/build.py")
    lib = C.CDLL(path)
    i32, dbl, vp = C.c_int32, C.c_double, C.c_void_p
    ctxp = C.c_void_p
    sig = {
        "am_version": (C.c_char_p, []),
        "am_ctx_create": (C.c_int, [i32, C.POINTER(ctxp)]),
        "am_ctx_destroy": (C.c_int, [ctxp]),
        "am_last_error": (C.c_char_p, [ctxp]),
        "am_params_default": (C.c_int, [C.POINTER(Params)]),
        "am_params_set": (C.c_int, [ctxp, C.POINTER(Params)]),
        "am_scene_upload": (C.c_int, [ctxp, vp, i32, vp, i32]),
        "am_scene_upload_ex": (C.c_int, [ctxp, vp, i32, vp, i32, vp, vp, i32]),
        "am_structure_pull": (C.c_int, [ctxp, vp, i32, vp, i32, C.POINTER(i32), C.POINTER(i32)]),
        "am_entities_pull": (C.c_int, [ctxp, vp, i32]),
        "am_jinv_pull": (C.c_int, [ctxp, vp, i32]),
        "am_state_push": (C.c_int, [ctxp, vp, vp, vp, vp, i32]),
        "am_state_pull": (C.c_int, [ctxp, vp, vp, vp, vp, i32]),
        "am_forces_push": (C.c_int, [ctxp, vp, vp, i32]),
        "am_forces_pull": (C.c_int, [ctxp, vp, vp, i32]),
        "am_clear_bodies": (C.c_int, [ctxp]),
        "am_apply_gravity": (C.c_int, [ctxp]),
        "am_springs_set": (C.c_int, [ctxp, vp, i32]),
        "am_apply_spring_forces": (C.c_int, [ctxp]),
        "am_wake": (C.c_int, [ctxp, vp]),
        "am_sleep": (C.c_int, [ctxp, vp]),
        "am_wake_all": (C.c_int, [ctxp]),
        "am_unmerge_all": (C.c_int, [ctxp, vp]),
        "am_sleep_state_pull": (C.c_int, [ctxp, vp, vp, vp, i32]),
        "am_deltav_pull": (C.c_int, [ctxp, vp, i32]),
        "am_update_contacts_map": (C.c_int, [ctxp]),
        "am_detect": (C.c_int, [ctxp, dbl, C.POINTER(i32)]),
        "am_contacts_push": (C.c_int, [ctxp, i32, vp, vp, vp, vp, vp, vp, vp, vp]),
        "am_contacts_pull": (C.c_int, [ctxp, C.POINTER(ContactArrays), i32, C.POINTER(i32)]),
        "am_lambdas_push": (C.c_int, [ctxp, vp, i32]),
        "am_warm_start": (C.c_int, [ctxp, i32, C.POINTER(i32), C.POINTER(i32)]),
        "am_redo_warm_start": (C.c_int, [ctxp]),
        "am_no_warm_start": (C.c_int, [ctxp]),
        "am_solve": (C.c_int, [ctxp, dbl, i32, C.POINTER(i32), C.POINTER(dbl)]),
        "am_solve_order_pull": (C.c_int, [ctxp, vp, i32, C.POINTER(i32)]),
        "am_colours_pull": (C.c_int, [ctxp, vp, i32, C.POINTER(i32)]),
        "am_colour_polls_set": (C.c_int, [ctxp, i32]),
        "am_update_in_collections": (C.c_int, [ctxp, dbl, C.POINTER(i32)]),
        "am_accumulate_for_unmerging": (C.c_int, [ctxp, dbl]),
        "am_unmerge": (C.c_int, [ctxp, dbl, C.POINTER(i32)]),
        "am_clear_top_level": (C.c_int, [ctxp]),
        "am_clear_body_pair_contacts": (C.c_int, [ctxp]),
        "am_accumulate_for_merging": (C.c_int, [ctxp, dbl]),
        "am_merge": (C.c_int, [ctxp, C.POINTER(i32)]),
        "am_body_pairs_pull": (C.c_int, [ctxp, vp, i32, C.POINTER(i32), C.POINTER(i32)]),
        "am_internal_contacts_pull": (C.c_int, [ctxp, C.POINTER(ContactArrays), i32, C.POINTER(i32)]),
        "am_changes_pull": (C.c_int, [ctxp, vp, i32, C.POINTER(i32)]),
        "am_advance_velocities": (C.c_int, [ctxp, dbl]),
        "am_advance_positions": (C.c_int, [ctxp, dbl]),
        "am_advance_positions_post": (C.c_int, [ctxp, dbl]),
        "am_step": (C.c_int, [ctxp, dbl, C.POINTER(StepStats)]),
        "am_motion_metric": (C.c_int, [ctxp, vp, i32, vp]),
        "am_autotune": (C.c_int, [ctxp, dbl, i32, i32, i32, C.POINTER(TuneTrial), i32, C.POINTER(i32),
                                  C.POINTER(i32)]),
        "am_mlp_init": (C.c_int, [ctxp, C.c_uint64]),
        "am_mlp_set_params": (C.c_int, [ctxp, vp, i32]),
        "am_mlp_get_params": (C.c_int, [ctxp, vp, i32]),
        "am_mlp_forward": (C.c_int, [ctxp, vp, i32, vp]),
        "am_mlp_gradients": (C.c_int, [ctxp, vp, vp, i32, vp, C.POINTER(C.c_float)]),
        "am_features_pull": (C.c_int, [ctxp, vp, vp, i32, C.POINTER(i32)]),
        "am_train_size": (C.c_int, [ctxp, C.POINTER(i32)]),
        "am_train_clear": (C.c_int, [ctxp]),
        "am_train_epochs": (C.c_int, [ctxp, i32, i32, C.c_float, C.c_uint64, C.POINTER(C.c_float)]),
        "am_start_lambdas_pull": (C.c_int, [ctxp, vp, i32, C.POINTER(i32)]),
        "am_impulse_add": (C.c_int, [ctxp, i32, vp, vp]),
        "am_kinematic_set": (C.c_int, [ctxp, vp, i32]),
        "am_kinematic_update": (C.c_int, [ctxp, dbl]),
        "am_sim_time_get": (C.c_int, [ctxp, C.POINTER(dbl)]),
        "am_sim_time_set": (C.c_int, [ctxp, dbl]),
        "am_apply_impulses": (C.c_int, [ctxp]),
        "am_apply_viscous_decay": (C.c_int, [ctxp]),
        "am_scene_iterations_pull": (C.c_int, [ctxp, vp, vp, i32, C.POINTER(i32)]),
        "am_motion_metric_noalloc": (C.c_int, [ctxp, vp, i32, vp]),
        "am_launch_shape_pull": (C.c_int, [ctxp, C.POINTER(i32), C.POINTER(i32)]),
    }
    for name, (res, args) in sig.items():
        f = getattr(lib, name)
        f.restype = res
        f.argtypes = args
    _lib = lib
    return lib


def default_params() -> Params:
    p = Params()
    load().am_params_default(C.byref(p))
    return p


def ptr(a):
    """Raw data pointer of a numpy array (or None)."""
    if a is None:
        return None
    return C.c_void_p(a.ctypes.data)


def dptr(a):
    return None if a is None else a.ctypes.data_as(_DP)


def iptr(a):
    return None if a is None else a.ctypes.data_as(_IP)


# Reference defaults (CollisionProcessor.java:1058-1083, Merging.java:31-48,
# Contact.java:518, RigidBodySystem.java:545-551); equal to am_params_default.
_DEFAULTS = dict(
    iterations=30, iterations_in_collection=1, tolerance=1e-5, omega=1.0, feedback_stiffness=0.5,
    enable_post_stabilization=0, enable_compliance=1, compliance=1e-3, restitution_override=0,
    friction_override=0, restitution=0.5, friction=0.1, sliding_threshold=0.01, warm_start=1, use_gravity=1,
    gravity_amount=1.0, gravity_angle_deg=90.0, viscous_linear_decay=1.0, viscous_angular_decay=1.0,
    spring_stiffness_mod=1.0, spring_damping_mod=1.0, enable_sleeping=1, sleep_step_accum=10, sleep_threshold=1e-5,
    enable_merging=1, enable_merge_pinned=1, enable_merge_stable_contact=1, enable_merge_let_it_breathe=1,
    enable_unmerging=1, enable_unmerge_friction=1, enable_unmerge_normal=1, enable_unmerge_relative_motion=1,
    update_contacts_in_collections=1, step_accum_merging=3, step_accum_unmerging=3, steps_between_merge_events=10,
    metric_position_level=0,
    threshold_merge=1e-2, threshold_unmerge=2e-2, threshold_breath=1e-5, pgs_block=0, pgs_grid=0, pgs_plain_launch=0, pgs_schedule=0,
    learned_warm_start=0, collect_training=0, organize_contacts=1, host_threads=0,
)


def default_params_host() -> Params:
    """The reference defaults without loading libam."""
    p = Params()
    for k, v in _DEFAULTS.items():
        setattr(p, k, v)
    return p

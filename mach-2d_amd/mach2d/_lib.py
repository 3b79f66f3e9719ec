"""ctypes binding of the C ABI in include/mach2d_hip.h (libmach2d_hip.so).

The shared library is built in-tree by mach-2d_amd/build.py (hipcc for
gfx950).  Loading fails loudly when it is missing: there is no CPU fallback.
"""
from __future__ import annotations

import ctypes as C
import os

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libmach2d_hip.so")

M2D_OK = 0
M2D_ERR_NONFINITE = 1
M2D_ERR_HIP = 3
M2D_ERR_ARG = 4
M2D_ERR_OUTSIDE_COUPLING = 5
M2D_ERR_SYNC_TIMEOUT = 6
M2D_ERR_ITER_CAP = 7

M2D_FP64 = 0
M2D_FP32_IR = 1

STATUS_NAMES = {
    M2D_OK: "ok",
    M2D_ERR_NONFINITE: "non-finite pivot or residual",
    M2D_ERR_HIP: "HIP runtime error",
    M2D_ERR_ARG: "invalid argument",
    M2D_ERR_OUTSIDE_COUPLING: "coupling to a neighbour outside the grid",
    M2D_ERR_SYNC_TIMEOUT: "inter-workgroup wait timed out",
    M2D_ERR_ITER_CAP: "iteration safety cap reached (nitm <= 0)",
}


class Status(C.Structure):
    _fields_ = [("status", C.c_int), ("nit", C.c_int), ("nitm_reached", C.c_int),
                ("outer", C.c_int), ("r0", C.c_double), ("rn", C.c_double),
                ("gammarp", C.c_double), ("device_ms", C.c_double)]

    def as_dict(self):
        return {k: getattr(self, k) for k, _ in self._fields_}


# every symbol include/mach2d_hip.h declares
EXPORTS = [
    "m2d_lu2d9", "m2d_fb2d9", "m2d_tdma2d9", "m2d_solve_msi9d",
    "m2d_lu2d5", "m2d_fb2d5", "m2d_solve_msi5d", "m2d_create_stencil", "m2d_norm_l1_9d",
    "m2d_norm_l1_9d_relative", "m2d_norm_l1_b", "m2d_last_status", "m2d_create",
    "m2d_destroy", "m2d_set_stream", "m2d_factor", "m2d_solve", "m2d_set_inner",
    "m2d_set_window", "m2d_get_window", "m2d_batch_set_window", "m2d_batch_get_window",
    "m2d_get_factor", "m2d_set_tuning", "m2d_set_staging", "m2d_tdma2d9_device",
    "m2d_residual_norm", "m2d_guess_scale", "m2d_guess_scale_energy",
    "m2d_version", "m2d_enable_kernel_timing", "m2d_kernel_timing",
    "m2d_batch_create", "m2d_batch_destroy", "m2d_batch_set_stream", "m2d_batch_factor",
    "m2d_batch_solve", "m2d_batch_solve_each", "m2d_batch_set_inner", "m2d_batch_set_tuning", "m2d_batch_get_tuning",
    "m2d_batch_tune", "m2d_assembly_set_stream", "m2d_get_density_at_nodes",
    "m2d_get_density_at_faces",
    "m2d_get_u_coefficients", "m2d_get_u_source", "m2d_get_v_coefficients", "m2d_get_v_source",
    "m2d_get_T_coefficients_and_source", "m2d_get_p_coefficients", "m2d_get_p_source",
    "m2d_get_velocities_at_internal_faces", "m2d_get_internal_simplec_coefficients",
    "m2d_get_pressure_correction_with_pl", "m2d_get_density_correction_with_pl",
    "m2d_get_u_v_at_real_nodes_with_pl", "m2d_get_velocity_correction_at_faces_with_pl",
    "m2d_initialize_boundary_faces_flags", "m2d_check_mass_conservation",
    "m2d_intflow_set_bcu", "m2d_intflow_set_bcv", "m2d_intflow_set_bcpl", "m2d_intflow_set_bcT",
    "m2d_intflow_velocities_at_boundary_faces", "m2d_intflow_pl_loop",
    "m2d_set_pl_graph", "m2d_pl_loop_info", "m2d_set_pl_solve_cap", "m2d_pl_loop_cap_info",
    "m2d_get_mean_cc_9d", "m2d_get_mean_cc_5d", "m2d_tstepper_dt0_scarborough",
    "m2d_tstepper_dt_scarborough",
    "m2d_get_real_centroids_xy", "m2d_get_metrics", "m2d_get_radius",
    "m2d_intflow_boundary_simplec", "m2d_intflow_extrapolate_u_v_to_fictitious",
    "m2d_intflow_boundary_T_from_H_conservation", "m2d_intflow_time_cycle_update",
    "m2d_norm_l1_5d", "m2d_get_average", "m2d_intflow_time_step", "m2d_guess_prepare_many",
    "m2d_unet_conv3x3", "m2d_unet_conv3x3_wgrad", "m2d_unet_relu_bwd", "m2d_unet_mode_bwd",
    "m2d_unet_to_bf16", "m2d_unet_adam", "m2d_unet_pack_weights", "m2d_unet_mse",
    "m2d_unet_pack_input", "m2d_unet_unpack_output", "m2d_solve_msi9d_noalloc",
    "m2d_tdma2d9_device_many", "m2d_set_tdma_mode",
    "m2d_unet_pack_weights_many", "m2d_unet_grad_in", "m2d_unet_mse_count",
]

_lib = None

_ip = C.POINTER(C.c_int)
_dp = C.POINTER(C.c_double)
_vp = C.c_void_p


def load():
    """Load the library (does not touch the GPU)."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise RuntimeError(
            "libmach2d_hip.so is not built (%s); run `python mach-2d_amd/build.py` "
            "or __graft_entry__.build()" % LIB_PATH)
    # PyTorch-ROCm carries its own HIP runtime: with it loaded first, this
    # library's HIP calls bind to that runtime, so device memory and streams
    # from torch and this library's kernels share one runtime.  Loaded the
    # other way round, a second runtime comes up and launches can fail
    # ("invalid device function").
    try:
        import torch  # noqa: F401
    except ImportError:
        pass
    L = C.CDLL(LIB_PATH)
    for f in (L.m2d_lu2d9, L.m2d_lu2d5):
        f.argtypes = [_vp, _vp, _vp, _ip, _ip, _ip]
        f.restype = None
    for f in (L.m2d_fb2d9, L.m2d_fb2d5):
        f.argtypes = [_vp, _vp, _vp, _ip, _ip, _ip, _vp, _dp, _ip, _vp]
        f.restype = None
    L.m2d_tdma2d9.argtypes = [_ip, _ip, _ip, _vp, _vp, _vp]
    L.m2d_tdma2d9.restype = None
    for f in (L.m2d_solve_msi9d, L.m2d_solve_msi5d):
        f.argtypes = [_ip, _ip, _ip, _dp, _vp, _vp, _vp]
        f.restype = None
    for f in (L.m2d_norm_l1_9d, L.m2d_norm_l1_9d_relative):
        f.argtypes = [_ip, _ip, _vp, _vp, _vp, _dp]
        f.restype = None
    L.m2d_norm_l1_b.argtypes = [_ip, _ip, _vp]
    L.m2d_norm_l1_b.restype = C.c_double
    L.m2d_last_status.argtypes = [C.POINTER(Status)]
    L.m2d_last_status.restype = C.c_int
    L.m2d_create.argtypes = [C.c_int, C.c_int, C.c_int, C.POINTER(_vp)]
    L.m2d_create.restype = C.c_int
    L.m2d_create_stencil.argtypes = [C.c_int, C.c_int, C.c_int, C.c_int, C.POINTER(_vp)]
    L.m2d_create_stencil.restype = C.c_int
    L.m2d_destroy.argtypes = [_vp]
    L.m2d_destroy.restype = C.c_int
    L.m2d_set_stream.argtypes = [_vp, _vp]
    L.m2d_set_stream.restype = C.c_int
    L.m2d_factor.argtypes = [_vp, _vp]
    L.m2d_factor.restype = C.c_int
    L.m2d_solve.argtypes = [_vp, _vp, _vp, _vp, C.c_double, C.c_int, _vp, C.c_int,
                            C.POINTER(Status)]
    L.m2d_solve.restype = C.c_int
    L.m2d_set_inner.argtypes = [_vp, C.c_double, C.c_int]
    L.m2d_set_inner.restype = C.c_int
    for f in (L.m2d_set_window, L.m2d_batch_set_window):
        f.argtypes, f.restype = [_vp, C.c_int], C.c_int
    for f in (L.m2d_get_window, L.m2d_batch_get_window):
        f.argtypes, f.restype = [_vp, C.POINTER(C.c_int)], C.c_int
    L.m2d_residual_norm.argtypes = [_vp, _vp, _vp, _vp, C.POINTER(C.c_double)]
    for f in (L.m2d_guess_scale, L.m2d_guess_scale_energy):
        f.argtypes = [_vp, _vp, _vp, _vp, C.POINTER(C.c_double)]
        f.restype = C.c_int
    L.m2d_set_staging.argtypes = [_vp, C.c_int]
    L.m2d_set_staging.restype = C.c_int
    L.m2d_residual_norm.restype = C.c_int
    L.m2d_get_factor.argtypes = [_vp, _vp, _vp]
    L.m2d_get_factor.restype = C.c_int
    L.m2d_set_tuning.argtypes = [_vp, C.c_int, C.c_int]
    L.m2d_set_tuning.restype = C.c_int
    _pp = C.POINTER(_vp)
    L.m2d_batch_create.argtypes = [C.c_int, _ip, _ip, C.c_int, C.POINTER(_vp)]
    L.m2d_batch_destroy.argtypes = [_vp]
    L.m2d_batch_set_stream.argtypes = [_vp, _vp]
    L.m2d_batch_factor.argtypes = [_vp, _pp]
    L.m2d_batch_solve.argtypes = [_vp, _pp, _pp, _pp, C.c_double, C.c_int, C.POINTER(Status)]
    L.m2d_batch_solve_each.argtypes = [_vp, _pp, _pp, _pp, C.POINTER(C.c_double), C.c_int,
                                       C.POINTER(Status)]
    L.m2d_batch_set_inner.argtypes = [_vp, C.c_double, C.c_int]
    L.m2d_batch_set_tuning.argtypes = [_vp, C.c_int, C.c_int]
    L.m2d_batch_get_tuning.argtypes = [_vp, _ip, _ip]
    L.m2d_batch_tune.argtypes = [_vp, _pp, _pp, C.c_int, _ip, _dp]
    for f in (L.m2d_batch_create, L.m2d_batch_destroy, L.m2d_batch_set_stream,
              L.m2d_batch_factor, L.m2d_batch_solve, L.m2d_batch_solve_each,
              L.m2d_batch_set_inner,
              L.m2d_batch_set_tuning, L.m2d_batch_get_tuning, L.m2d_batch_tune):
        f.restype = C.c_int
    L.m2d_assembly_set_stream.argtypes = [_vp]
    L.m2d_assembly_set_stream.restype = None
    for nm in ("get_density_at_nodes", "get_density_at_faces", "get_u_coefficients", "get_u_source",
               "get_v_coefficients", "get_v_source", "get_T_coefficients_and_source",
               "get_p_coefficients", "get_p_source", "get_velocities_at_internal_faces",
               "get_internal_simplec_coefficients", "get_pressure_correction_with_pl",
               "get_density_correction_with_pl", "get_u_v_at_real_nodes_with_pl",
               "get_velocity_correction_at_faces_with_pl", "initialize_boundary_faces_flags",
               "check_mass_conservation"):
        getattr(L, "m2d_" + nm).restype = None   # pointer arguments, by reference
    L.m2d_tdma2d9_device.argtypes = [C.c_int, C.c_int, C.c_int, _vp, _vp, _vp, _vp]
    L.m2d_tdma2d9_device.restype = C.c_int
    L.m2d_tdma2d9_device_many.argtypes = [C.c_int, C.c_int, C.c_int, C.c_int, _vp, _vp, _vp,
                                          _vp]
    L.m2d_tdma2d9_device_many.restype = C.c_int
    L.m2d_set_tdma_mode.argtypes = [C.c_int]
    L.m2d_set_tdma_mode.restype = C.c_int
    L.m2d_solve_msi9d_noalloc.argtypes = [_ip, _ip, _ip, _dp, _vp, _vp, _vp, _vp]
    L.m2d_solve_msi9d_noalloc.restype = C.c_int
    L.m2d_enable_kernel_timing.argtypes = [_vp, C.c_int]
    L.m2d_enable_kernel_timing.restype = C.c_int
    L.m2d_kernel_timing.argtypes = [_vp, C.c_int, _dp, C.POINTER(C.c_long)]
    L.m2d_kernel_timing.restype = C.c_int
    L.m2d_intflow_pl_loop.argtypes = [_vp, _vp, C.c_int, C.c_double, C.c_double, C.c_double,
                                      C.c_double, C.c_int, C.c_int, C.c_double, _ip,
                                      C.POINTER(C.c_double)]
    L.m2d_intflow_pl_loop.restype = C.c_int
    L.m2d_set_pl_graph.argtypes = [_vp, C.c_int]
    L.m2d_set_pl_graph.restype = C.c_int
    L.m2d_pl_loop_info.argtypes = [_vp, _ip, _ip]
    L.m2d_pl_loop_info.restype = C.c_int
    L.m2d_set_pl_solve_cap.argtypes = [_vp, C.c_int]
    L.m2d_set_pl_solve_cap.restype = C.c_int
    L.m2d_pl_loop_cap_info.argtypes = [_vp, _ip, _ip]
    L.m2d_pl_loop_cap_info.restype = C.c_int
    for f in (L.m2d_get_mean_cc_9d, L.m2d_get_mean_cc_5d):
        f.argtypes = [_ip, _ip, _vp]
        f.restype = C.c_double
    L.m2d_tstepper_dt0_scarborough.argtypes = [_ip, _ip, _vp, _vp, _vp]
    L.m2d_tstepper_dt0_scarborough.restype = C.c_double
    L.m2d_tstepper_dt_scarborough.argtypes = [_ip, _ip, _dp, _vp, _vp, _vp, _vp, _dp, _dp, _dp]
    L.m2d_tstepper_dt_scarborough.restype = C.c_double
    L.m2d_get_real_centroids_xy.argtypes = [_ip, _ip, _ip] + [_vp] * 4
    L.m2d_get_metrics.argtypes = [_ip, _ip] + [_vp] * 19
    L.m2d_get_radius.argtypes = [_ip, _ip, _ip] + [_vp] * 6
    for f in (L.m2d_get_real_centroids_xy, L.m2d_get_metrics, L.m2d_get_radius):
        f.restype = None
    L.m2d_norm_l1_5d.argtypes = [_ip, _ip, _vp, _vp, _vp, _dp]
    L.m2d_norm_l1_5d.restype = None
    L.m2d_intflow_time_step.argtypes = [_vp, _vp, _vp, _vp, C.POINTER(C.c_double), _vp]
    L.m2d_intflow_time_step.restype = C.c_int
    L.m2d_guess_prepare_many.argtypes = [_vp, C.c_int, _vp, _vp, _vp, C.c_int,
                                         C.POINTER(C.c_double), C.POINTER(C.c_double)]
    L.m2d_guess_prepare_many.restype = C.c_int
    L.m2d_get_average.argtypes = [_ip, _ip, _vp]
    L.m2d_get_average.restype = C.c_double
    L.m2d_version.argtypes = []
    L.m2d_version.restype = C.c_char_p
    _lib = L
    return L


def last_status() -> Status:
    st = Status()
    load().m2d_last_status(C.byref(st))
    return st


class SolverError(RuntimeError):
    def __init__(self, code, where=""):
        self.code = code
        super().__init__("%s: status %d (%s)" % (where, code, STATUS_NAMES.get(code, "?")))

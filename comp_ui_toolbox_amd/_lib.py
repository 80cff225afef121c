"""ctypes binding of libborn.so (include/born.h).

There is no fallback: if the library is missing or cannot be loaded, every
entry point raises `BornLibraryError`.
"""
from __future__ import annotations

import ctypes as C
import os
from pathlib import Path

_PKG = Path(__file__).resolve().parent
LIB_PATH = Path(os.environ.get("BORN_LIBRARY", _PKG / "libborn.so"))

BORN_OK = 0
STATUS_NAMES = {
    1: "NumberArguments", 2: "NoSymmetricGridsSetup", 3: "NoScatteringOptionsGPUActive",
    4: "NoComplexDoubles", 5: "NoOperatorBorn", 6: "NoNumericScalarMode",
    7: "NoValidDoubleMatrix", 8: "ConversionFailed", 9: "ErrorCUDA",
    10: "InvalidArgument", 11: "Unsupported", 12: "OutOfMemory",
}

PRECISIONS = {"fp32": 0, "split_bf16": 1, "split_fp16": 2}
FILTER_CODES = {"off": 0, "raised_cosine": 1, "logistic": 2, "boxcar": 3}

EXPORTED = (
    "born_plan_create_tables", "born_plan_create_geometry", "born_plan_destroy", "born_plan_size",
    "born_plan_set_precision", "born_forward", "born_adjoint", "born_forward_dev", "born_adjoint_dev",
    "born_plan_get_table", "born_plan_table_shape", "born_energy_rx", "born_energy_rx_dev",
    "born_time_signals", "born_plan_path", "born_plan_force_general", "born_plan_set_timing",
    "born_plan_get_timing", "born_last_error", "born_status_id",
    "born_batch_create", "born_batch_destroy", "born_batch_forward_dev", "born_batch_adjoint_dev",
    "born_batch_set_graph", "born_batch_autotune", "born_plan_autotune", "born_batch_set_timing",
    "born_batch_get_timing", "born_tgc_set", "born_tgc_apply", "born_tgc_apply_dev",
    "born_apply_tgc", "born_plan_set_correlation", "born_plan_kernels",
    "born_energy_rx_tgc", "born_energy_rx_tgc_dev", "born_debug_fail_allocation",
    "born_debug_live_allocations", "born_columns", "born_columns_dev",
    "born_plan_set_sparse_forward", "born_apply_dev_noalloc",
)


class BornLibraryError(RuntimeError):
    pass


class BornError(RuntimeError):
    """Failure of a library call; `identifier` is the reference's error ID
    (e.g. 'combined_quick_gpu:NoValidDoubleMatrix')."""

    def __init__(self, status: int, identifier: str, message: str):
        super().__init__(f"{identifier}: {message}")
        self.status = status
        self.identifier = identifier


class MixDesc(C.Structure):
    _fields_ = [("N_f", C.c_int32), ("indices_f_to_unique", C.POINTER(C.c_double)),
                ("N_active", C.c_int32), ("indices_active", C.POINTER(C.c_double)),
                ("prefactors", C.POINTER(C.c_double))]


class MeasDesc(C.Structure):
    _fields_ = [("N_f_unique", C.c_int32), ("indices_f_to_unique", C.POINTER(C.c_double)),
                ("p_incident", C.POINTER(C.c_double)), ("N_mix", C.c_int32),
                ("mixes", C.POINTER(MixDesc))]


class TablesDesc(C.Structure):
    _fields_ = [("N_dimensions", C.c_int32), ("N_points_axis", C.c_int32 * 3),
                ("N_elements_axis", C.c_int32 * 2), ("N_points", C.c_int32),
                ("N_elements", C.c_int32), ("N_f_unique", C.c_int32),
                ("h_ref", C.POINTER(C.c_double)), ("indices_grid_FOV_shift", C.POINTER(C.c_double)),
                ("N_measurements", C.c_int32), ("measurements", C.POINTER(MeasDesc)),
                ("device", C.c_int32), ("precision", C.c_int32)]


class GeometryDesc(C.Structure):
    _fields_ = [("N_dimensions", C.c_int32), ("N_points_axis", C.c_int32 * 3),
                ("delta_axis", C.c_double * 3), ("z0", C.c_double),
                ("N_elements_axis", C.c_int32 * 2), ("pitch_axis", C.c_double * 2),
                ("N_face_points_axis", C.c_int32 * 2), ("face_delta_axis", C.c_double * 2),
                ("face_weights", C.POINTER(C.c_double)), ("N_f_unique", C.c_int32),
                ("frequencies", C.POINTER(C.c_double)), ("wavenumbers", C.POINTER(C.c_double)),
                ("filter_rx_kind", C.c_int32), ("filter_tx_kind", C.c_int32),
                ("filter_rx_param", C.c_double), ("filter_tx_param", C.c_double),
                ("N_measurements", C.c_int32), ("measurements", C.POINTER(MeasDesc)),
                ("N_tx_active", C.POINTER(C.c_int32)),
                ("tx_indices_active", C.POINTER(C.POINTER(C.c_double))),
                ("v_d", C.POINTER(C.POINTER(C.c_double))),
                ("device", C.c_int32), ("precision", C.c_int32)]


_lib = None


def lib() -> C.CDLL:
    """Load libborn.so once; raise if it is not there."""
    global _lib
    if _lib is not None:
        return _lib
    if not LIB_PATH.exists():
        raise BornLibraryError(f"{LIB_PATH} is missing: build it with `python -m comp_ui_toolbox_amd.build`")
    try:
        L = C.CDLL(str(LIB_PATH))
    except OSError as e:
        raise BornLibraryError(f"cannot load {LIB_PATH}: {e}") from e
    vp = C.c_void_p
    pd = C.POINTER(C.c_double)
    L.born_plan_create_tables.argtypes = [C.POINTER(TablesDesc), C.POINTER(vp)]
    L.born_plan_create_geometry.argtypes = [C.POINTER(GeometryDesc), C.POINTER(vp)]
    L.born_plan_destroy.argtypes = [vp]
    L.born_plan_size.argtypes = [vp, C.POINTER(C.c_int64), C.POINTER(C.c_int64)]
    L.born_plan_set_precision.argtypes = [vp, C.c_int32]
    L.born_forward.argtypes = [vp, pd, C.c_int32, pd]
    L.born_adjoint.argtypes = [vp, pd, C.c_int32, pd]
    L.born_forward_dev.argtypes = [vp, vp, C.c_int32, vp, vp]
    L.born_adjoint_dev.argtypes = [vp, vp, C.c_int32, vp, vp]
    L.born_apply_dev_noalloc.argtypes = [vp, C.c_int32, vp, C.c_int32, vp, vp]
    L.born_plan_get_table.argtypes = [vp, C.c_int32, C.c_int32, vp, C.c_int64]
    L.born_plan_table_shape.argtypes = [vp, C.c_int32, C.c_int32, C.POINTER(C.c_int64), C.POINTER(C.c_int64)]
    L.born_energy_rx.argtypes = [vp, C.c_int32, pd]
    L.born_energy_rx_dev.argtypes = [vp, C.c_int32, vp, vp]
    L.born_time_signals.argtypes = [vp, pd, C.c_double, C.c_double, vp, C.c_int32, vp, C.c_int64,
                                    C.POINTER(C.c_int32), vp]
    L.born_plan_set_correlation.argtypes = [vp, C.c_int32]
    L.born_plan_kernels.argtypes = [vp, C.POINTER(C.c_int32)]
    L.born_tgc_set.argtypes = [vp, C.POINTER(C.c_int32), pd]
    L.born_tgc_apply.argtypes = [vp, C.c_int32, pd, C.c_int32, pd]
    L.born_apply_tgc.argtypes = [vp, C.c_int32, pd, C.c_int32, pd]
    L.born_tgc_apply_dev.argtypes = [vp, C.c_int32, vp, vp, C.c_int32, vp]
    L.born_energy_rx_tgc.argtypes = [vp, C.c_int32, pd]
    L.born_energy_rx_tgc_dev.argtypes = [vp, C.c_int32, vp, vp]
    L.born_debug_fail_allocation.argtypes = [C.c_int64]
    L.born_columns.argtypes = [vp, pd, C.c_int32, pd]
    L.born_plan_set_sparse_forward.argtypes = [vp, C.c_int32]
    L.born_columns_dev.argtypes = [vp, pd, C.c_int32, vp, vp]
    L.born_debug_live_allocations.argtypes = []
    L.born_plan_path.argtypes = [vp]
    L.born_plan_force_general.argtypes = [vp, C.c_int32]
    L.born_plan_set_timing.argtypes = [vp, C.c_int32]
    L.born_plan_get_timing.argtypes = [vp, C.POINTER(C.c_double), C.POINTER(C.c_int64)]
    L.born_batch_create.argtypes = [C.POINTER(vp), C.c_int32, C.POINTER(vp)]
    L.born_batch_destroy.argtypes = [vp]
    L.born_batch_forward_dev.argtypes = [vp, C.POINTER(vp), C.POINTER(vp), vp]
    L.born_batch_adjoint_dev.argtypes = [vp, C.POINTER(vp), C.POINTER(vp), vp]
    L.born_batch_set_graph.argtypes = [vp, C.c_int32]
    L.born_batch_autotune.argtypes = [vp, vp, C.POINTER(C.c_double), C.POINTER(C.c_double)]
    L.born_plan_autotune.argtypes = [vp, vp, C.POINTER(C.c_double), C.POINTER(C.c_double)]
    L.born_batch_set_timing.argtypes = [vp, C.c_int32]
    L.born_batch_get_timing.argtypes = [vp, C.POINTER(C.c_double), C.POINTER(C.c_int64)]
    L.born_last_error.restype = C.c_char_p
    L.born_status_id.restype = C.c_char_p
    L.born_status_id.argtypes = [C.c_int]
    for name in EXPORTED:
        if name not in ("born_last_error", "born_status_id", "born_plan_path", "born_debug_live_allocations"):
            getattr(L, name).restype = C.c_int
    L.born_plan_path.restype = C.c_int
    L.born_debug_live_allocations.restype = C.c_int64
    _lib = L
    return L


def check(status: int) -> None:
    if status != BORN_OK:
        L = lib()
        ident = L.born_status_id(status).decode()
        msg = L.born_last_error().decode()
        raise BornError(status, ident, msg)


def dptr(a):
    """POINTER(c_double) of a contiguous float64 numpy array (or None)."""
    if a is None:
        return None
    return a.ctypes.data_as(C.POINTER(C.c_double))

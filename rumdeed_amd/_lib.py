"""ctypes binding of librumdeed.so (the C ABI declared in include/rumdeed.h).

There is no fallback: if the library is missing or a call fails, an
exception is raised with the library's own error message.
"""
from __future__ import annotations

import ctypes
import os
from ctypes import POINTER, c_char_p, c_double, c_int32, c_int64, c_uint64, c_void_p

import numpy as np

PKG = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(PKG, "librumdeed.so")

RD_OK = 0
RD_ERR_ARG, RD_ERR_HIP, RD_ERR_CAPACITY, RD_ERR_STATE = 1, 2, 3, 4
RD_GEOM_PLANAR = 1
RD_GEOM_TIP = 2
RD_PREC_FP64 = 0
RD_PREC_MIXED = 1
RD_SPECIES_ELEC = 1
RD_SPECIES_ION = 2


class RumdeedError(RuntimeError):
    def __init__(self, code: int, msg: str):
        super().__init__(f"librumdeed error {code}: {msg}")
        self.code = code


RD_EMIT_NONE = 0
RD_EMIT_TIP_FE = 3
RD_EMIT_PLANAR_GTF = 9
RD_EMIT_PLANAR_FE = 10


class Geometry(ctypes.Structure):
    """rd_geometry (include/rumdeed.h)."""

    _fields_ = [("kind", c_int32), ("image_charge", c_int32), ("n_ic_max", c_int32),
                ("reserved", c_int32), ("V", c_double), ("d", c_double),
                ("d_tip", c_double), ("R_base", c_double), ("h_tip", c_double),
                ("box_top", c_double)]


_dp = POINTER(c_double)
_ip = POINTER(c_int32)


class Emitter(ctypes.Structure):
    """rd_emitter (include/rumdeed.h)."""

    _fields_ = [("mode", c_int32), ("delay", c_int32), ("x0", c_double), ("y0", c_double),
                ("lx", c_double), ("ly", c_double), ("T", c_double), ("w_tip", c_double),
                ("wf_nx", c_int32), ("wf_ny", c_int32), ("wf_table", _dp),
                ("quad_n", c_int32), ("ndim", c_int32), ("quad_levels", c_int32),
                ("reserved", c_int32)]


class StepRecord(ctypes.Structure):
    """rd_step_record (include/rumdeed.h)."""

    _fields_ = [("step", c_int32), ("n", c_int32), ("emitted", c_int32), ("n_round", c_int32),
                ("absorbed", c_int32), ("absorbed_top", c_int32), ("absorbed_bot", c_int32),
                ("dropped", c_int32), ("start_rounds", c_int32), ("supply_level", c_int32),
                ("supply_cells", c_int32), ("supply_fail", c_int32),
                ("n_sup", c_double), ("ramo_current", c_double), ("mh_std", c_double),
                ("a_rate", c_double), ("df_avg", c_double), ("f_avg", c_double * 3),
                ("ramo", c_double * 3), ("avg_elec_vel", c_double * 3), ("supply_err", c_double)]

    def as_dict(self):
        d = {}
        for k, _ in self._fields_:
            v = getattr(self, k)
            d[k] = list(v) if k in ("f_avg", "ramo", "avg_elec_vel") else v
        return d

# rd_emit_record / rd_absorb_record (include/rumdeed.h)
import numpy as _np  # noqa: E402

EMIT_RECORD = _np.dtype([("x", "<f8"), ("y", "<f8"), ("z", "<f8"), ("emitter", "<i4"),
                         ("section", "<i4"), ("id", "<i4"), ("species", "<i4")])
ABSORB_RECORD = _np.dtype([("x", "<f8"), ("y", "<f8"), ("z", "<f8"), ("vx", "<f8"),
                           ("vy", "<f8"), ("vz", "<f8"), ("emitter", "<i4"), ("section", "<i4"),
                           ("id", "<i4"), ("where", "<i4")])
PLANE_RECORD = _np.dtype([("x", "<f8"), ("y", "<f8"), ("vx", "<f8"), ("vy", "<f8"),
                          ("vz", "<f8"), ("emitter", "<i4"), ("section", "<i4"), ("id", "<i4"),
                          ("plane", "<i4")])
MAX_PLANES = 10

# name -> (restype, argtypes)
_SIGS = {
    "rd_version": (c_char_p, []),
    "rd_last_error": (c_char_p, []),
    "rd_device_count": (c_int32, [_ip]),
    "rd_ctx_create": (c_int32, [c_int32, c_int64, POINTER(c_void_p)]),
    "rd_ctx_destroy": (c_int32, [c_void_p]),
    "rd_set_geometry": (c_int32, [c_void_p, POINTER(Geometry)]),
    "rd_set_time_step": (c_int32, [c_void_p, c_double]),
    "rd_set_two_time_step": (c_int32, [c_void_p, c_int32]),
    "rd_put_particles": (c_int32, [c_void_p, c_int32, _dp, _dp, _dp, _dp, _ip]),
    "rd_particle_count": (c_int32, [c_void_p, _ip]),
    "rd_get_particles": (c_int32, [c_void_p, _dp, _dp, _dp, _dp, _ip]),
    "rd_accel": (c_int32, [c_void_p, c_int32]),
    "rd_get_accel": (c_int32, [c_void_p, _dp]),
    "rd_field_batch": (c_int32, [c_void_p, c_int32, _dp, _dp, c_int32]),
    "rd_field_batch_static": (c_int32, [c_void_p, c_int32, _dp, _dp, c_int32]),
    "rd_set_force_options": (c_int32, [c_void_p, c_int32]),
    "rd_set_partial_budget": (c_int32, [c_void_p, c_int64]),
    "rd_work_bytes": (c_int32, [c_void_p, POINTER(c_int64)]),
    "rd_field_grid": (c_int32, [c_void_p, c_double, c_double, c_double, c_double, c_int32,
                                c_int32, c_double, c_int32, _dp]),
    "rd_set_emitter": (c_int32, [c_void_p, POINTER(Emitter)]),
    "rd_set_seed": (c_int32, [c_void_p, c_uint64, c_uint64]),
    "rd_add_particles": (c_int32, [c_void_p, c_int32, _dp, _dp, _ip, c_int32, c_int32, _ip]),
    "rd_update_position": (c_int32, [c_void_p, c_int32, c_int32, POINTER(StepRecord)]),
    "rd_remove_particles": (c_int32, [c_void_p, c_int32, POINTER(StepRecord)]),
    "rd_do_emission": (c_int32, [c_void_p, c_int32, c_int32, POINTER(StepRecord)]),
    "rd_run": (c_int32, [c_void_p, c_int32, c_int32, POINTER(StepRecord)]),
    "rd_get_state": (c_int32, [c_void_p, _dp, _dp, _dp, _dp, _dp, _dp, _ip]),
    "rd_get_life_time": (c_int32, [c_void_p, _ip]),
    "rd_pool_create": (c_int32, [c_int32, c_int64, c_int32, POINTER(c_void_p)]),
    "rd_slot_footprint": (c_int32, [c_int64, POINTER(c_int64)]),
    "rd_slot_open": (c_int32, [c_void_p, c_int64, _ip]),
    "rd_slot_close": (c_int32, [c_void_p, c_int32]),
    "rd_slot_select": (c_int32, [c_void_p, c_int32]),
    "rd_slot_step": (c_int32, [c_void_p, c_int32, _ip]),
    "rd_pool_step": (c_int32, [c_void_p, c_int32, POINTER(StepRecord)]),
    "rd_time_accel": (c_int32, [c_void_p, c_int32, c_int32, _dp, _dp]),
    "rd_time_field_grid": (c_int32, [c_void_p, c_double, c_double, c_double, c_double,
                                     c_int32, c_int32, c_double, c_int32, c_int32, _dp, _dp]),
    "rd_time_copy": (c_int32, [c_void_p, c_int64, c_int32, _dp]),
    "rd_set_graphs": (c_int32, [c_void_p, c_int32]),
    "rd_set_jump_pairing": (c_int32, [c_void_p, c_int64]),
    "rd_set_solo_jumps": (c_int32, [c_void_p, c_int32]),
    "rd_set_jump_wait": (c_int32, [c_void_p, c_int64]),
    "rd_jump_repeats": (c_int32, [c_void_p, POINTER(c_int64)]),
    "rd_set_logs": (c_int32, [c_void_p, c_int32]),
    "rd_get_logs": (c_int32, [c_void_p, c_int32, c_void_p, _ip, c_int32, c_void_p, _ip]),
    "rd_set_planes": (c_int32, [c_void_p, c_int32, c_void_p]),
    "rd_get_plane_logs": (c_int32, [c_void_p, c_int32, c_void_p, _ip]),
}

_lib = None


def lib() -> ctypes.CDLL:
    """Load librumdeed.so (raises if it has not been built)."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: build it with `python -m rumdeed_amd.build` "
                "(the HIP library is required; there is no CPU fallback)")
        L = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in _SIGS.items():
            f = getattr(L, name)
            f.restype = res
            f.argtypes = args
        _lib = L
    return _lib


def exported_symbols():
    return list(_SIGS)


def check(code: int) -> None:
    if code != RD_OK:
        msg = lib().rd_last_error()
        raise RumdeedError(code, msg.decode() if msg else "")


def dptr(a):
    if a is None:
        return None
    return a.ctypes.data_as(_dp)


def iptr(a):
    if a is None:
        return None
    return a.ctypes.data_as(_ip)


def f64(a, shape=None):
    a = np.ascontiguousarray(a, dtype=np.float64)
    if shape is not None:
        a = a.reshape(shape)
    return a

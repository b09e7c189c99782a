"""ctypes binding of libvxmix.so (the C ABI declared in include/vxmix.h).

Loading fails loudly when the library has not been built: there is no CPU
fallback for any entry point.
"""
from __future__ import annotations

import ctypes
import threading
from pathlib import Path

LIB_PATH = Path(__file__).resolve().parent / "libvxmix.so"

VX_OK = 0
VX_ERR_INVALID_ARGUMENT = 1
VX_ERR_UNSUPPORTED = 2
VX_ERR_LAUNCH = 3
VX_LEVELS_INNER = 0
VX_LEVELS_OUTER = 1

c_void_p = ctypes.c_void_p
c_i32 = ctypes.c_int32
c_i64 = ctypes.c_int64
c_f64 = ctypes.c_double


class VxGrid(ctypes.Structure):
    _fields_ = [
        ("kbot", c_void_p),
        ("dxt", c_void_p), ("dxu", c_void_p), ("dyt", c_void_p), ("dyu", c_void_p),
        ("cost", c_void_p), ("cosu", c_void_p), ("dzt", c_void_p), ("dzw", c_void_p),
        ("nx", c_i64), ("ny", c_i64), ("nz", c_i32), ("time_layout", c_i32),
    ]


class VxTdmaSystem(ctypes.Structure):
    _fields_ = [
        ("a", c_void_p), ("b", c_void_p), ("c", c_void_p), ("d", c_void_p),
        ("b_edge", c_void_p), ("d_edge", c_void_p),
        ("kbot", c_void_p), ("kbot_sx", c_i64), ("kbot_sy", c_i64),
        ("x", c_void_p),
        ("nx", c_i64), ("ny", c_i64), ("nz", c_i32), ("_pad", c_i32), ("sx", c_i64), ("sy", c_i64),
    ]


class VxIsoParams(ctypes.Structure):
    _fields_ = [(name, c_f64) for name in (
        "drhodT", "drhodS", "K_iso_steep", "iso_slopec", "iso_dslope", "dt_tracer", "grav", "rho_0")]


class VxTerms(ctypes.Structure):
    _fields_ = [("arr", c_void_p * 12), ("sign", c_f64 * 12), ("n", c_i32), ("_pad", c_i32)]


class VxTkeParams(ctypes.Structure):
    _fields_ = [("dt_mom", c_f64), ("alpha_tke", c_f64), ("c_eps", c_f64), ("K_h_tke", c_f64),
                ("hor_diffusion", c_i32), ("_pad", c_i32)]


class VxEkeParams(ctypes.Structure):
    _fields_ = [("dt_tracer", c_f64), ("alpha_eke", c_f64), ("eke_c_eps", c_f64)]


class VxIdemixParams(ctypes.Structure):
    _fields_ = [("dt_tracer", c_f64), ("tau_v", c_f64), ("tau_h", c_f64), ("eke_diss_surfbot_frac", c_f64),
                ("hor_diffusion", c_i32), ("eke_diss_mode", c_i32)]


# name -> (restype, argtypes)
_SIGNATURES = {
    "vx_version": (ctypes.c_char_p, []),
    "vx_max_nz": (c_i32, []),
    "vx_last_error": (ctypes.c_char_p, []),
    "vx_tdma_f64": (ctypes.c_int, [c_void_p] + [c_void_p] * 6 + [c_void_p, c_i64, c_i64, c_void_p,
                                                                c_i64, c_i64, c_i32, c_i64, c_i64]),
    "vx_tdma_mixed": (ctypes.c_int, [c_void_p] + [c_void_p] * 6 + [c_void_p, c_i64, c_i64, c_void_p,
                                                                  c_i64, c_i64, c_i32, c_i64, c_i64, c_i32]),
    "vx_tdma_adjoint_f64": (ctypes.c_int, [c_void_p] + [c_void_p] * 5 + [c_void_p, c_i64, c_i64]
                            + [c_void_p] * 8 + [c_i64, c_i64, c_i32, c_i64, c_i64]),
    "vx_tdma_plan_create": (ctypes.c_int, [ctypes.POINTER(VxTdmaSystem), c_i32, c_i32,
                                           ctypes.POINTER(c_void_p)]),
    "vx_tdma_plan_run": (ctypes.c_int, [c_void_p, c_void_p]),
    "vx_tdma_plan_tune": (ctypes.c_int, [c_void_p, c_void_p]),
    "vx_tdma_plan_graph_launch": (ctypes.c_int, [c_void_p, c_void_p]),
    "vx_tdma_plan_info": (ctypes.c_int, [c_void_p, ctypes.POINTER(c_i32), ctypes.POINTER(c_i64),
                                         ctypes.POINTER(c_i32), c_i32]),
    "vx_tdma_plan_destroy": (None, [c_void_p]),
    "vx_iso_pre_f64": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid), ctypes.POINTER(VxIsoParams),
                                      c_void_p, c_void_p, c_i32, c_void_p] + [c_void_p] * 7),
    "vx_iso_workspace_bytes": (c_i64, [ctypes.POINTER(VxGrid), c_i32]),
    "vx_iso_diffusion_f64": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid), ctypes.POINTER(VxIsoParams),
                                            c_void_p, c_i32, c_i32, c_void_p] + [c_void_p] * 7
                             + [c_void_p, c_void_p, c_void_p, c_void_p]),
    "vx_iso_diffusion_ts_f64": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid), ctypes.POINTER(VxIsoParams),
                                               c_void_p, c_void_p, c_i32, c_i32, c_void_p] + [c_void_p] * 7
                                + [c_void_p] * 6),
    "vx_iso_pre_diffusion_ts_f64": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid), ctypes.POINTER(VxIsoParams),
                                                   c_void_p, c_void_p, c_i32, c_i32, c_void_p] + [c_void_p] * 7
                                    + [c_void_p] * 6),
    "vx_iso_pre_diffusion_ts_workspace_bytes": (c_i64, [ctypes.POINTER(VxGrid)]),
    "vx_iso_pre_diffusion_ts_f64_noalloc": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid),
                                                           ctypes.POINTER(VxIsoParams), c_void_p, c_void_p, c_i32,
                                                           c_i32, c_void_p] + [c_void_p] * 7 + [c_void_p] * 5),
    "vx_iso_skew_diffusion_f64": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid), ctypes.POINTER(VxIsoParams),
                                                 c_void_p, c_i32, c_i32, c_void_p] + [c_void_p] * 6
                                  + [c_void_p, c_void_p, c_void_p, c_void_p]),
    "vx_vertmix_tempsalt_f64": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid), c_f64, c_void_p, c_void_p, c_i32,
                                               c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_i32]),
    "vx_implicit_vert_friction_f64": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid), c_f64, c_void_p, c_void_p,
                                                     c_i32, c_i32] + [c_void_p] * 6),
    "vx_integrate_tke_f64": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid), ctypes.POINTER(VxTkeParams), c_void_p,
                                            c_i32, c_i32] + [c_void_p] * 4 + [ctypes.POINTER(VxTerms), c_void_p,
                                                                              c_void_p]),
    "vx_integrate_eke_f64": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid), ctypes.POINTER(VxEkeParams), c_void_p,
                                            c_i32, c_i32] + [c_void_p] * 4 + [ctypes.POINTER(VxTerms), c_void_p,
                                                                              c_void_p]),
    "vx_integrate_idemix_f64": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid), ctypes.POINTER(VxIdemixParams),
                                               c_void_p, c_i32, c_i32] + [c_void_p] * 5
                                + [ctypes.POINTER(VxTerms), ctypes.POINTER(VxTerms), c_void_p]),
    "vx_enforce_boundaries_f64": (ctypes.c_int, [c_void_p, c_void_p, c_i64, c_i64, c_i64, c_i64, c_i32]),
    "vx_kbot_from_edge_mask": (ctypes.c_int, [c_void_p, c_void_p, c_i64, c_i32, c_void_p]),
    "vx_iso_diag_streamfunction_f64": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid)] + [c_void_p] * 5),
    "vx_iso_adjoint_workspace_bytes": (c_i64, [ctypes.POINTER(VxGrid)]),
    "vx_iso_diffusion_adjoint_f64": (ctypes.c_int, [c_void_p, ctypes.POINTER(VxGrid),
                                                    ctypes.POINTER(VxIsoParams), c_void_p, c_i32]
                                     + [c_void_p] * 8 + [c_void_p] * 4 + [c_void_p]),
}

_lock = threading.Lock()
_lib = None


def exported_symbols():
    return tuple(_SIGNATURES)


def lib():
    """The loaded library (raises RuntimeError if it has not been built)."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is None:
            if not LIB_PATH.exists():
                raise RuntimeError(
                    f"{LIB_PATH} is missing: build it with `python -c 'import __graft_entry__ as g; g.build()'` "
                    "or `python veros_amd/build.py`; there is no CPU fallback")
            L = ctypes.CDLL(str(LIB_PATH))
            for name, (res, args) in _SIGNATURES.items():
                fn = getattr(L, name)
                fn.restype = res
                fn.argtypes = args
            _lib = L
    return _lib


def check(rc: int, what: str):
    """Raise the exception class the reference raises for the same condition."""
    if rc == VX_OK:
        return
    msg = lib().vx_last_error().decode(errors="replace")
    if rc == VX_ERR_INVALID_ARGUMENT:
        raise ValueError(f"{what}: {msg}")
    if rc == VX_ERR_UNSUPPORTED:
        raise NotImplementedError(f"{what}: {msg}")
    raise RuntimeError(f"{what}: {msg}")


def max_nz() -> int:
    return int(lib().vx_max_nz())


def version() -> str:
    return lib().vx_version().decode()

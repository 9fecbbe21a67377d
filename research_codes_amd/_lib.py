"""ctypes binding of libsphk.so (include/sphk.h, sphk_step.h, sphk_tree.h, sphk_dtree.h).

The library is built in-tree by research_codes_amd.build.  Loading fails
loudly when it is missing: there is no CPU fallback for the product path.
"""
from __future__ import annotations

import ctypes as C
from pathlib import Path

PKG = Path(__file__).resolve().parent
LIB_PATH = PKG / "libsphk.so"

_P = C.c_void_p
_I32P = C.POINTER(C.c_int32)
_DP = C.POINTER(C.c_double)

SPHK_FP64 = 0
SPHK_MIXED = 1
ERRORS = {0: "SPHK_OK", -1: "SPHK_E_ARG", -2: "SPHK_E_CAPACITY", -3: "SPHK_E_DEVICE",
          -4: "SPHK_E_STATE", -5: "SPHK_E_NONFINITE"}


class SphkError(RuntimeError):
    def __init__(self, code: int, where: str, msg: str):
        super().__init__(f"{where}: {ERRORS.get(code, code)}: {msg}")
        self.code = code


class Params(C.Structure):
    _fields_ = [("eta", C.c_double), ("ksrh", C.c_double), ("hmax", C.c_double),
                ("uniform_softening", C.c_int), ("list_cap", C.c_int), ("persistent", C.c_int),
                ("pinned_src", C.c_int)]


DENS_SRC = ("id", "m", "x", "y", "z", "vx", "vy", "vz", "ksr", "rs")
DENS_OUT = ("dens", "divv", "rotv", "grdh", "ksr", "np", "itr")
HYDRO_SRC = ("id", "m", "x", "y", "z", "vx", "vy", "vz", "hinv", "pres", "presc", "bswt",
             "dens", "vsnd", "alph", "alphu", "thrm", "eta")
HYDRO_OUT = ("ax", "ay", "az", "gx", "gy", "gz", "udot", "vsmx", "diffu")
HYDRO_GRAD = ("x", "y", "z", "vx", "vy", "vz", "hinv", "pres", "presc", "bswt", "dens", "vsnd", "alph",
              "alphu", "thrm", "eta")
DENS_COT = ("dens", "ksr", "divv", "rotv", "grdh")
DENS_GRAD = ("x", "y", "z", "vx", "vy", "vz", "ksr")
GRAV_SRC = ("m", "x", "y", "z", "eps2")
GRAV_OUT = ("ax", "ay", "az", "pot", "eta")


def _struct(name, fields):
    return type(name, (C.Structure,), {"_fields_": [(f, _P) for f in fields]})


DensSrc = _struct("DensSrc", DENS_SRC)
DensOut = _struct("DensOut", DENS_OUT)
HydroSrc = _struct("HydroSrc", HYDRO_SRC)
HydroOut = _struct("HydroOut", HYDRO_OUT)
HydroGrad = _struct("HydroGrad", HYDRO_GRAD)
DensCot = _struct("DensCot", DENS_COT)
DensGrad = _struct("DensGrad", DENS_GRAD)
GravSrc = _struct("GravSrc", GRAV_SRC)
GravOut = _struct("GravOut", GRAV_OUT)

STATE_FIELDS = ("m", "x", "y", "z", "vx", "vy", "vz", "ax", "ay", "az", "vx2", "vy2", "vz2",
                "uene", "uene2", "udot", "alph", "alph2", "adot", "alphu", "alphu2", "adotu",
                "diffu", "ksr", "dens", "pres", "vsnd", "divv", "rotv", "bswt", "grdh", "vsmx",
                "pot", "eta", "achx", "achy", "achz", "g1x", "g1y", "g1z", "g2x", "g2y", "g2z")
State = _struct("State", STATE_FIELDS)


class Phys(C.Structure):
    _fields_ = [(n, C.c_double) for n in ("ninv", "ksrh", "G", "alpha_max", "alpha_min",
                                          "alphu_max", "alphu_min", "eps_u", "c_dt", "dt_max",
                                          "eps_const")]


# name -> (restype, argtypes); every symbol declared in include/*.h
SIGNATURES = {
    # sphk.h
    "sphk_init": (C.c_int, [C.c_int, C.POINTER(_P)]),
    "sphk_finalize": (C.c_int, [_P]),
    "sphk_set_params": (C.c_int, [_P, C.POINTER(Params)]),
    "sphk_get_params": (C.c_int, [_P, C.POINTER(Params)]),
    "sphk_last_error": (C.c_char_p, []),
    "sphk_device": (C.c_int, [_P]),
    "sphk_stream": (_P, [_P]),
    "sphk_synchronize": (C.c_int, [_P]),
    "sphk_density_dev": (C.c_int, [_P, C.c_int, _P, _P, _P, DensSrc, DensSrc, DensOut, C.c_int, _P]),
    "sphk_hydro_dev": (C.c_int, [_P, C.c_int, _P, _P, _P, HydroSrc, HydroSrc, HydroOut, C.c_int, _P]),
    "sphk_gravity_dev": (C.c_int, [_P, C.c_int, _P, _P, _P, GravSrc, _P, _P, GravSrc, GravSrc,
                                   GravOut, C.c_int, _P]),
    "sphk_density_dev_n": (C.c_int, [_P, C.c_int, C.c_int64, _P, _P, _P, DensSrc, DensSrc, DensOut, C.c_int, _P]),
    "sphk_hydro_dev_n": (C.c_int, [_P, C.c_int, C.c_int64, _P, _P, _P, HydroSrc, HydroSrc, HydroOut, C.c_int, _P]),
    "sphk_gravity_dev_n": (C.c_int, [_P, C.c_int, C.c_int64, _P, _P, _P, GravSrc, _P, _P, GravSrc, GravSrc,
                                   GravOut, C.c_int, _P]),
    "sphk_density_dispatch": (C.c_int, [_P, C.c_int, C.c_int, _P, _P, DensSrc, DensSrc, C.c_int]),
    "sphk_density_retrieve": (C.c_int, [_P, C.c_int, C.c_int, _P, DensOut]),
    "sphk_hydro_dispatch": (C.c_int, [_P, C.c_int, C.c_int, _P, _P, HydroSrc, HydroSrc, C.c_int]),
    "sphk_hydro_retrieve": (C.c_int, [_P, C.c_int, C.c_int, _P, HydroOut]),
    "sphk_gravity_dispatch": (C.c_int, [_P, C.c_int, C.c_int, _P, _P, _P, GravSrc, GravSrc,
                                        GravSrc, C.c_int]),
    "sphk_gravity_retrieve": (C.c_int, [_P, C.c_int, C.c_int, _P, GravOut]),
    "sphk_timing": (C.c_int, [_P, C.c_int]),
    "sphk_kernel_time": (C.c_int, [_P, C.c_int, _DP, C.POINTER(C.c_int)]),
    "sphk_reset_kernel_time": (C.c_int, [_P]),
    # sphk_step.h
    "sphk_eos_balsara_dev": (C.c_int, [_P, C.c_int, State, Phys, _P]),
    "sphk_softening_dev": (C.c_int, [_P, C.c_int, _P, C.c_double, C.c_double, _P, _P]),
    "sphk_density_commit_dev": (C.c_int, [_P, C.c_int, State, DensOut, _P, _P, _P, C.c_double, C.c_int, _P,
                                          _P]),
    "sphk_gravity_writeback_dev": (C.c_int, [_P, C.c_int, State, Phys, GravOut, _P]),
    "sphk_hydro_prep_dev": (C.c_int, [_P, C.c_int, State, _P, _P, _P, _P, _P]),
    "sphk_hydro_writeback_dev": (C.c_int, [_P, C.c_int, State, Phys, HydroOut, _P]),
    "sphk_predict_dev": (C.c_int, [_P, C.c_int, State, C.c_double, _P]),
    "sphk_correct_dev": (C.c_int, [_P, C.c_int, State, C.c_double, _P]),
    "sphk_diagnostics": (C.c_int, [_P, C.c_int, State, Phys, _DP, _P]),
    "sphk_diagnostics_static": (C.c_int, [_P, C.c_int, State, Phys, _P, _P]),
    # sphk_tree.h
    "sphk_morton_order": (C.c_int, [C.c_int, _P, _P, _P, _P]),
    "sphk_tree_build": (C.c_int, [C.c_int, _P, _P, _P, _P, _P, C.c_int, C.c_int, C.POINTER(_P)]),
    "sphk_tree_free": (None, [_P]),
    "sphk_tree_group_fixed": (C.c_int, [_P, C.c_int]),
    "sphk_tree_n_walk": (C.c_int, [_P]),
    "sphk_tree_n_node": (C.c_int, [_P]),
    "sphk_tree_i_off": (_I32P, [_P]),
    "sphk_tree_list_gather": (C.c_int, [_P, _P]),
    "sphk_tree_list_symmetry": (C.c_int, [_P, _P]),
    "sphk_tree_list_long": (C.c_int, [_P, C.c_double]),
    "sphk_tree_list": (C.c_int, [_P, C.c_int, C.POINTER(_I32P), C.POINTER(_I32P),
                                 C.POINTER(_I32P), C.POINTER(_I32P)]),
    "sphk_tree_moments": (C.c_int, [_P, C.POINTER(_DP), C.POINTER(_DP), C.POINTER(_DP),
                                    C.POINTER(_DP), C.POINTER(_DP)]),
}

SIGNATURES.update({
    # sphk_dtree.h (all array arguments are device pointers)
    "sphk_morton_order_dev": (C.c_int, [C.c_int, _P, _P, _P, _P, _P]),
    "sphk_dtree_build": (C.c_int, [C.c_int, _P, _P, _P, _P, _P, C.c_int, C.c_int, _P, C.POINTER(_P)]),
    "sphk_dtree_rebuild": (C.c_int, [_P, C.c_int, _P, _P, _P, _P, _P, C.c_int, C.c_int, _P]),
    "sphk_dtree_detach": (C.c_int, [_P]),
    "sphk_dtree_free": (None, [_P]),
    "sphk_dtree_n_walk": (C.c_int, [_P]),
    "sphk_dtree_n_node": (C.c_int, [_P]),
    "sphk_dtree_i_off": (_P, [_P]),
    "sphk_dtree_list_gather": (C.c_int, [_P, _P]),
    "sphk_dtree_list_symmetry": (C.c_int, [_P, _P]),
    "sphk_dtree_list_long": (C.c_int, [_P, C.c_double]),
    "sphk_dtree_list": (C.c_int, [_P, C.c_int, C.POINTER(_P), C.POINTER(_P), C.POINTER(_P),
                                  C.POINTER(_P), C.POINTER(C.c_int64), C.POINTER(C.c_int64)]),
    "sphk_dtree_list_size": (C.c_int, [_P, C.c_int, C.POINTER(C.c_int64), C.POINTER(C.c_int64)]),
    "sphk_dtree_list_copy": (C.c_int, [_P, C.c_int, _P, _P, _P, _P]),
    "sphk_dtree_moments": (C.c_int, [_P] + [C.POINTER(_P)] * 5),
    "sphk_dtree_nodes": (C.c_int, [_P] + [C.POINTER(_P)] * 6),
    "sphk_copy_dev": (C.c_int, [_P, _P, C.c_size_t, _P]),
    "sphk_permute_work_bytes": (C.c_size_t, [C.c_int, C.c_int, C.POINTER(C.c_int)]),
    "sphk_permute_dev": (C.c_int, [C.c_int, _P, C.c_int, C.POINTER(_P), C.POINTER(C.c_int), _P, C.c_size_t,
                                   _P]),
    "sphk_equal_dev": (C.c_int, [C.c_int, C.c_int, C.POINTER(_P), C.POINTER(_P), _P, _P]),
    "sphk_unbound_mass_dev": (C.c_int, [_P, C.c_int, State, _P, C.c_int, C.c_double, _DP, _P]),
    # sphk_adjoint.h
    "sphk_gravity_vjp_dev": (C.c_int, [_P, C.c_int, _P, _P, _P, GravSrc, _P, _P, GravSrc, GravSrc, C.c_double]
                             + [_P] * 11 + [_P]),
    "sphk_gravity_vjp_packed_dev": (C.c_int, [_P, C.c_int, _P, _P, _P, GravSrc, _P, _P, GravSrc, GravSrc, C.c_double]
                                    + [_P] * 7 + [_P]),
    "sphk_dtree_spread_dev": (C.c_int, [_P] + [_P] * 7),
    "sphk_hydro_vjp_dev": (C.c_int, [_P, C.c_int, _P, _P, _P, HydroSrc, HydroOut, HydroGrad, _P]),
    "sphk_density_vjp_dev": (C.c_int, [_P, C.c_int, _P, _P, _P, DensSrc, DensCot, DensGrad, _P]),
})

_lib = None


def lib() -> C.CDLL:
    """Load libsphk.so (raises if it has not been built)."""
    global _lib
    if _lib is None:
        if not LIB_PATH.exists():
            raise ImportError(f"{LIB_PATH} is missing: run `python -m research_codes_amd.build` "
                              "(the HIP library is required; there is no CPU fallback)")
        L = C.CDLL(str(LIB_PATH))
        for name, (res, args) in SIGNATURES.items():
            f = getattr(L, name)
            f.restype = res
            f.argtypes = args
        _lib = L
    return _lib


def raw_stream() -> int:
    """torch's current stream on the current device as a hipStream_t (the
    address alone: no Stream object is made, 0.6 against 2.7 us a call)."""
    import torch
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())


def check(rc: int, where: str) -> None:
    if rc != 0:
        raise SphkError(rc, where, lib().sphk_last_error().decode(errors="replace"))

"""ctypes binding of ``libli_sparse_attn.so`` (the C ABI in include/li_sparse_attn.h).

The library is loaded once, from this package directory.  There is no
fallback: if it is missing or does not export the ABI, importing this module
raises ``ImportError`` naming the build command.

torch is imported first so that the HIP runtime torch ships with is already
mapped when the library is loaded: the library's ``libamdhip64.so.7``
dependency then resolves (by SONAME) to that same runtime, and torch's
streams and device pointers are valid in the library's launches.  Loading
the library first would map a second, independent HIP runtime.
"""
import ctypes
import os

import torch  # noqa: F401  (must precede the CDLL below)

LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libli_sparse_attn.so")
ABI_VERSION = 12

LI_OK = 0
LI_ERR_INVALID_ARG = -1
LI_ERR_SHAPE = -2
LI_ERR_K_LEN = -3
LI_ERR_INDEX_RANGE = -4
LI_ERR_UNSUPPORTED = -5
LI_ERR_LAUNCH = -6
LI_ERR_TOO_LARGE = -7

LI_DTYPE_BF16 = 0
LI_DTYPE_F16 = 1

LI_METRIC_COSINE = 0
LI_METRIC_SCALED_DOT = 1
LI_METRIC_DOT = 2

LI_BUDGET_HISTORY = 0
LI_BUDGET_TOTAL = 1

LI_BSA_BALANCE = 1
LI_BSA_SORTED = 2

_i64p = ctypes.POINTER(ctypes.c_int64)
_i32p = ctypes.POINTER(ctypes.c_int32)
_vp = ctypes.c_void_p
_i32 = ctypes.c_int32
_i64 = ctypes.c_int64


class TileGeom(ctypes.Structure):
    _fields_ = [("T", _i32), ("H", _i32), ("W", _i32), ("tt", _i32), ("th", _i32), ("tw", _i32),
                ("nh", _i32), ("nw", _i32)]


class PrepJob(ctypes.Structure):
    _fields_ = [("src", _vp), ("src_strides", _i64 * 4), ("geom", TileGeom), ("dst", _vp), ("dst_strides", _i64 * 5),
                ("dst_off", _i64), ("scales", _vp), ("scale_strides", _i64 * 3), ("mean", _vp),
                ("mean_normalized", _vp), ("mean_strides", _i64 * 4), ("pool_off", _i64)]


class MaskParams(ctypes.Structure):
    _fields_ = [("metric", _i32), ("budget_mode", _i32), ("topk_ratio", ctypes.c_double),
                ("min_budget", _i32), ("n_recent", _i32), ("force_diag", _i32), ("force_sink", _i32),
                ("force_neighbors", _i32), ("nq", _i32), ("nk", _i32), ("nh", _i32), ("nw", _i32),
                ("num_txt_blk", _i32), ("kmax", _i32), ("row_budget", _vp), ("scale", ctypes.c_float),
                ("k_normalized", _i32)]


# name -> (restype, argtypes); mirrors include/li_sparse_attn.h
SIGNATURES = {
    "li_abi_version": (ctypes.c_int, []),
    "li_status_string": (ctypes.c_char_p, [ctypes.c_int]),
    "li_last_error": (ctypes.c_char_p, []),
    "li_q_prep": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _vp, _i64p, _vp, _i64p, _vp, _i64p,
                                 ctypes.POINTER(TileGeom), _vp]),
    "li_kv_prep": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _vp, _i64p, _vp, _i64p, _vp, _i64p, _vp, _i64p,
                                  _vp, _i64p, _i64, _i64, ctypes.POINTER(TileGeom), _vp]),
    "li_untile": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _vp, _i64p, _vp, _i64p,
                                 ctypes.POINTER(TileGeom), _vp]),
    "li_block_mask": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _vp, _i64p, _vp, _i64p,
                                     ctypes.POINTER(MaskParams), _vp, _vp, _vp, _vp]),
    "li_check_block_ids": (ctypes.c_int, [_vp, _i64, _i32, _vp, _vp]),
    "li_bsa_fwd": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _i32, _i32, _vp, _vp, _vp, _vp, _i64p, _i32,
                                  _vp, _i64p, ctypes.c_float, _i32, _vp, _vp, _vp, _i64, _i32, _vp]),
    "li_bsa_fwd_workspace_size": (ctypes.c_int64, [_i32, _i32, _i32, _i32, _i32]),
    "li_bsa_fwd_workspace_size_cols": (ctypes.c_int64, [_i32, _i32, _i32, _i32, _i32, _i32]),
    "li_bsa_fwd_gather": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _vp, _i64p, _vp, _i64p, _vp, _i64p, _vp, _vp,
                                         _i32, ctypes.POINTER(TileGeom), ctypes.POINTER(TileGeom), _vp, _i64p, _i32,
                                         _vp, _i64p, ctypes.c_float, _vp, _i64p, _vp, _vp, _i64, _i32, _vp]),
    "li_bsa_fwd_gather_noalloc": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _vp, _i64p, _vp, _i64p, _vp, _i64p,
                                                 _vp, _vp, _i32, ctypes.POINTER(TileGeom), ctypes.POINTER(TileGeom),
                                                 _vp, _i64p, _i32, _vp, _i64p, ctypes.c_float, _vp, _i64p, _vp, _i32,
                                                 _vp]),
    "li_bsa_fwd_qo": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _vp, _i64p, _vp, _vp, _vp, _vp, _i32,
                                     ctypes.POINTER(TileGeom), _vp, _i64p, _i32, _vp, _i64p, ctypes.c_float, _vp,
                                     _i64p, _vp, _vp, _i64, _i32, _vp]),
    "li_bsa_fwd_noalloc_scratch_bytes": (ctypes.c_int64, []),
    "li_tile_prep_fp8": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _vp, _i64p, _vp, _i64p, _vp, _i64p, _vp, _i64p,
                                        _i64, _i64, ctypes.POINTER(TileGeom), _vp]),
    "li_kv_prep_fp8": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _vp, _i64p, _vp, _i64p, _vp, _i64p, _vp, _i64p,
                                      _vp, _i64p, _vp, _i64p, _i64, _i64, ctypes.POINTER(TileGeom), _vp]),
    "li_bsa_fwd_fp8": (ctypes.c_int, [_i32, _i32, _i32, _i32, _i32, _vp, _vp, _vp, _vp, _vp, _vp, _i64p, _i32, _vp,
                                      _i64p, ctypes.c_float, _i32, _vp, _vp, _vp, _i64, _i32, _vp]),
    "li_bsa_fwd_fp8_gather": (ctypes.c_int, [_i32, _i32, _i32, _vp, _vp, _vp, _vp, _vp, _i64p, _vp, _i32,
                                             ctypes.POINTER(TileGeom), ctypes.POINTER(TileGeom), _vp, _i64p, _i32, _vp,
                                             _i64p, ctypes.c_float, _vp, _i64p, _vp, _vp, _i64, _i32, _vp]),
    "li_attn_fwd_dense": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _i32, _i32, _vp, _i64p, _vp, _i64p, _vp,
                                         _i64p, _vp, _vp, _i32, ctypes.c_float, _vp, _i64p, _vp, _vp, _i64, _vp]),
    "li_pool": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _vp, _i64p, _vp, _i64p, _i64,
                               ctypes.POINTER(TileGeom), _vp]),
    "li_prep": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, ctypes.POINTER(PrepJob), _i32, _vp]),
    "li_pool_pair": (ctypes.c_int, [ctypes.c_int, _i32, _i32, _i32, _vp, _i64p, _vp, _i64p, _i64,
                                    ctypes.POINTER(TileGeom), _vp, _i64p, _vp, _i64p, _i64,
                                    ctypes.POINTER(TileGeom), _vp, _vp]),
}


def _load():
    if not os.path.exists(LIB_PATH):
        raise ImportError(f"{LIB_PATH} is not built; run `python light-interaction-project_amd/build_lib.py` "
                          "(or __graft_entry__.build()) first")
    lib = ctypes.CDLL(LIB_PATH)
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = res
        fn.argtypes = args
    v = lib.li_abi_version()
    if v != ABI_VERSION:
        raise ImportError(f"{LIB_PATH} has ABI version {v}, expected {ABI_VERSION}; rebuild it")
    return lib


lib = _load()


def status_string(code):
    return lib.li_status_string(code).decode()


class LiError(RuntimeError):
    def __init__(self, fn, code):
        msg = f"{fn} failed: {status_string(code)} (status {code})"
        if code == LI_ERR_LAUNCH:
            msg += f": {lib.li_last_error().decode()}"
        super().__init__(msg)
        self.code = code


def check(fn, code):
    if code != LI_OK:
        raise LiError(fn, code)


def i64_array(vals):
    vals = list(vals)
    return (ctypes.c_int64 * len(vals))(*vals)

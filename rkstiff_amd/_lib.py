"""ctypes binding of librkstiff_amd.so (the C ABI declared in include/rkstiff_amd.h).

The library is the only compute path of this package: importing a solver that
needs it raises ``RuntimeError`` when the shared object is missing, and every
call that launches device work requires a HIP device.  There is no CPU fallback.
"""
import ctypes
import os
import threading

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "librkstiff_amd.so")

RKS_OK, RKS_ERR_INVALID, RKS_ERR_HIP, RKS_MAXLOOPS, RKS_MINSTEP, RKS_PAUSED, RKS_RUNNING = range(7)
METHOD_IDS = {"ETD35": 0, "ETD34": 1, "ETD4": 2, "ETD5": 3, "IF34": 4, "IF45DP": 5, "IF4": 6}
NL_ADVECT_RFFT, NL_CUBIC_FFT, NL_NONE, NL_AC2D_RFFT2, NL_HANKEL_CUBIC = 0, 1, 2, 3, 4
F64, F32, MIXED = 0, 1, 2

EXPORTS = (
    "rks_plan_create", "rks_plan_destroy", "rks_plan_info", "rks_set_storage", "rks_evolve",
    "rks_resume", "rks_step", "rks_reset", "rks_nl_eval", "rks_coeffs", "rks_combine",
    "rks_error_s", "rks_get_stats", "rks_read_log", "rks_read_snapshots", "rks_get_tableau",
    "rks_sizeof", "rks_last_error", "rks_set_config",
    "rks_mlp_create", "rks_mlp_destroy", "rks_mlp_get_params", "rks_mlp_train", "rks_mlp_forward",
    "rks_mlp_gradient", "rks_mlp_infer_single", "rks_plan_set_proposer", "rks_set_records",
    "rks_read_records", "rks_hankel_create", "rks_hankel_destroy", "rks_hankel_apply", "rks_hankel_cubic",
    "rks_hankel_cubic_noalloc", "rks_dense_coeffs", "rks_dense_ws_bytes", "rks_dense_coeffs_ws",
    "rks_dense_combine",
    "rks_plan_buckets", "rks_plan_set_launch", "rks_plan_tiles", "rks_plan_set_priority",
)

# learned step-size proposer (include/rkstiff_amd.h)
PROPOSER_NIN, PROPOSER_REC, PROPOSER_NPARAM = 66, 68, 156673
POLICIES = {"propose": 0, "guard": 1, "grow": 2}


class Config(ctypes.Structure):
    _fields_ = [("epsilon", ctypes.c_double), ("incr_f", ctypes.c_double),
                ("decr_f", ctypes.c_double), ("safety_f", ctypes.c_double),
                ("adapt_cutoff", ctypes.c_double), ("minh", ctypes.c_double),
                ("max_s", ctypes.c_double), ("min_s", ctypes.c_double),
                ("max_loops", ctypes.c_int), ("contour_points", ctypes.c_int),
                ("modecutoff", ctypes.c_double), ("contour_radius", ctypes.c_double)]


class InstanceDesc(ctypes.Structure):
    _fields_ = [("n", ctypes.c_int), ("L_is_complex", ctypes.c_int),
                ("L", ctypes.c_void_p), ("kx", ctypes.c_void_p), ("nl_coef", ctypes.c_double),
                ("ny", ctypes.c_int), ("nl_scale", ctypes.c_double)]


class DenseTerm(ctypes.Structure):
    """rks_dense_term: alpha * mat (x + s2 x2)."""
    _fields_ = [("mat", ctypes.c_void_p), ("x", ctypes.c_void_p), ("x2", ctypes.c_void_p),
                ("s2", ctypes.c_double), ("alpha", ctypes.c_double)]


DENSE_MAX_TERMS = 8


class Stats(ctypes.Structure):
    _fields_ = [("tc", ctypes.c_double), ("h_used", ctypes.c_double),
                ("h_next", ctypes.c_double), ("h", ctypes.c_double),
                ("steps", ctypes.c_int), ("attempts", ctypes.c_int),
                ("rejects", ctypes.c_int), ("status", ctypes.c_int),
                ("log_count", ctypes.c_int), ("snap_count", ctypes.c_int),
                ("nl_calls", ctypes.c_int), ("coef_updates", ctypes.c_int)]


# tableau mirror (rkstiff_amd/csrc/rks_types.h)
MAX_STAGES, MAX_TERMS, MAX_COEF, MAX_FRAC, MAX_SLOTS = 8, 8, 32, 16, 8


class Term(ctypes.Structure):
    _fields_ = [("src", ctypes.c_int), ("src2", ctypes.c_int), ("coef", ctypes.c_int),
                ("hmode", ctypes.c_int), ("scale", ctypes.c_double), ("scale2", ctypes.c_double),
                ("den", ctypes.c_double)]


class Stage(ctypes.Structure):
    _fields_ = [("ecoef", ctypes.c_int), ("nterm", ctypes.c_int), ("has_nl", ctypes.c_int),
                ("nl_slot", ctypes.c_int), ("hsum", ctypes.c_int), ("pad", ctypes.c_int),
                ("t", Term * MAX_TERMS)]


class Frac(ctypes.Structure):
    _fields_ = [("fnum", ctypes.c_int), ("fden", ctypes.c_int), ("mask", ctypes.c_int),
                ("pad", ctypes.c_int)]


class Coef(ctypes.Structure):
    _fields_ = [("nb", ctypes.c_int), ("hmul", ctypes.c_int), ("frac", ctypes.c_int),
                ("pad", ctypes.c_int), ("kind", ctypes.c_int * 4), ("w", ctypes.c_double * 4),
                ("outer", ctypes.c_double), ("den", ctypes.c_double)]


class Tableau(ctypes.Structure):
    _fields_ = [("method", ctypes.c_int), ("adaptive", ctypes.c_int), ("q", ctypes.c_int),
                ("nl1_policy", ctypes.c_int), ("fsal_slot", ctypes.c_int), ("nslot", ctypes.c_int),
                ("nstage", ctypes.c_int), ("nerr", ctypes.c_int), ("ncoef", ctypes.c_int),
                ("nfrac", ctypes.c_int), ("uses_contour", ctypes.c_int),
                ("coef_rs", ctypes.c_int * MAX_COEF), ("coef_off", ctypes.c_int * MAX_COEF),
                ("err_coef", ctypes.c_int),
                ("err_factored", ctypes.c_int), ("err_hpow", ctypes.c_int), ("pad2", ctypes.c_int),
                ("err_scale", ctypes.c_double),
                ("st", Stage * MAX_STAGES), ("err", Term * MAX_TERMS),
                ("coef", Coef * MAX_COEF), ("frac", Frac * MAX_FRAC)]


_lib = None
_lock = threading.Lock()


def load(path=None):
    """Load the shared library once; raise RuntimeError if it is not built."""
    global _lib
    with _lock:
        if _lib is not None:
            return _lib
        p = path or LIB_PATH
        if not os.path.exists(p):
            raise RuntimeError(
                f"rkstiff_amd: HIP library {p} is not built; run __graft_entry__.build() "
                "(hipcc, gfx950). There is no CPU fallback.")
        lib = ctypes.CDLL(p)
        vp, ip, dp = ctypes.c_void_p, ctypes.c_int, ctypes.c_double
        P = ctypes.POINTER
        lib.rks_plan_create.argtypes = [ip, ip, ip, P(Config), ip, P(InstanceDesc), P(vp)]
        lib.rks_plan_destroy.argtypes = [vp]
        lib.rks_plan_info.argtypes = [vp, P(ip), P(ip), P(ip), P(ip)]
        lib.rks_set_storage.argtypes = [vp, ip, ip, ip]
        lib.rks_evolve.argtypes = [vp, P(vp), P(vp), P(dp), P(dp), P(dp), vp]
        lib.rks_resume.argtypes = [vp, vp]
        lib.rks_step.argtypes = [vp, P(vp), P(vp), P(dp), vp]
        lib.rks_reset.argtypes = [vp, vp]
        lib.rks_nl_eval.argtypes = [vp, P(vp), P(vp), vp]
        lib.rks_coeffs.argtypes = [vp, ip, dp, vp, vp]
        lib.rks_combine.argtypes = [vp, ip, ip, dp, vp, P(vp), vp, vp]
        lib.rks_error_s.argtypes = [vp, ip, vp, vp, vp, vp]
        lib.rks_get_stats.argtypes = [vp, P(Stats), vp]
        lib.rks_read_log.argtypes = [vp, ip, P(dp), ip, vp]
        lib.rks_read_snapshots.argtypes = [vp, ip, vp, P(dp), ip, vp]
        lib.rks_get_tableau.argtypes = [ip, vp, ip]
        lib.rks_sizeof.argtypes = [ip]
        lib.rks_set_config.argtypes = [vp, P(Config), vp]
        fp = P(ctypes.c_float)
        lib.rks_mlp_create.argtypes = [fp, fp, fp, P(vp)]
        lib.rks_mlp_destroy.argtypes = [vp]
        lib.rks_mlp_get_params.argtypes = [vp, fp]
        lib.rks_mlp_train.argtypes = [vp, vp, ip, vp, ip, ip, ip, dp, dp, vp, vp]
        lib.rks_mlp_forward.argtypes = [vp, vp, ip, vp, vp]
        lib.rks_mlp_gradient.argtypes = [vp, vp, ip, ip, dp, vp, vp, vp, vp]
        lib.rks_mlp_infer_single.argtypes = [vp, vp, ip, ip, vp, vp]
        lib.rks_plan_set_proposer.argtypes = [vp, vp, ip, dp, dp, dp, ip]
        lib.rks_set_records.argtypes = [vp, ip]
        lib.rks_read_records.argtypes = [vp, vp, P(ip), vp]
        lib.rks_hankel_create.argtypes = [ip, P(dp), dp, P(vp)]
        lib.rks_hankel_destroy.argtypes = [vp]
        lib.rks_hankel_apply.argtypes = [vp, ip, vp, vp, ip, ip, vp]
        lib.rks_hankel_cubic.argtypes = [vp, dp, vp, vp, ip, vp]
        lib.rks_hankel_cubic_noalloc.argtypes = [vp, dp, vp, vp, ip, vp]
        lib.rks_dense_coeffs.argtypes = [ip, ip, ip, vp, P(dp), ip, dp, vp, vp]
        lib.rks_dense_ws_bytes.argtypes = [ip, ip, ip, ip, P(ctypes.c_size_t)]
        lib.rks_dense_coeffs_ws.argtypes = [ip, ip, ip, vp, P(dp), ip, dp, vp, vp, ctypes.c_size_t, vp]
        lib.rks_dense_combine.argtypes = [ip, ip, vp, ip, vp, vp]
        lib.rks_plan_buckets.argtypes = [vp, P(ip), P(ip), P(ip), P(ip), P(ip), ip]
        lib.rks_plan_set_launch.argtypes = [vp, ip, P(ip), P(ip), ip]
        lib.rks_plan_tiles.argtypes = [vp, P(ip), ip]
        lib.rks_plan_set_priority.argtypes = [vp, P(dp)]
        lib.rks_last_error.restype = ctypes.c_char_p
        for name in EXPORTS:
            if name not in ("rks_last_error",):
                getattr(lib, name).restype = ctypes.c_int
        assert lib.rks_sizeof(0) == ctypes.sizeof(Tableau), "tableau layout mismatch"
        assert lib.rks_sizeof(4) == ctypes.sizeof(InstanceDesc), "instance descriptor layout mismatch"
        assert lib.rks_sizeof(5) == ctypes.sizeof(Config), "config layout mismatch"
        assert lib.rks_sizeof(6) == ctypes.sizeof(Stats), "stats layout mismatch"
        _lib = lib
        return lib


def check(rc):
    """Raise for a non-OK return code (ValueError for invalid arguments)."""
    if rc == RKS_OK:
        return
    msg = load().rks_last_error().decode()
    if rc == RKS_ERR_INVALID:
        raise ValueError(msg)
    raise RuntimeError(f"rkstiff_amd error {rc}: {msg}")


def tableau(method):
    """Host-side copy of a method tableau (no device needed)."""
    t = Tableau()
    check(load().rks_get_tableau(METHOD_IDS[method], ctypes.byref(t), ctypes.sizeof(t)))
    return t


def ptr_array(ptrs):
    return (ctypes.c_void_p * len(ptrs))(*ptrs)


def dbl_array(vals):
    return (ctypes.c_double * len(vals))(*vals)

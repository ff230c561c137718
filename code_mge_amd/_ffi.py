"""ctypes binding of include/mge.h (libmge.so, built in-tree).

The library is required: importing a solver without it raises, there is
no CPU fallback.
"""
import ctypes as C
import os

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "lib", "libmge.so")

MGE_OK = 0
ERRORS = {
    -10: "MGE_ERR_NEG_C2", -11: "MGE_ERR_WALL_RHO", -12: "MGE_ERR_WSOL_NAN",
    -13: "MGE_ERR_RES_NAN", -14: "MGE_ERR_PERIODIC", -15: "MGE_ERR_DISTYPE",
    -16: "MGE_ERR_SMOO_DIM", -20: "MGE_ERR_ARG", -21: "MGE_ERR_HIP",
    -22: "MGE_ERR_NOMEM", -23: "MGE_ERR_STATE", -24: "MGE_ERR_RESTART",
}
WARNINGS = {1: "MGE_WARN_ZERO_CLOUD", 2: "MGE_WARN_BCTYPE"}

BODY_NONE, BODY_CYLINDER, BODY_SPHERE, BODY_ELLIPSOID = 0, 1, 2, 3


class MgeParams(C.Structure):
    _fields_ = [
        ("mstage", C.c_int),
        ("cstp", C.c_double * 8),
        ("cdis", C.c_double * 8),
        ("cfl", C.c_double),
        ("vt", C.c_int),
        ("vis2", C.c_double),
        ("vis4", C.c_double),
        ("smoo", C.c_double),
        ("mgtype", C.c_int),
        ("gamma", C.c_double),
        ("rho0", C.c_double), ("p0", C.c_double), ("c0", C.c_double), ("ei0", C.c_double),
        ("u0", C.c_double), ("v0", C.c_double), ("w0", C.c_double), ("h0", C.c_double),
        ("eqntype", C.c_int),
        ("dissip", C.c_int),
        ("viscl", C.c_double), ("prlmean", C.c_double), ("gas_const", C.c_double),
        ("drop", C.c_double),
        ("distype", C.c_int),
        ("precision", C.c_int),
        ("epsentr", C.c_double),
        ("execmode", C.c_int),
        ("dtstep", C.c_double),
        ("smoother", C.c_int),
        ("ffreeze", C.c_double),
        ("lfreeze", C.c_double),
    ]


class MgePinGrid(C.Structure):
    _fields_ = [("name", C.c_int), ("points", C.c_int * 3), ("origin", C.c_double * 3), ("length", C.c_double * 3)]


class MgeJob(C.Structure):
    _fields_ = [
        ("job", C.c_char * 64), ("model", C.c_char * 64), ("mesh", C.c_char * 512), ("surface", C.c_char * 512),
        ("nlevel", C.c_int), ("mcyc", C.c_int * 16),
        ("mach", C.c_double), ("reynolds", C.c_double), ("gamma", C.c_double), ("prlmean", C.c_double),
        ("alphad", C.c_double), ("betad", C.c_double),
        ("cflf", C.c_double), ("vis2", C.c_double), ("vis4", C.c_double), ("smoo", C.c_double),
        ("epsentr", C.c_double),
        ("mgtype", C.c_int), ("mstage", C.c_int),
        ("cstp", C.c_double * 8), ("cdis", C.c_double * 8),
        ("eqntype", C.c_int), ("distype", C.c_int), ("dissip", C.c_int),
        ("n", C.c_int * 3),
        ("lo", C.c_double * 3), ("hi", C.c_double * 3), ("dom_lo", C.c_double * 3), ("dom_hi", C.c_double * 3),
        ("bctype", C.c_int * 6),
        ("iflow", C.c_int),
        ("execmode", C.c_int), ("nperiod", C.c_int), ("nstep", C.c_int),
        ("dt", C.c_double), ("pmean", C.c_double), ("tmean", C.c_double), ("rgasmean", C.c_double),
    ]


class MgeCutRec(C.Structure):
    _fields_ = [
        ("faceid", C.c_int), ("zz", C.c_int),
        ("ccid", C.c_int * 3), ("scid", C.c_int * 3),
        ("psurf", C.c_double * 3), ("nvec", C.c_double * 3),
        ("radcur", C.c_double * 2), ("rr", C.c_double),
        ("npoint", C.c_int),
        ("ijk", (C.c_int * 3) * 8),
        ("coef", C.c_double * 8),
        ("psol", C.c_double), ("wsol", C.c_double * 5),
    ]


class MgeBody(C.Structure):
    _fields_ = [
        ("kind", C.c_int), ("axis", C.c_int),
        ("center", C.c_double * 3), ("semi", C.c_double * 3), ("rot", C.c_double * 9),
    ]


class MgeError(RuntimeError):
    def __init__(self, code, where, msg=""):
        self.code = code
        super().__init__(f"{where}: {ERRORS.get(code, code)} {msg}".strip())


_lib = None


def lib():
    """Load libmge.so; raise if it has not been built."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise MgeError(-21, "load", f"{LIB_PATH} is missing; run code_mge_amd/build.py")
    L = C.CDLL(LIB_PATH)
    P, I, D = C.c_void_p, C.c_int, C.c_double
    dp = C.POINTER(C.c_double)
    L.mge_last_error.restype = C.c_char_p
    L.mge_geom_level.argtypes = [C.POINTER(MgeBody), I, I, I, dp, dp, dp, C.c_void_p,
                                 C.POINTER(MgeCutRec), I, C.POINTER(I)]
    L.mge_geom_level_tri.argtypes = [dp, I, I, I, I, dp, dp, dp, C.c_void_p, C.POINTER(MgeCutRec), I,
                                     C.POINTER(I)]
    L.mge_case_create.argtypes = [C.POINTER(MgeParams), I, C.POINTER(P)]
    L.mge_case_destroy.argtypes = [P]
    L.mge_level_define.argtypes = [P, I, I, I, I, dp, dp, dp, D, C.POINTER(I), C.POINTER(I),
                                   C.c_void_p, I, C.POINTER(MgeCutRec), I]
    L.mge_init_flow.argtypes = [P]
    L.mge_timestep.argtypes = [P, I, I]
    L.mge_euler.argtypes = [P, I, I, I, I, I, I, I, I, dp]
    L.mge_bcond.argtypes = [P, I, I]
    L.mge_bc_cutcell.argtypes = [P, I, I]
    L.mge_bc_overlap.argtypes = [P, I]
    L.mge_movco.argtypes = [P, I]
    L.mge_movfin.argtypes = [P, I, I]
    L.mge_solve.argtypes = [P, C.POINTER(I), dp, I, C.POINTER(I), C.POINTER(C.c_longlong)]
    L.mge_download.argtypes = [P, I, I, C.c_char_p, dp]
    L.mge_upload.argtypes = [P, I, I, C.c_char_p, dp]
    L.mge_get_cuts.argtypes = [P, I, I, C.POINTER(MgeCutRec)]
    L.mge_get_dtim.argtypes = [P, I, I]
    L.mge_get_dtim.restype = D
    L.mge_wall_force.argtypes = [P, I, dp]
    L.mge_synchronize.argtypes = [P]
    L.mge_kernel_timing.argtypes = [P, I, C.c_char_p, dp, C.POINTER(C.c_longlong), dp]
    L.mge_cycles.argtypes = [P, I, I, I, dp, C.POINTER(C.c_longlong)]
    L.mge_solve_step.argtypes = [P, C.POINTER(I), I, dp, I, C.POINTER(I), C.POINTER(C.c_longlong)]
    L.mge_shift_time_levels.argtypes = [P]
    L.mge_upload_solut.argtypes = [P, I, I, C.c_double, dp, C.POINTER(I)]
    L.mge_upload_solut_noalloc.argtypes = [P, I, I, C.c_double, dp, C.POINTER(I)]
    L.mge_case_bytes.argtypes = [P]
    L.mge_case_bytes.restype = C.c_longlong
    L.mge_autotune.argtypes = [P, I, C.POINTER(I), dp]
    L.mge_read_job.argtypes = [C.c_char_p, C.POINTER(MgeJob)]
    L.mge_write_solut.argtypes = [P, C.c_char_p, I]
    L.mge_read_solut.argtypes = [P, C.c_char_p, I]
    L.mge_job_params.argtypes = [C.POINTER(MgeJob), I, C.POINTER(MgeParams)]
    L.mge_job_level.argtypes = [C.POINTER(MgeJob), I, C.POINTER(I), C.POINTER(I)]
    L.mge_read_pin.argtypes = [C.c_char_p, I, C.POINTER(MgePinGrid), C.POINTER(I)]
    L.mge_read_p3d.argtypes = [C.c_char_p, I, dp, C.POINTER(I)]
    L.mge_input_error.restype = C.c_char_p
    L.mge_set_kc.argtypes = [P, I, I]
    L.mge_stage_tile.argtypes = [P, I, C.POINTER(I), C.POINTER(I)]
    L.mge_set_tile.argtypes = [P, I, I, I]
    L.mge_set_freeze.argtypes = [P, I, I]
    L.mge_comp_create.argtypes = [I, C.POINTER(P), C.POINTER(I), C.POINTER(I), C.POINTER(I), C.POINTER(P)]
    L.mge_comp_solve.argtypes = [P, C.POINTER(I), dp, I, C.POINTER(I), C.POINTER(C.c_longlong)]
    L.mge_comp_destroy.argtypes = [P]
    L.mge_batch_create.argtypes = [I, I, C.POINTER(P)]
    L.mge_batch_destroy.argtypes = [P]
    L.mge_batch_add.argtypes = [P, P, D, I]
    L.mge_batch_remove.argtypes = [P, I]
    L.mge_batch_run.argtypes = [P, I, C.POINTER(I)]
    L.mge_batch_status.argtypes = [P, I, C.POINTER(I), C.POINTER(I), dp, dp]
    L.mge_batch_log.argtypes = [P, I, dp, I]
    L.mge_batch_stage_tile.argtypes = [P, I, I, C.POINTER(I), C.POINTER(I)]
    _lib = L
    return L


def check(rc, where):
    """Raise on a negative status; return warnings (positive) unchanged."""
    if rc < 0:
        msg = lib().mge_last_error()
        raise MgeError(rc, where, msg.decode() if msg else "")
    return rc


EXPORTED = [
    "mge_geom_level", "mge_case_create", "mge_case_destroy", "mge_level_define",
    "mge_init_flow", "mge_timestep", "mge_euler", "mge_bcond", "mge_bc_cutcell",
    "mge_bc_overlap", "mge_movco", "mge_movfin", "mge_solve", "mge_download",
    "mge_upload", "mge_get_cuts", "mge_get_dtim", "mge_wall_force", "mge_synchronize",
    "mge_kernel_timing", "mge_last_error", "mge_cycles",
    "mge_batch_create", "mge_batch_destroy", "mge_batch_add", "mge_batch_remove", "mge_batch_run",
    "mge_batch_status", "mge_batch_log", "mge_batch_stage_tile", "mge_case_bytes", "mge_autotune", "mge_set_kc", "mge_geom_level_tri",
    "mge_stage_tile", "mge_set_tile", "mge_set_freeze", "mge_comp_create", "mge_comp_solve", "mge_comp_destroy",
    "mge_read_job", "mge_job_params", "mge_job_level", "mge_read_pin", "mge_read_p3d", "mge_input_error",
    "mge_write_solut", "mge_read_solut", "mge_solve_step", "mge_shift_time_levels",
    "mge_upload_solut", "mge_upload_solut_noalloc",
]

"""ctypes binding of libpychem_hip.so (the C ABI in include/pychem_hip.h).

The library is mandatory: if it is missing or cannot be loaded this module
raises, there is no CPU fallback.
"""
import ctypes
import os

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libpychem_hip.so")
_LIB = None

c_int, c_double, c_void_p, c_longlong = ctypes.c_int, ctypes.c_double, ctypes.c_void_p, ctypes.c_longlong
P_int = ctypes.POINTER(ctypes.c_int)
P_double = ctypes.POINTER(ctypes.c_double)
P_ll = ctypes.POINTER(ctypes.c_longlong)

# pq_scf_observer_fn: (user, cycle, spin, dE) -> nonzero to keep observing
SCF_OBSERVER = ctypes.CFUNCTYPE(c_int, c_void_p, c_int, c_int, c_double)

# name -> (restype, argtypes); mirrors include/pychem_hip.h
SIGNATURES = {
    "pq_last_error": (ctypes.c_char_p, []),
    "pq_version": (c_int, []),
    "pq_device_count": (c_int, []),
    "pq_cache_release": (c_int, []),
    "pq_scf_dots_work": (ctypes.c_longlong, [ctypes.c_longlong, c_int]),
    "pq_scf_dots": (c_int, [ctypes.POINTER(c_void_p), ctypes.POINTER(c_void_p), c_int, ctypes.POINTER(c_void_p), c_int,
                            ctypes.c_longlong, c_void_p, ctypes.POINTER(c_double), c_void_p]),
    "pq_lincomb": (c_int, [ctypes.POINTER(c_void_p), ctypes.POINTER(c_double), c_int, ctypes.c_longlong, c_void_p,
                           c_void_p]),
    "pq_scf_work": (ctypes.c_longlong, [c_int, c_int, c_int, c_int, c_int]),
    "pq_scf_run": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_void_p, c_int, c_int, c_int,
                           c_int, c_double, c_int, c_int, c_int, c_double, c_double, c_int, c_void_p, c_void_p,
                           c_void_p, c_void_p, c_void_p, P_double, P_double, P_double, c_void_p]),
    "pq_cache_bytes": (ctypes.c_longlong, []),
    "pq_boys": (c_int, [c_int, c_void_p, c_int, c_void_p, c_void_p]),
    "pq_basis_create": (c_int, [c_int, P_int, P_int, P_int, P_double, P_double, P_double,
                                c_int, P_double, P_double, ctypes.POINTER(c_void_p)]),
    "pq_basis_destroy": (None, [c_void_p]),
    "pq_basis_create_batch": (c_int, [c_int, c_int, P_int, P_int, P_int, P_double, P_double, P_double, P_int,
                                      c_int, P_double, P_double, P_int, ctypes.POINTER(c_void_p)]),
    "pq_basis_molecules": (c_int, [c_void_p, P_ll, P_int, P_int, P_int]),
    "pq_jk_set_params": (c_int, [c_void_p, c_int, c_int, c_int, c_void_p]),
    "pq_jk_class": (c_int, [c_void_p, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p, P_int, c_void_p]),
    "pq_jk_graph_create": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p]),
    "pq_jk_graph_launch": (c_int, [c_void_p, c_void_p]),
    "pq_jk_set_streams": (c_int, [c_void_p, c_int]),
    "pq_basis_set_spherical": (c_int, [c_void_p, P_int]),
    "pq_basis_info": (c_int, [c_void_p, P_ll]),
    "pq_one_electron": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p]),
    "pq_schwarz": (c_int, [c_void_p, P_double, c_void_p]),
    "pq_eri_build": (c_int, [c_void_p, c_double, c_double, c_void_p]),
    "pq_eri_plan": (c_int, [c_void_p, c_double, c_double, c_void_p]),
    "pq_eri_compute": (c_int, [c_void_p, c_void_p]),
    "pq_eri_recompute": (c_int, [c_void_p, c_void_p]),
    "pq_set_timing": (c_int, [c_void_p, c_int]),
    "pq_get_timings": (c_int, [c_void_p, P_double, P_double, P_double]),
    "pq_eri_run_class": (c_int, [c_void_p, c_int, c_int, c_void_p]),
    "pq_eri_nclass": (c_int, []),
    "pq_eri_stats": (c_int, [c_void_p, P_ll, c_int]),
    "pq_jk": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p]),
    "pq_jk_general": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p]),
    "pq_eri_set_operator": (c_int, [c_void_p, c_int, ctypes.c_double]),
    "pq_jk_class_times": (c_int, [c_void_p, P_double, P_ll, P_ll, c_int]),
    "pq_jk_general_noalloc": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p]),
    "pq_eri_dense": (c_int, [c_void_p, c_void_p, c_void_p]),
    "pq_eri_blocks": (c_int, [c_void_p, c_int, P_int, P_double, c_void_p]),
    "pq_eri_dense_slab": (c_int, [c_void_p, c_int, c_int, c_void_p, c_void_p]),
    "pq_gemm_f64": (c_int, [c_int, c_int, c_int, c_int, c_int, c_double, c_void_p, c_longlong, c_longlong,
                            c_void_p, c_longlong, c_longlong, c_double, c_void_p, c_longlong, c_longlong,
                            c_int, c_void_p]),
    "pq_mp2_ovov": (c_int, [c_void_p, c_int, c_int, c_void_p, c_void_p, c_int, c_int, c_void_p, c_void_p,
                            c_void_p, c_longlong, c_int, c_void_p]),
    "pq_purify": (c_int, [c_void_p, c_int, c_int, c_void_p, c_void_p, c_double, c_int, P_int,
                          ctypes.POINTER(c_double), c_void_p]),
    "pq_gemm_bf16x3": (c_int, [c_int, c_int, c_int, c_int, c_int, c_double, c_void_p, c_longlong, c_longlong,
                               c_void_p, c_longlong, c_longlong, c_double, c_void_p, c_longlong, c_longlong,
                               c_int, c_void_p]),
    "pq_mlp_linear_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int,
                                  c_void_p]),
    "pq_mlp_linear_bwd": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                  c_int, c_int, c_int, c_int, c_void_p]),
    "pq_mlp_mse": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_longlong, ctypes.c_float, c_void_p]),
    "pq_mlp_adam": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_longlong, ctypes.c_float, ctypes.c_float,
                            ctypes.c_float, ctypes.c_float, c_int, c_void_p]),
    "pq_mlp_forward": (c_int, [c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p]),
    "pq_mlp_backward": (c_int, [c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                c_int, c_void_p]),
    "pq_mlp_adam_multi": (c_int, [c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, ctypes.c_float,
                                  ctypes.c_float, ctypes.c_float, ctypes.c_float, c_int, c_void_p]),
    "pq_scf_set_observer": (c_int, [SCF_OBSERVER, c_void_p, c_double, c_void_p, c_void_p]),
    "pq_eigh_refine_work": (ctypes.c_longlong, [c_int]),
    "pq_eigh_batched": (c_int, [c_void_p, c_int, c_int, c_void_p, c_void_p, c_void_p]),
    "pq_purify_batched": (c_int, [c_void_p, c_void_p, c_int, c_int, c_double, c_int, c_void_p, c_void_p, c_void_p]),
    "pq_batch_pack": (c_int, [c_int, c_int] + [c_void_p] * 8),
    "pq_batch_fock": (c_int, [c_int, c_int] + [c_void_p] * 7),
    "pq_batch_test": (c_int, [c_int, c_int] + [c_void_p] * 6 + [c_double, c_double, c_int] + [c_void_p] * 6),
    "pq_batch_diis_work": (ctypes.c_longlong, [c_int, c_int]),
    "pq_batch_diis": (c_int, [c_int, c_int] + [c_void_p] * 5 + [c_int, c_int, c_int] + [c_void_p] * 4),
    "pq_batch_lift": (c_int, [c_int, c_int, c_void_p, c_void_p, c_void_p]),
    "pq_eigh_refine": (c_int, [c_void_p, c_void_p, c_int, c_int, c_double, c_void_p, c_void_p, P_double, c_void_p]),
    "pq_mp2_energy": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int,
                              c_int, P_double, c_void_p]),
}


class HipError(RuntimeError):
    pass


class PurifyStalled(HipError):
    """pq_scf_run returned -2: a purification did not become idempotent
    (degenerate levels at the Fermi level)."""


def lib():
    global _LIB
    if _LIB is None:
        if not os.path.exists(LIB_PATH):
            raise HipError("libpychem_hip.so not built (run python -m pychem_amd.build)")
        L = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(L, name)
            fn.restype = res
            fn.argtypes = args
        _LIB = L
    return _LIB


def check(rc, what):
    if rc != 0:
        msg = lib().pq_last_error()
        cls = PurifyStalled if rc == -2 and what == "pq_scf_run" else HipError
        raise cls("%s failed (%d): %s" % (what, rc, msg.decode() if msg else ""))


def iptr(a):
    return a.ctypes.data_as(P_int)


def dptr(a):
    return a.ctypes.data_as(P_double)

"""The library's product plans, as host code computes them (no device needed; fmlh_internal_*)."""
import collections
import ctypes

import freeml_amd as fh

SKINNY_NN, SKINNY_NT, MFMA, SPLIT = range(4)  # GemmPlan::Kind
Plan = collections.namedtuple("Plan", "kind tile k_groups splits ws_elems")


def plan(M, N, K, b_trans, lda=None, ldb=None):
    """Plan of a product of 16-byte aligned operands (row strides: those of packed matrices)."""
    out = [ctypes.c_int() for _ in range(4)]
    ws = ctypes.c_size_t()
    fh.lib().fmlh_internal_plan(M, N, K, b_trans, lda or K, ldb or (K if b_trans else N), *map(ctypes.byref, out), ctypes.byref(ws))
    return Plan(*(v.value for v in out), ws.value)


def engine_workspace(C, V, batch, rows):
    f = fh.lib().fmlh_internal_engine_workspace
    f.restype = ctypes.c_size_t
    return f(C, V, batch, rows)


def strided_tile(mode, M, N, K, l_rs, l_cs, r_rs, r_cs, o_rs, o_cs, batch=1, l_plane=0, r_plane=0):
    """Side of the split tiles a strided product of 16-byte aligned operands takes; 0: none."""
    u, z = ctypes.c_uint32, ctypes.c_size_t
    return fh.lib().fmlh_internal_strided_tile(mode, *map(u, (M, N, K, l_rs, l_cs, r_rs, r_cs, o_rs, o_cs, batch)),
                                               z(l_plane), z(r_plane))

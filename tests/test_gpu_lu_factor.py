"""The bottom level's LU factor, bit for bit the oracle's, signs of zeros
included: operators of either sign, with entries that are infinite or NaN at
the start, and ones whose factor overflows or divides by a denormal pivot on
the way; with the operator's band, with interchanges and on periodic levels."""
import ctypes

import numpy as np
import pytest

import pgmg_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [((4, 4, 4), 0, False), ((11, 7, 9), 0, False), ((11, 7, 9), 0, True), ((1, 1, 129), 0, False), ((30, 1, 17), 0, False),
         ((8, 6, 10), 7, False)]


def same_bits(a, b):
    n = np.isnan(a)
    return np.array_equal(n, np.isnan(b)) and np.array_equal(a[~n].view(np.int64), b[~n].view(np.int64))


def operators(A):
    o, n, m = A.shape[:3]
    mid = o // 2, n // 2, m // 2
    off = 12 if m > 1 else 4  # a neighbour inside the grid
    yield "as it is", A
    yield "negative", -A + 0.0
    for at, e, value in ((mid, 13, np.inf), (mid, off, -np.inf), (mid, off, np.nan), (mid, 13, np.nan),
                         ((0, 0, 0), 13, -np.inf), ((o - 1, n - 1, m - 1), 13, np.nan)):
        B = A.copy()
        B[at + (e,)] = value
        yield "%s at %s, %d" % (value, at, e), B
    yield "next to the largest", A / np.abs(A).max() * 1.7e308  # overflows where rows grow
    yield "denormal", A * 1e-310


@pytest.mark.parametrize("shape,prd,pivots", CASES)
def test_factor_bitwise(shape, prd, pivots):
    m, n, o = shape
    N = m * n * o
    A = O.gen_operator(P.FAM_Q1_ANISO, 5, m, n, o, prd=prd)
    if pivots:  # entries off the diagonal lead
        A[..., 13] *= 0.05
    elif prd:  # regular, also where every axis wraps
        A[..., 13] *= 1.5
    LU, ipiv = np.zeros((N, N)), np.zeros(N, dtype=np.int32)
    with P.Hierarchy(m, n, o, prd=prd, bottom=P.BOTTOM_LU, max_levels=1) as h:
        for what, B in operators(A):
            print("case", shape, prd, pivots, what, flush=True)
            h.set_operator27(B)
            h.compute_rats()
            ok, want, want_ipiv = O.lu_factor(B, prd=prd)
            assert h.lu_active() == bool(ok)
            if not ok:
                continue
            P._check(P.lib().pgmg_get_lu_factor(h.h, LU.ctypes.data_as(ctypes.POINTER(ctypes.c_double)),
                                                ipiv.ctypes.data_as(ctypes.POINTER(ctypes.c_int))))
            assert np.array_equal(ipiv - 1, want_ipiv)
            assert same_bits(LU, want)

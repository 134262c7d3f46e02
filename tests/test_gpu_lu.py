"""The bottom level's direct solve, bit for bit the oracle's: unknowns around
the edges of the 64-row and 32-column blocks, up to the most the direct solve
takes, factors with the operator's band, with interchanges and of periodic
levels, right-hand sides with zeros and at the limits of the fast quotient."""
import numpy as np
import pytest

import pgmg_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 2, 2), (31, 1, 1), (1, 33, 1), (3, 3, 7), (4, 4, 4), (5, 13, 1), (1, 1, 129), (2, 1, 500), (11, 7, 9),
          (10, 10, 10), (9, 12, 9), (11, 31, 6), (23, 1, 89)]
CASES = [(s, 0, False) for s in SHAPES] + [(s, 0, True) for s in [(4, 4, 4), (11, 7, 9), (1, 1, 129), (5, 5, 13)]] + \
        [(s, p, False) for s, p in [((8, 6, 10), 7), ((9, 7, 5), 1), ((3, 11, 4), 4)]]


@pytest.mark.parametrize("shape,prd,pivots", CASES)
def test_direct_solve_bitwise(shape, prd, pivots):
    m, n, o = shape
    print("case", shape, prd, pivots, flush=True)
    A = O.gen_operator(P.FAM_Q1_ANISO, 5, m, n, o, prd=prd)
    if pivots:  # entries off the diagonal lead
        A[..., 13] *= 0.05
    elif prd:  # regular, also where every axis wraps
        A[..., 13] *= 1.5
    b = O.gen_rhs(5, m, n, o)
    ok, LU, ipiv = lu_of(A, prd)
    assert ok
    assert (ipiv != np.arange(ipiv.size)).any() == pivots
    zeros = b.copy()
    zeros[:, :, ::2] = 0.0
    zeros[o // 2:] = 0.0
    tiny = b * 1e-160
    tiny[0, 0, 0] = 1e-310
    with P.Hierarchy(m, n, o, prd=prd, bottom=P.BOTTOM_LU, max_levels=1) as h:
        h.set_operator27(A)
        h.compute_rats()
        assert h.lu_active()
        for rhs in (b, zeros, tiny, b * 1e160, np.zeros_like(b)):
            h.set_rhs(rhs)
            h.solve_exact(0, smooth=False)
            ref = O.lu_solve(LU, ipiv, rhs.reshape(-1))
            assert np.array_equal(h.get_x().reshape(-1), ref.reshape(-1))


def lu_of(A, prd):
    ok, LU, ipiv = O.lu_factor(A, prd=prd)
    return ok, LU, np.asarray(ipiv)

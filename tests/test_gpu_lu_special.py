"""The bottom level's direct solve of sources with infinities, NaN and zeros of
either sign: bit for bit the oracle's column by column, with the operator's
band, with interchanges and on periodic levels."""
import numpy as np
import pytest

import pgmg_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [((1, 1, 1), 0, False), ((4, 4, 4), 0, False), ((1, 1, 129), 0, False), ((5, 13, 1), 0, False), ((11, 7, 9), 0, False),
         ((11, 7, 9), 0, True), ((1, 1, 129), 0, True),
         ((8, 6, 10), 7, False), ((9, 7, 5), 1, False), ((11, 31, 6), 0, False)]


def same_bits(a, b):
    a, b = a.reshape(-1), b.reshape(-1)
    n = np.isnan(a)
    return np.array_equal(n, np.isnan(b)) and np.array_equal(a[~n].view(np.int64), b[~n].view(np.int64))


def sources(shape):
    m, n, o = shape
    b = O.gen_rhs(5, m, n, o)
    for value in (np.inf, -np.inf, np.nan, -0.0, 1e308):
        for at in sorted({0, b.size // 2, b.size - 1}):
            r = b.copy()
            r.flat[at] = value
            yield r
        yield np.full_like(b, value)
    r = np.zeros_like(b)  # one unknown of infinity, the ones before it 0
    r.flat[b.size // 2] = np.inf
    yield r
    yield -np.abs(np.where(b > 0, b, 0.0))
    r = np.where(b > 0, 0.0, -0.0)
    r.flat[b.size // 3] = 1.0
    yield r


@pytest.mark.parametrize("shape,prd,pivots", CASES)
def test_direct_solve_special_sources(shape, prd, pivots):
    m, n, o = shape
    print("case", shape, prd, pivots, flush=True)
    A = O.gen_operator(P.FAM_Q1_ANISO, 5, m, n, o, prd=prd)
    if pivots:  # entries off the diagonal lead
        A[..., 13] *= 0.05
    elif prd:  # regular, also where every axis wraps
        A[..., 13] *= 1.5
    ok, LU, ipiv = O.lu_factor(A, prd=prd)
    assert ok
    with P.Hierarchy(m, n, o, prd=prd, bottom=P.BOTTOM_LU, max_levels=1) as h:
        h.set_operator27(A)
        h.compute_rats()
        assert h.lu_active()
        for r in sources(shape):
            h.set_rhs(r)
            h.solve_exact(0, smooth=False)
            assert same_bits(h.get_x(), O.lu_solve(LU, ipiv, r.reshape(-1)))

"""Backward and symmetric colour sweeps of the levels that take row launches:
bit for bit the oracle's for rows of one and several segments (128 points), odd
and even, a last segment of one point, 7 and 27 points, each set of periodic
axes, x holding infinities and NaN."""
import numpy as np
import pytest

import pgmg_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [((127, 13, 14), 0), ((128, 14, 13), 0), ((129, 13, 13), 0), ((130, 12, 14), 0), ((256, 9, 10), 0), ((257, 10, 9), 0),
         ((385, 9, 8), 0), ((33, 30, 31), 0), ((1, 150, 140), 0), ((2, 101, 102), 0), ((150, 1, 140), 0),
         ((128, 14, 13), 7), ((129, 12, 15), 1), ((65, 18, 20), 6), ((258, 9, 11), 3)]


def same_bits(a, b):
    return np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)])


@pytest.mark.parametrize("family", [P.FAM_Q1_ANISO, P.FAM_FACE7_UNIFORM])
@pytest.mark.parametrize("shape,prd", CASES)
def test_symmetric_sweeps_bitwise(shape, prd, family):
    m, n, o = shape
    assert m * n * o > 20000  # smaller levels take one workgroup
    print("case", shape, prd, family, flush=True)
    A = O.gen_operator(family, 5, m, n, o, prd=prd)
    b = O.gen_rhs(5, m, n, o)
    x = O.test_field(m, n, o, 3)
    bad = x.copy()
    bad[o // 2, n // 2, m // 2] = np.inf
    bad[0, 0, m - 1] = np.nan
    mg = O.Multigrid(A, colour8=True, prd=prd)
    mg.set_rhs(b)
    with P.Hierarchy(m, n, o, prd=prd) as h:
        h.set_operator27(A)
        h.set_rhs(b)
        for x0 in (x, bad):
            h.set_x(x0)
            mg.set_x(0, x0)
            for _ in range(2):
                h.gauss_seidel(1, 0)
                mg.gauss_seidel(1, 0)
                assert same_bits(h.get_x(), mg.get_x(0))

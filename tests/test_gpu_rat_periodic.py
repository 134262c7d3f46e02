"""Galerkin operators and restriction with periodic axes, interior and boundary
points: bit for bit the oracle's on every level, for each set of periodic axes,
odd and even sizes and axes too short for an interior."""
import numpy as np
import pytest

import pgmg_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [((33, 20, 14), p) for p in range(1, 8)] + [((21, 18, 17), 7), ((80, 70, 3), 3), ((2, 40, 41), 5), ((130, 1, 30), 6),
         ((5, 60, 6), 7), ((64, 61, 40), 2)]


@pytest.mark.parametrize("shape,prd", CASES)
def test_levels_bitwise(shape, prd):
    m, n, o = shape
    print("case", shape, prd, flush=True)
    A = O.gen_operator(P.FAM_Q1_ANISO, 5, m, n, o, prd=prd)
    b = O.gen_rhs(5, m, n, o)
    mg = O.Multigrid(A, prd=prd, colour8=True)
    with P.Hierarchy(m, n, o, prd=prd) as h:
        h.set_operator27(A)
        h.compute_rats()
        for level in range(1, h.nlevels):
            same = np.array_equal(h.get_operator27(level), mg.get_A(level))
            assert same, level
        h.set_rhs(b)
        x = O.test_field(m, n, o, 3)
        h.set_x(x)
        h.restriction(1)
        assert np.array_equal(h.get_rhs(1), O.restrict(A, x, b, h.dims[1], prd=prd))

"""Forward colour sweeps of small periodic levels in one launch each: bit for
bit the oracle's for each set of periodic axes, where tiles (4 rows x 2 planes)
end inside and outside the grid, odd and even rows, axes of one and two points,
one and two tiles to a CU, any number of sweeps, x holding infinities and NaN,
and in cycles."""
import numpy as np
import pytest

import pgmg_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

CASES = [((17, 17, 17), 7), ((20, 13, 11), 1), ((20, 14, 11), 2), ((9, 4, 40), 4), ((2, 33, 30), 7), ((1, 50, 40), 3),
         ((55, 1, 30), 6), ((40, 30, 1), 4), ((33, 34, 31), 5), ((24, 60, 64), 7), ((79, 5, 6), 7)]


def same_bits(a, b):
    return np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)])


@pytest.mark.parametrize("shape,prd", CASES)
def test_sweeps_bitwise(shape, prd):
    m, n, o = shape
    A = O.gen_operator(P.FAM_Q1_ANISO, 5, m, n, o, prd=prd)
    b = O.gen_rhs(5, m, n, o)
    x = O.test_field(m, n, o, 3)
    bad = x.copy()
    bad[o // 2, n // 2, m // 2] = np.inf
    bad[0, 0, m - 1] = np.nan
    with P.Hierarchy(m, n, o, prd=prd) as h:
        h.set_operator27(A)
        h.compute_rats()
        h.set_rhs(b)
        mg = O.Multigrid(A, colour8=True, prd=prd)
        mg.set_rhs(b)
        for x0 in (x, bad):
            mg.set_x(0, x0)
            for sweeps in (1, 2, 3, 4):
                print("case", shape, prd, sweeps, flush=True)
                h.set_x(x0)
                h.gauss_seidel(0, 0, sweeps)
                mg.gauss_seidel(0, 0)
                assert same_bits(h.get_x(), mg.get_x(0)), sweeps


@pytest.mark.parametrize("precision", [P.PREC_FP64, P.PREC_MIXED])
@pytest.mark.parametrize("v_down,v_up", [(2, 2), (1, 2), (2, 1), (0, 1)])
@pytest.mark.parametrize("dims,prd", [((34, 40, 27), 7), ((48, 46, 44), 3)])
def test_cycles_bitwise(precision, v_down, v_up, dims, prd):
    m, n, o = dims
    A = O.gen_operator(P.FAM_FACE7_UNIFORM, 8, m, n, o, prd=prd)
    A[..., 13] *= 1.001  # regular, also where every axis wraps
    b = O.gen_rhs(8, m, n, o)
    mg = O.Multigrid(A, colour8=True, v_down=v_down, v_up=v_up, prd=prd)
    mg.set_rhs(b)
    cycles, _ = mg.solve(1e-6, 8, mixed=precision == P.PREC_MIXED)
    with P.Hierarchy(m, n, o, precision=precision, v_down=v_down, v_up=v_up, prd=prd) as h:
        h.set_operator27(A)
        h.compute_rats()
        h.set_rhs(b)
        c, _ = h.solve(1e-6, 8, check=False)
        print("case", dims, prd, c, flush=True)
        assert c == cycles
        assert np.array_equal(h.get_x(), mg.get_x(0))

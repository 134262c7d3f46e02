"""Forward colour sweeps of small levels in one launch each: bit for bit the
oracle's sweeps where tiles (4 rows x 2 planes) end inside and outside the
grid, for odd and even rows, the shortest and longest rows that take them in
each precision, any number of sweeps (an odd number ends in the other array),
and x holding infinities and NaN."""
import numpy as np
import pytest

import pgmg_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(17, 17, 17), (20, 13, 11), (9, 4, 40), (11, 101, 1), (1200, 1, 1), (2, 33, 30), (1, 50, 40), (33, 33, 33),
          (55, 9, 7), (57, 8, 6), (79, 5, 6), (81, 6, 5), (33, 64, 32)]


def same_bits(a, b):
    return np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)])


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "%dx%dx%d" % s)
def test_sweeps_bitwise(shape):
    m, n, o = shape
    A = O.gen_operator(P.FAM_Q1_ANISO, 5, m, n, o)
    b = O.gen_rhs(5, m, n, o)
    x = O.test_field(m, n, o, 3)
    bad = x.copy()
    bad[o // 2, n // 2, m // 2] = np.inf
    bad[0, 0, m - 1] = np.nan
    with P.Hierarchy(m, n, o) as h:
        h.set_operator27(A)
        h.compute_rats()
        h.set_rhs(b)
        for x0 in (x, bad):
            for sweeps in (1, 2, 3, 4):
                print("case", shape, sweeps, flush=True)
                h.set_x(x0)
                h.gauss_seidel(0, 0, sweeps)
                mg = O.Multigrid(A, colour8=True)
                mg.set_rhs(b)
                mg.set_x(0, x0)
                for _ in range(sweeps):
                    mg.gauss_seidel(0, 0)
                assert same_bits(h.get_x(), mg.get_x(0)), sweeps


@pytest.mark.parametrize("precision", [P.PREC_FP64, P.PREC_MIXED])
@pytest.mark.parametrize("v_down,v_up", [(2, 2), (1, 2), (2, 1), (0, 1)])
def test_cycles_bitwise(precision, v_down, v_up):
    m, n, o = 34, 40, 27
    A = O.gen_operator(P.FAM_FACE7_UNIFORM, 8, m, n, o)
    b = O.gen_rhs(8, m, n, o)
    mg = O.Multigrid(A, colour8=True, v_down=v_down, v_up=v_up)
    mg.set_rhs(b)
    cycles, _ = mg.solve(1e-7, 40, mixed=precision == P.PREC_MIXED)
    with P.Hierarchy(m, n, o, precision=precision, v_down=v_down, v_up=v_up) as h:
        h.set_operator27(A)
        h.compute_rats()
        h.set_rhs(b)
        c, _ = h.solve(1e-7, 40)
        assert c == cycles
        assert np.array_equal(h.get_x(), mg.get_x(0))


@pytest.mark.parametrize("precision", [P.PREC_FP64, P.PREC_MIXED])
@pytest.mark.parametrize("v_down,v_up", [(2, 2), (1, 2), (3, 1), (0, 1)])
def test_batch_equals_alone(precision, v_down, v_up):
    # levels with and without tiles, of both workgroup sizes, at levels 0 to 2;
    # the second batch has too many tiles at a level for tile launches
    dims = [(34, 40, 27), (20, 13, 11), (65, 70, 40), (17, 17, 17), (79, 20, 18), (50, 49, 33)]
    for repeat in (1, 8):
        with P.Batch(1 << 31, max_slots=64, precision=precision, v_down=v_down, v_up=v_up) as batch:
            slots = [(d, batch.admit(*d, P.FAM_Q1_ANISO, 70 + q, 1e-6, 12)) for _ in range(repeat)
                     for q, d in enumerate(dims)]
            batch.run()
            for q, (d, s) in enumerate(slots):
                print("case", d, repeat, flush=True)
                with P.Hierarchy(*d, precision=precision, v_down=v_down, v_up=v_up) as h:
                    h.generate_problem(P.FAM_Q1_ANISO, 70 + q % len(dims))
                    h.compute_rats()
                    c, _ = h.solve(1e-6, 12, check=False)
                    assert batch.status(s)[1] == c
                    assert np.array_equal(batch.get_x(s), h.get_x())

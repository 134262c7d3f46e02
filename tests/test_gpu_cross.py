"""Operators that are a 7-point cross (every other entry zero) take kernels
that read 7 of the 27 coefficient planes.  They must give the bits of the
27-plane kernels for every x, infinities and NaN included: the same operator
with one entry outside the cross set to 1e-300 at one point (a term that
leaves that point's sum unchanged) takes the 27-plane kernels."""
import numpy as np
import pytest

import pgmg_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# levels of at least 65536 points: rows packed several to a wavefront, with
# and without a point out, one row to a wavefront, segmented rows (both
# precisions), every periodic axis
CASES = [((12, 75, 80), 0), ((33, 50, 41), 0), ((70, 31, 32), 0), ((129, 29, 19), 0), ((131, 22, 23), 0),
         ((257, 17, 16), 0), ((262, 15, 17), 0), ((517, 11, 13), 0), ((34, 46, 42), 7), ((129, 28, 19), 1),
         ((262, 16, 16), 6)]


def same_bits(a, b):
    return np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)])


def operations(m, n, o, prd, A, x, precision, b):
    """x after sweeps both ways, residual, product and norm; then a solve."""
    out = []
    with P.Hierarchy(m, n, o, precision=precision, prd=prd) as h:
        h.set_operator27(A)
        h.compute_rats()
        h.set_rhs(b)
        h.set_x(x)
        h.gauss_seidel(0, 0, 2)
        out.append(h.get_x())
        h.gauss_seidel(1, 0, 1)
        out += [h.get_x(), h.residual(), h.apply_operator(x), np.array([h.l2_error_all()])]
        h.clear_x()
        try:
            h.solve(1e-9, 3, check=False)
        except P.PgmgError as e:
            assert e.code == 12  # NaN, from an operator or source that holds one
        out.append(h.get_x())
    return out


@pytest.mark.parametrize("precision", [P.PREC_FP64, P.PREC_MIXED])
@pytest.mark.parametrize("dims,prd", CASES)
def test_cross_equals_27_planes(dims, prd, precision):
    m, n, o = dims
    print("case", dims, prd, precision, flush=True)
    A = O.gen_operator(P.FAM_FACE7_UNIFORM, 3, m, n, o, prd=prd)
    b = O.gen_rhs(3, m, n, o)
    A27 = A.copy()
    A27[o // 2, n // 2, m // 2, 0] = 1e-300
    x = O.test_field(m, n, o, 4)
    for spot in (None, np.inf, np.nan):
        xs = x.copy()
        if spot is not None:
            # away from the point whose entry differs, and on a row end
            xs[0, 0, m - 1] = spot
            xs[o - 1, n - 1, 1] = -spot
        for got, want in zip(operations(m, n, o, prd, A, xs, precision, b),
                             operations(m, n, o, prd, A27, xs, precision, b)):
            assert same_bits(got, want), spot


def test_operator_replaced_by_a_denser_one():
    m, n, o = 50, 37, 40
    seven, dense = (O.gen_operator(f, 5, m, n, o) for f in (P.FAM_FACE7_UNIFORM, P.FAM_Q1_ANISO))
    b = O.gen_rhs(5, m, n, o)
    with P.Hierarchy(m, n, o) as h:
        for A in (seven, dense, seven):
            h.set_operator27(A)
            h.compute_rats()
            h.set_rhs(b)
            h.clear_x()
            h.v_cycle()
            mg = O.Multigrid(A, colour8=True)
            mg.set_rhs(b)
            mg.v_cycle()
            assert np.array_equal(h.get_x(), mg.get_x(0))


@pytest.mark.parametrize("precision", [P.PREC_FP64, P.PREC_MIXED])
def test_batch_of_crosses_and_others_equals_alone(precision):
    dims = [(50, 37, 40), (129, 29, 19), (33, 50, 41), (20, 17, 30), (262, 15, 17), (50, 37, 40)]
    fams = [P.FAM_FACE7_UNIFORM, P.FAM_FACE7_LOGUNI, P.FAM_Q1_ANISO, P.FAM_FACE7_UNIFORM, P.FAM_FACE7_UNIFORM, P.FAM_Q1_ANISO]

    def alone(m, n, o, fam, seed):
        with P.Hierarchy(m, n, o, precision=precision) as h:
            h.generate_problem(fam, seed)
            h.compute_rats()
            c, _ = h.solve(1e-7, 12, check=False)
            return c, h.get_x()

    with P.Batch(1 << 31, max_slots=16, precision=precision) as batch:
        slots = [batch.admit(*d, f, 60 + q, 1e-7, 12) for q, (d, f) in enumerate(zip(dims, fams))]
        slots += [batch.admit_operator(O.gen_operator(f, 60 + q, *d), O.gen_rhs(60 + q, *d), 1e-7, 12)
                  for q, (d, f) in enumerate(zip(dims, fams))]
        batch.run()
        for q, (d, f) in enumerate(zip(dims, fams)):
            c, x = alone(*d, f, 60 + q)
            for s in (slots[q], slots[q + len(dims)]):
                assert batch.status(s)[1] == c, (d, f)
                assert np.array_equal(batch.get_x(s), x), (d, f)

"""Problems of one level whose point pairs do not fit a workgroup's wavefronts a
colour pair at a time, or not at all (one point along x): bit for bit the
oracle's, alone and in a batch, entries and values that are not finite among
them, and a batch's step of 900 points at most twice as long as one of 729."""
import time

import numpy as np
import pytest

import pgmg_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(1, 30, 30), (1, 32, 32), (1, 25, 31), (1, 1, 900), (1, 800, 1), (1, 1, 1000), (9, 9, 9), (1, 1, 3),
          (3, 5, 68), (3, 68, 5), (1, 24, 32), (1, 2, 400)]


@pytest.mark.parametrize("precision", [P.PREC_FP64, P.PREC_MIXED])
def test_batch_equals_oracle(precision):
    probs = [(O.gen_operator(P.FAM_Q1_ANISO, 20 + q, *s), O.gen_rhs(20 + q, *s)) for q, s in enumerate(SHAPES)]
    with P.Batch(1 << 28, max_slots=16, precision=precision) as batch:
        slots = [batch.admit_operator(A, b, 1e-8, 20) for A, b in probs]
        batch.run()
        for s, (A, b) in zip(slots, probs):
            mg = O.Multigrid(A, colour8=True)
            mg.set_rhs(b)
            cycles, _ = mg.solve(1e-8, 20, mixed=precision == P.PREC_MIXED)
            print("case", b.shape, cycles, flush=True)
            assert batch.status(s)[1] == cycles
            assert np.array_equal(batch.get_x(s), mg.get_x(0))


def same_bits(a, b):
    return np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)])


@pytest.mark.parametrize("shape,prd", [(s, 0) for s in SHAPES] + [((1, 154, 4), 6), ((1, 30, 30), 7), ((1, 9, 8), 1), ((1, 1, 700), 4),
                                                         ((244, 1, 2), 6), ((169, 6, 1), 6), ((20, 1, 13), 2)])
def test_sweeps_bitwise(shape, prd):
    m, n, o = shape
    print("case", shape, prd, flush=True)
    A, b = O.gen_operator(P.FAM_Q1_ANISO, 5, m, n, o, prd=prd), O.gen_rhs(5, m, n, o)
    x = O.test_field(m, n, o, 3)
    x[o // 2, n // 2, m // 2] = np.inf
    with P.Hierarchy(m, n, o, prd=prd) as h:
        h.set_operator27(A)
        h.set_rhs(b)
        h.set_x(x)
        h.gauss_seidel(0, 0, 2)
        mg = O.Multigrid(A, colour8=True, prd=prd)
        mg.set_rhs(b)
        mg.set_x(0, x)
        for _ in range(2):
            mg.gauss_seidel(0, 0)
        assert same_bits(h.get_x(), mg.get_x(0))


def test_batch_entry_outside_the_plane():
    # 1e200, infinite in FP32, meets the halo's 0: NaN in the first FP32 cycle,
    # as on a lone hierarchy
    m, n, o = 1, 30, 30
    A, b = O.gen_operator(P.FAM_Q1_ANISO, 5, m, n, o), O.gen_rhs(5, m, n, o)
    A[o // 2, n // 2, 0, 12] = 1e200
    with P.Batch(1 << 28, max_slots=1) as batch, P.Hierarchy(m, n, o, precision=P.PREC_MIXED) as h:
        s = batch.admit_operator(A, b, 1e-8, 3)
        batch.run()
        assert batch.status(s)[:2] == (P.SLOT_FAILED, 1)
        h.set_operator27(A)
        h.set_rhs(b)
        h.compute_rats()
        with pytest.raises(P.PgmgError):
            h.solve(1e-8, 3)
        assert np.isnan(h.get_x()).any()
        assert same_bits(batch.get_x(s), h.get_x())


def sweeps_time(shape, prd):
    best = 1e9
    with P.Hierarchy(*shape, prd=prd) as h:
        h.generate_problem(P.FAM_Q1_ANISO, 5)
        for _ in range(6):
            t = time.perf_counter()
            for _ in range(10):
                h.gauss_seidel(0, 0, 24)
            h.synchronize()
            best = min(best, (time.perf_counter() - t) / 10)
    return 1e6 * best


def test_periodic_sweeps_time():
    # 616 points, of one and of two along x, ghosts refreshed in each sweep
    print("start", flush=True)
    one, two = sweeps_time((1, 154, 4), 6), sweeps_time((2, 77, 4), 6)
    print("24 sweeps: 1x154x4 %.1f us, 2x77x4 %.1f us" % (one, two), flush=True)
    assert one < 1.05 * two


def test_periodic_plane_sweeps_time():
    # 488 points, one plane and two
    print("start", flush=True)
    one, two = sweeps_time((244, 1, 2), 6), sweeps_time((122, 2, 2), 6)
    print("24 sweeps: 244x1x2 %.1f us, 122x2x2 %.1f us" % (one, two), flush=True)
    assert one < 1.15 * two


def batch_time(shape, precision):
    best = 1e9
    with P.Batch(1 << 28, max_slots=16, precision=precision) as batch:
        for _ in range(4):
            slots = [batch.admit(*shape, P.FAM_Q1_ANISO, 20 + q, 1e-30, 60) for q in range(16)]
            t = time.perf_counter()
            batch.run()
            best = min(best, time.perf_counter() - t)
            for s in slots:
                batch.release(s)
    return best


@pytest.mark.parametrize("precision", [P.PREC_FP64, P.PREC_MIXED])
def test_batch_time(precision):
    flat, cube = batch_time((1, 30, 30), precision), batch_time((9, 9, 9), precision)
    print("16 problems, 60 cycles: 1x30x30 %.2f ms, 9x9x9 %.2f ms" % (1e3 * flat, 1e3 * cube), flush=True)
    assert flat < 2 * cube

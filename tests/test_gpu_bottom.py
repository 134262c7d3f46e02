"""Forward colour sweeps of levels of at most 1024 points by one workgroup, bit
for bit the oracle's: shapes whose point pairs take 8, 12 and more wavefronts
(the last on the one-point-a-thread kernel), a single point, lines and planes,
periodic axes, x holding infinities and NaN, alone and in a batch."""
import numpy as np
import pytest

import pgmg_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(9, 9, 9), (10, 10, 10), (8, 8, 16), (17, 6, 10), (5, 9, 13), (1, 1, 1), (1, 1, 900), (1000, 1, 1), (1, 32, 32),
          (32, 1, 32), (3, 18, 18), (2, 2, 2)]
PERIODIC = [((8, 6, 10), 7), ((9, 7, 5), 7), ((2, 9, 8), 1), ((12, 8, 9), 6)]


def same_bits(a, b):
    return np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)])


@pytest.mark.parametrize("shape,prd", [(s, 0) for s in SHAPES] + PERIODIC)
def test_sweeps_bitwise(shape, prd):
    m, n, o = shape
    print("case", shape, prd, flush=True)
    A = O.gen_operator(P.FAM_Q1_ANISO, 5, m, n, o, prd=prd)
    b = O.gen_rhs(5, m, n, o)
    x = O.test_field(m, n, o, 3)
    bad = x.copy()
    bad[o // 2, n // 2, m // 2] = np.inf
    with P.Hierarchy(m, n, o, prd=prd) as h:
        h.set_operator27(A)
        h.compute_rats()
        h.set_rhs(b)
        for x0 in (x, bad):
            for sweeps in (1, 3):
                h.set_x(x0)
                h.gauss_seidel(0, 0, sweeps)
                mg = O.Multigrid(A, colour8=True, prd=prd)
                mg.set_rhs(b)
                mg.set_x(0, x0)
                for _ in range(sweeps):
                    mg.gauss_seidel(0, 0)
                assert same_bits(h.get_x(), mg.get_x(0)), sweeps


@pytest.mark.parametrize("precision", [P.PREC_FP64, P.PREC_MIXED])
def test_batch_equals_oracle(precision):
    probs = []
    for q, (m, n, o) in enumerate(s for s in SHAPES if min(s) > 1):
        probs.append((O.gen_operator(P.FAM_FACE7_UNIFORM, 20 + q, m, n, o), O.gen_rhs(20 + q, m, n, o)))
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

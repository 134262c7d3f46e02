"""A small batch of 7-point and 27-point problems shares its launches: it takes no
longer than one of the same grids with 27 points alone, and keeps each lone
solve's bits, with few and with many 7-point problems."""
import time

import numpy as np
import pytest

import pgmg_amd as P

pytestmark = pytest.mark.gpu


def batch(problems, precision, cycles, reps=1):
    need = sum(P.footprint(*p[:3], precision=precision) for p in problems)
    best = 1e9
    with P.Batch(int(1.1 * need) + (64 << 20), max_slots=len(problems), precision=precision) as b:
        for _ in range(reps):
            slots = [b.admit(*p, 1e-30, cycles) for p in problems]
            t = time.perf_counter()
            b.run()
            best = min(best, time.perf_counter() - t)
            xs = [b.get_x(s) for s in slots]
            for s in slots:
                b.release(s)
    return best, xs


def test_time():
    print("start", flush=True)
    both, _ = batch([(65, 65, 65, P.FAM_FACE7_UNIFORM, 3), (65, 65, 65, P.FAM_Q1_ANISO, 4)], P.PREC_MIXED, 25, 5)
    dense, _ = batch([(65, 65, 65, P.FAM_Q1_ANISO, 3), (65, 65, 65, P.FAM_Q1_ANISO, 4)], P.PREC_MIXED, 25, 5)
    print("7 and 27 points %.2f ms, 27 points %.2f ms" % (1e3 * both, 1e3 * dense), flush=True)
    assert both < 1.13 * dense


@pytest.mark.parametrize("precision", [P.PREC_FP64, P.PREC_MIXED])
@pytest.mark.parametrize("count", [1, 5])
def test_bits(count, precision):
    cycles = 6
    problems = [(65, 66, 64, P.FAM_FACE7_UNIFORM, q) for q in range(count)] + [(41, 50, 40, P.FAM_Q1_ANISO, 9), (9, 8, 7, P.FAM_Q1_ANISO, 9)]
    _, xs = batch(problems, precision, cycles)
    for p, x in zip(problems, xs):
        print("case", count, precision, p, flush=True)
        with P.Hierarchy(*p[:3], precision=precision) as h:
            h.generate_problem(*p[3:])
            h.compute_rats()
            h.solve(1e-30, cycles, check=False)
            assert np.array_equal(x, h.get_x())

"""pgmg_clear_x returns when the level's x is clear: what was queued before it,
and its own fill, are complete (and their errors reported by it)."""
import time

import pytest

import pgmg_amd as P

pytestmark = pytest.mark.gpu


def test_clear_x_waits():
    with P.Hierarchy(161, 130, 147) as h:
        h.generate_problem(P.FAM_Q1_ANISO, 3)
        h.gauss_seidel(0, 0)
        h.synchronize()
        print("sweeps", flush=True)
        h.gauss_seidel(0, 0, 200)  # tens of milliseconds, queued in a few
        t0 = time.perf_counter()
        h.clear_x(0)
        t1 = time.perf_counter()
        h.synchronize()
        t2 = time.perf_counter()
        assert t2 - t1 < 0.1 * (t1 - t0)
        assert not h.get_x(0).any()

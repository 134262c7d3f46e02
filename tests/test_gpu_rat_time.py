"""Set-up of small levels with periodic axes takes no longer for its launches: the
first coarse operator of 32^3, all axes periodic, against the same grid without
(one launch of the wrapped form against two)."""
import time

import pytest

import pgmg_amd as P

pytestmark = pytest.mark.gpu


def rats(prd):
    best = 1e9
    with P.Hierarchy(32, 32, 32, prd=prd, max_levels=2) as h:
        h.generate_problem(P.FAM_Q1_ANISO, 5)
        for _ in range(20):
            t = time.perf_counter()
            h.compute_rats()
            best = min(best, time.perf_counter() - t)
    return 1e6 * best


def test_small_periodic_setup_time():
    print("start", flush=True)
    periodic, plain = rats(7), rats(0)
    print("32^3: periodic %.0f us, not %.0f us" % (periodic, plain), flush=True)
    assert periodic < 1.6 * plain

"""Calls of very small systems, whose time is launches, waits and allocations:
an operator's upload takes no work that only larger levels have a use for, and
a new hierarchy's first read-out allocates nothing.  Each against a call of the
same hierarchy that does as much."""
import time

import numpy as np
import pytest

import pgmg_amd as P

pytestmark = pytest.mark.gpu


def timed(call):
    t = time.perf_counter()
    call()
    return time.perf_counter() - t


def test_operator_upload():
    with P.Hierarchy(5, 5, 5) as h:
        h.generate_problem(P.FAM_Q1_ANISO, 1)
        A, b = h.get_operator27(0), h.get_rhs()
        print("start", flush=True)
        op = np.median([timed(lambda: h.set_operator27(A)) for _ in range(100)])
        rhs = np.median([timed(lambda: h.set_rhs(b)) for _ in range(100)])
        print("operator %.1f us, source %.1f us" % (1e6 * op, 1e6 * rhs), flush=True)
        # the same transfer, packing and wait, and the launch of the tail copies
        assert op < 2.35 * rhs


def test_first_readout():
    first, second = [], []
    print("start", flush=True)
    for _ in range(30):
        with P.Hierarchy(9, 9, 9) as h:
            h.synchronize()
            first.append(timed(h.get_x))
            second.append(timed(h.get_x))
    print("first %.1f us, second %.1f us" % (1e6 * np.median(first), 1e6 * np.median(second)), flush=True)
    assert np.median(first) < 1.6 * np.median(second)

"""Periodic levels large enough for the launches of their own that interior
points get there, against the oracle: Galerkin operators from 16384 coarse
points on (each set of periodic axes, bit for bit) and with a thread a point
(131072 interior ones: index by index with an operator whose sums are exact, and
the order of the sums on boxes cut out of the grid), and restriction with the
shell as a launch of its own (100000 coarse points)."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import pgmg_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def level1(h, A):
    h.set_operator27(A)
    h.compute_rats()
    return h.get_operator27(1)


def test_galerkin_each_periodic_set():
    m, n, o = 53, 52, 56
    A = {prd: O.gen_operator(P.FAM_Q1_ANISO, 5, m, n, o, prd=prd) for prd in range(1, 8)}
    dims = {prd: P.hierarchy_shape(m, n, o, prd)[1] for prd in A}
    with ThreadPoolExecutor(7) as pool:
        want = dict(zip(A, pool.map(lambda prd: O.rat(A[prd], dims[prd], prd=prd), A)))
    for prd in A:
        print("case", prd, dims[prd], flush=True)
        assert np.prod(dims[prd]) >= 16384
        with P.Hierarchy(m, n, o, prd=prd, max_levels=2) as h:
            assert np.array_equal(level1(h, A[prd]), want[prd])


def test_galerkin_thread_a_point():
    small, times = (16, 12, 10), (7, 9, 11)
    m, n, o = (s * t for s, t in zip(small, times))
    rng = np.random.default_rng(3)
    tile = rng.integers(-512, 512, size=(small[2], small[1], small[0], 27)).astype(np.float64)
    A = np.tile(tile, (times[2], times[1], times[0], 1))
    coarse = tuple(s // 2 for s in small)
    want = np.tile(O.rat(tile, coarse, prd=7), (times[2], times[1], times[0], 1))
    print("case", (m, n, o), flush=True)
    with P.Hierarchy(m, n, o, prd=7, max_levels=2) as h:
        assert np.prod([c - 2 for c in h.dims[1]]) >= 131072
        assert np.array_equal(level1(h, A), want)
    # a box of even offset has the grid's own coarse entries where no sum
    # reaches its edge
    h = P.Hierarchy(m, n, o, prd=5, max_levels=2)
    h.generate_problem(P.FAM_Q1_ANISO, 7)
    h.compute_rats()
    A, Ac = h.get_operator27(0), h.get_operator27(1)
    h.close()
    for i, j, k in ((2, 2, 2), (40, 52, 46), (90, 86, 88)):
        box = np.ascontiguousarray(A[k:k + 20, j:j + 20, i:i + 20])
        got = Ac[k // 2 + 2:k // 2 + 8, j // 2 + 2:j // 2 + 8, i // 2 + 2:i // 2 + 8]
        assert np.array_equal(got, O.rat(box, (10, 10, 10), prd=7)[2:8, 2:8, 2:8])


@pytest.mark.parametrize("shape,prd", [((96, 80, 112), 7), ((97, 82, 110), 5), ((94, 96, 101), 2)])
def test_restriction_shell(shape, prd):
    m, n, o = shape
    print("case", shape, prd, flush=True)
    b, x = O.gen_rhs(5, m, n, o), O.test_field(m, n, o, 3)
    with P.Hierarchy(m, n, o, prd=prd, max_levels=2) as h:
        assert np.prod(h.dims[1]) >= 100000
        h.generate_problem(P.FAM_FACE7_UNIFORM, 5)
        h.set_rhs(b)
        h.set_x(x)
        h.restriction(1)
        assert np.array_equal(h.get_rhs(1), O.restrict(h.get_operator27(0), x, b, h.dims[1], prd=prd))
        assert not h.get_x(1).any()

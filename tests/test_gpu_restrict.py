"""Restriction from and onto grid edges, bit for bit the oracle's: odd and even
extents on every axis (an even axis injects its last cube), axes of one and two
points, fine values of infinity and NaN next to the edge (a clamped load that
belongs to no term must not reach the sum), and a coarse level large enough
for the shell to be a launch of its own."""
import numpy as np
import pytest

import pgmg_amd as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(11, 12, 13), (12, 11, 14), (16, 16, 16), (17, 17, 17), (2, 40, 21), (40, 2, 21), (21, 40, 2), (1, 60, 31),
          (60, 1, 31), (31, 60, 1), (3, 4, 100), (94, 95, 98)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "%dx%dx%d" % s)
def test_restriction_bitwise(shape):
    m, n, o = shape
    print("case", shape, flush=True)
    A = O.gen_operator(P.FAM_FACE7_UNIFORM, 5, m, n, o)
    b = O.gen_rhs(5, m, n, o)
    bad = b.copy()
    bad[o - 1, n - 1, m - 1] = np.inf
    bad[0, n // 2, 0] = np.nan
    x = O.test_field(m, n, o, 3)
    with P.Hierarchy(m, n, o) as h:
        h.set_operator27(A)
        h.compute_rats()
        for rhs in (b, bad):
            h.set_rhs(rhs)
            h.set_x(x)
            h.restriction(1)
            mg = O.Multigrid(A)
            mg.set_rhs(rhs)
            mg.set_x(0, x)
            mg.restriction(1)
            got, want = h.get_rhs(1), mg.get_r(1)
            assert np.array_equal(np.isnan(got), np.isnan(want))
            assert np.array_equal(got[~np.isnan(got)], want[~np.isnan(want)])
            assert not h.get_x(1).any()

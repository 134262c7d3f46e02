"""Level vectors to host arrays in chunks: fewer points than a chunk, chunk
edges, more chunks than the buffer holds, growing and shrinking sizes on one
hierarchy and calls from several threads."""
import threading

import numpy as np
import pytest

import pgmg_amd as P

pytestmark = pytest.mark.gpu

CHUNK = 1 << 17
SHAPES = [(5, 3, 4), (64, 64, 32), (64, 64, 33), (127, 129, 8), (128, 128, 32), (131, 128, 40), (128, 128, 128 + 5), (257, 130, 71)]


@pytest.mark.parametrize("shape", SHAPES)
def test_round_trip(shape):
    print("case", shape, shape[0] * shape[1] * shape[2] / CHUNK, flush=True)
    rng = np.random.default_rng(3)
    with P.Hierarchy(*shape) as h:
        for level in [len(h.dims) - 1, 0, len(h.dims) - 1, 0]:
            x = rng.standard_normal(h.shape(level))
            h.set_x(x, level)
            assert np.array_equal(h.get_x(level), x)


def test_threads():
    rng = np.random.default_rng(4)
    with P.Hierarchy(128, 128, 67) as h:
        x, b = rng.standard_normal(h.shape(0)), rng.standard_normal(h.shape(0))
        h.set_x(x)
        h.set_rhs(b)
        wrong = []

        def read(get, want):
            for _ in range(4):
                if not np.array_equal(get(0), want):
                    wrong.append(get)

        ts = [threading.Thread(target=read, args=a) for a in [(h.get_x, x), (h.get_rhs, b), (h.get_x, x)]]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not wrong

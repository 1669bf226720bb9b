"""Modular reduction at its edges: products, sums and differences of values next
to 0, 2^32 and p through a two-row transform whose weights are chosen, against
big integers (exact, and canonical as stored)."""
import random

import numpy as np
import pytest

from lambda_vm_amd import workload

pytestmark = pytest.mark.gpu
P = workload.P
EPS = (1 << 32) - 1
EDGES = sorted({v % P for e in (0, 1, 2, EPS, EPS + 1, 2 * EPS, 1 << 63, P - EPS, P - EPS - 1, P - (1 << 31), P // 2,
                                (1 << 48), (EPS << 32) % P, 0x80000000, 0xFFFFFFFE00000001)
                for v in (e - 1, e, e + 1)})


@pytest.mark.parametrize("seed", range(6))
def test_two_row_transform_at_edges(gpu, seed):
    rng = random.Random(seed)
    m = 600
    draw = lambda: rng.choice(EDGES) if rng.random() < 0.8 else rng.randrange(P)  # noqa: E731
    a, b = [draw() for _ in range(m)], [draw() for _ in range(m)]
    # the inverse transform of two rows is (a + b, a - b); weights (w0, w1) then the forward one
    w0, w1 = draw(), draw()
    h = gpu.coset_lde_dev(gpu.DeviceBuffer.from_array(np.array([a, b], dtype=np.uint64)), 2, m, 1,
                          gpu.DeviceBuffer.from_array(np.array([w0, w1], dtype=np.uint64)))
    got = h.download()
    for c in range(m):
        x, y = (a[c] + b[c]) * w0 % P, (a[c] - b[c]) * w1 % P
        assert [int(got[0, c]), int(got[1, c])] == [(x + y) % P, (x - y) % P], (a[c], b[c], w0, w1)

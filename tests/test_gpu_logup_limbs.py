"""LogUp over words in [p, 2^64) and the same residues below p give the same aux
trace and contribution, at row counts that end inside a thread's four rows."""
import random

import numpy as np
import pytest

from lambda_vm_amd import air, workload

pytestmark = pytest.mark.gpu
P = np.uint64(workload.P)


def canon(a):
    return np.where(a >= P, a - P, a)


@pytest.mark.parametrize("n", [1, 5, 1023, 4098])
def test_words_above_p(gpu, n):
    rng = np.random.default_rng(n)
    desc = air.descriptor(air.logup_air(24, air.four_bus_interactions()))
    low = rng.integers(0, (1 << 32) - 1, size=(n, 24), dtype=np.uint64)
    r = random.Random(n)
    fp3 = lambda: [r.randrange(workload.P) for _ in range(3)]  # noqa: E731
    z, alpha = fp3(), gpu.fp3_powers(fp3(), desc.alpha_powers_len)
    got = []
    for tr in (low, low + P):
        aux, L, _ = gpu.logup_aux_dev(gpu.DeviceBuffer.from_array(tr), n, 24, desc, alpha, z)
        got.append((canon(aux.to_array(np.uint64, (n, desc.num_out_cols, 3))), [x % workload.P for x in L]))
    assert np.array_equal(got[0][0], got[1][0]) and got[0][1] == got[1][1]

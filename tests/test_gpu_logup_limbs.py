"""LogUp over words in [p, 2^64) and the same residues below p give the same aux
trace and contribution, at row counts that end inside a thread's four rows; zero
fingerprints against big integers (exact)."""
import random

import numpy as np
import pytest

import pyref
from lambda_vm_amd import air, logup, workload

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


@pytest.mark.parametrize("buses", [1, 4])  # one output column, and columns shared out over slices
@pytest.mark.parametrize("n,hits", [(9, [(0, 2)]), (9, [(1, 8)]), (11, [(0, 4), (1, 4)]), (12, [(1, 3), (1, 9)])])
def test_zero_fingerprint_leaves_out_its_own_interaction(gpu, buses, n, hits):
    """A fingerprint of zero has no inverse: its interaction adds nothing to the
    four rows inverted together, every other term is what the formula gives."""
    desc = logup.build_fingerprint_descriptor(air.four_bus_interactions()[:2 * buses])
    tr = np.random.default_rng(n).integers(0, workload.P, size=(n, 24), dtype=np.uint64)
    r = random.Random(n + buses)
    alpha = gpu.fp3_powers([r.randrange(workload.P) for _ in range(3)], desc.alpha_powers_len)

    def linear(coef, col, lo, hi, v, row):
        return (int(v) + sum(int(coef[t]) * int(tr[row, col[t]]) for t in range(lo, hi))) % workload.P

    def combination(k, row):
        lc = [int(desc.bus_ids[k]), 0, 0]
        for e in range(desc.elem_offsets[k], desc.elem_offsets[k + 1]):
            base = linear(desc.term_coef, desc.term_col, desc.term_offsets[e], desc.term_offsets[e + 1],
                          desc.elem_const[e], row)
            lc = pyref.f3add(lc, pyref.f3scale(alpha[desc.elem_alpha_idx[e]], base))
        return lc

    # the interactions hit share one combination, and z is its value
    k0, i0 = hits[0]
    for k, i in hits[1:]:
        for w in range(2):
            tr[i, (8 if k else 0) + w] = tr[i0, (8 if k0 else 0) + w]
    z = combination(k0, i0)
    want = np.zeros((desc.num_out_cols, n, 3), dtype=np.uint64)
    for c in range(desc.num_out_cols):
        for ki in range(desc.out_col_offsets[c], desc.out_col_offsets[c + 1]):
            k = int(desc.out_col_interactions[ki])
            fps = [pyref.f3sub(z, combination(k, i)) for i in range(n)]
            for i in range(n):
                if any(f == [0, 0, 0] for f in fps[i & ~3:(i & ~3) + 4]):
                    continue
                m = linear(desc.mult_term_coef, desc.mult_term_col, desc.mult_term_offsets[k],
                           desc.mult_term_offsets[k + 1], desc.mult_const[k], i)
                want[c, i] = pyref.f3add(want[c, i], pyref.f3scale(pyref.f3inv(fps[i]), m))
    assert all(pyref.f3sub(z, combination(k, i)) == [0, 0, 0] for k, i in hits)
    aux, L, terms = gpu.logup_aux_dev(gpu.DeviceBuffer.from_array(tr), n, 24, desc, alpha, z, want_terms=True)
    assert np.array_equal(canon(terms.to_array(np.uint64, want.shape)), want)
    got = canon(aux.to_array(np.uint64, (n, desc.num_out_cols, 3)))
    assert np.array_equal(got[:, :-1], want[:-1].transpose(1, 0, 2))
    assert [x % workload.P for x in L] == [int(want[:, :, q].astype(object).sum()) % workload.P for q in range(3)]

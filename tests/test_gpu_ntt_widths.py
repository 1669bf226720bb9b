"""Coset LDE at the widths where a pass's 16-word windows span one, two, four or
more rows, whole and ragged runs, and block counts at which the cosets are shared
out: per table and batched, every LDE word against the oracle (canonical, exact)."""
import numpy as np
import pytest

from lambda_vm_amd import workload

pytestmark = pytest.mark.gpu
P = np.uint64(workload.P)


def canon(a):
    return np.where(a >= P, a - P, a)


@pytest.mark.parametrize("m", [1, 2, 3, 4, 6, 7, 9, 12, 15, 20, 33, 48, 83])
@pytest.mark.parametrize("log_n,blowup", [(1, 4), (2, 1), (4, 2), (7, 8), (9, 4), (11, 2), (13, 4)])
def test_lde_matches_oracle(gpu, ora, m, log_n, blowup):
    n = 1 << log_n
    tr = workload.trace_table(31, m, n, m)
    want, nodes = ora.lde_commit(tr, blowup, 3)
    d, w = gpu.DeviceBuffer.from_array(tr), gpu.coset_weights_dev(n, 3)
    h = gpu.coset_lde_dev(d, n, m, blowup, w)
    got = h.download()
    assert np.array_equal(got, canon(want))  # stored canonical
    assert h.root == nodes[0].tobytes()
    # beside tables of the other window classes
    others = [(m2, gpu.splitmix_table_dev(n, m2, 3, m2)) for m2 in (2, 6, 16, 21)]
    roots, hs = gpu.batch_lde_commit([(d, w, n, m, blowup)] + [(t, w, n, m2, blowup) for m2, t in others])
    assert roots[0] == h.root
    assert np.array_equal(hs[0].download(), got)
    for (m2, t), r in zip(others, roots[1:]):
        assert gpu.coset_lde_dev(t, n, m2, blowup, w).root == r
    x = gpu.ntt_forward(tr)
    assert np.array_equal(canon(x), canon(ora.fft_two_half(tr)))
    assert np.array_equal(canon(gpu.ntt_inverse(tr)), canon(ora.fft_two_half(tr, inverse=True)))

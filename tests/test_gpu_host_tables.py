"""Host tables in and out through the page-locked ring (512 KiB slots, 8 of
them): below a slot, at its edge, words past it, more slots than the ring has,
a row longer than a slot. Natural-order rows, tree and a second copy out,
against the oracle (whole numbers, exact)."""
import threading

import numpy as np
import pytest

from lambda_vm_amd import workload

pytestmark = pytest.mark.gpu
P = np.uint64(workload.P)


def _canon(a):
    return np.where(a >= P, a - P, a)


@pytest.mark.parametrize("n,m,blowup", [(2, 1, 1), (64, 3, 2), (4096, 8, 2), (4096, 17, 2), (16384, 5, 4),
                                        (8192, 33, 4), (2, 70000, 2), (1 << 15, 21, 2)])
def test_rows_match_oracle(gpu, ora, n, m, blowup):
    tr = workload.trace_table(31, m, n, m)
    want_lde, want_nodes = ora.lde_commit(tr, blowup, 7)
    w = gpu.coset_weights_dev(n, 7).to_array(np.uint64, (n,))
    h, rows = gpu.coset_lde_row_major_with_merkle_tree_keep(tr, n, m, blowup, w)
    assert h.root == want_nodes[0].tobytes()
    assert np.array_equal(_canon(rows), _canon(want_lde))
    assert np.array_equal(h.download(), rows)
    h2, none = gpu.coset_lde_row_major_with_merkle_tree_keep(tr, n, m, blowup, w, retain_host_lde=False)
    assert none is None and h2.root == h.root


def test_threads_have_their_own_slots(gpu):
    """Four threads with different tables at once, each result as alone."""
    n, m, blowup = 1 << 13, 40, 2  # 5 MiB out: every slot is used again
    w = gpu.coset_weights_dev(n, 7).to_array(np.uint64, (n,))
    traces = [workload.trace_table(33, t, n, m) for t in range(4)]
    alone = [gpu.coset_lde_row_major_with_merkle_tree_keep(t, n, m, blowup, w)[1] for t in traces]
    got = [None] * 4

    def work(i):
        got[i] = gpu.coset_lde_row_major_with_merkle_tree_keep(traces[i], n, m, blowup, w)[1]

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, g in zip(alone, got):
        assert np.array_equal(a, g)

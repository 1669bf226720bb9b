"""Batches of small tables on both sides of the sum of leaves (2^15) up to which
they are hashed one permutation per 16 lanes, alone and beside a table of more
than 2^13 leaves: roots and trees as for each table by itself."""
import numpy as np
import pytest

from lambda_vm_amd import workload

pytestmark = pytest.mark.gpu


# rows of the tables, at blowup 2 (a table of n rows has n leaves)
@pytest.mark.parametrize("rows", [[8192] * 4, [8192] * 4 + [2], [4096] * 8, [8192] * 3 + [4096, 2048, 1024, 1024],
                                  [2, 64, 8192, 16384], [8192] * 5 + [16384]])
def test_batch_trees_match_single_tables(gpu, rows):
    tables = []
    for t, n in enumerate(rows):
        m = 3 + 9 * (t % 3)
        tables.append((gpu.DeviceBuffer.from_array(workload.trace_table(41, t, n, m)), gpu.coset_weights_dev(n, 7),
                       n, m, 2))
    singles = [gpu.coset_lde_dev(tr, n, m, b, w) for tr, w, n, m, b in tables]
    plan = gpu.BatchPlan(tables, use_graph=True)
    want = [h.root for h in singles]
    assert plan.run() == want and plan.run() == want
    plan.close()
    roots, handles = gpu.batch_lde_commit(tables)
    assert roots == want
    for h, s in zip(handles, singles):
        assert np.array_equal(h.nodes(), s.nodes())


# (rows, blowup): five tables of 2^13 leaves (past the sum) beside tables of two
# leaves, of one leaf (its own root) and of one column
@pytest.mark.parametrize("shapes", [[(8192, 2)] * 5 + [(2, 1)], [(2, 1)] + [(8192, 2)] * 5 + [(2, 2), (2, 1), (4, 1)],
                                    [(16384, 4), (2, 1)], [(2, 1)]])
def test_one_leaf_tables(gpu, shapes):
    tables = [(gpu.DeviceBuffer.from_array(workload.trace_table(43, t, n, 1 + t % 3)), gpu.coset_weights_dev(n, 7), n,
               1 + t % 3, b) for t, (n, b) in enumerate(shapes)]
    want = [gpu.coset_lde_dev(tr, n, m, b, w).root for tr, w, n, m, b in tables]
    for graph in (True, False):
        plan = gpu.BatchPlan(tables, use_graph=graph)
        assert plan.run() == want and plan.run() == want
        assert [plan.take(t).root for t in range(len(tables))] == want
        plan.close()
    roots, handles = gpu.batch_lde_commit(tables)
    assert roots == want
    for h, root in zip(handles, roots):
        assert h.nodes()[0].tobytes() == root and h.root == root

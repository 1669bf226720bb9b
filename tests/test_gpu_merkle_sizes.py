"""Merkle trees at the sizes where the level kernels change: single blocks and
remainders of the 16-lanes-per-node tree top, its threshold, and the wide
levels above it. Every node against the oracle (bytes, exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num", [2, 4, 8, 16, 63, 64, 65, 128, 2048, 4096, 8192, 16383, 16384, 16385, 32768, 32769,
                                 65536, 131072])
def test_tree_matches_oracle_at_kernel_edges(gpu, ora, num):
    leaves = np.random.default_rng(num).integers(0, 256, size=(num, 32), dtype=np.uint8)
    assert np.array_equal(gpu.build_merkle_tree(leaves), ora.merkle_build(leaves))


# (rows, columns, blowup): one leaf, blocks of fewer than 32 leaves, the edge of
# the small-table kernel (2^13 leaves) and the first size past it; 2m = 16, 17*2,
# 50 = 2*17 + 16 and 2 words (padding in the last, a fresh and the first block)
@pytest.mark.parametrize("n,m,blowup", [(2, 1, 1), (2, 8, 2), (4, 17, 4), (32, 25, 2), (64, 17, 1), (256, 9, 8),
                                        (4096, 8, 4), (4096, 25, 4), (8192, 17, 2), (8192, 5, 4), (4096, 34, 8)])
def test_commitment_nodes_at_leaf_kernel_edges(gpu, ora, n, m, blowup):
    from lambda_vm_amd import workload
    tr = workload.trace_table(21, n, n, m)
    want_lde, want_nodes = ora.lde_commit(tr, blowup, 7)
    d, w = gpu.DeviceBuffer.from_array(tr), gpu.coset_weights_dev(n, 7)
    h = gpu.coset_lde_dev(d, n, m, blowup, w)
    assert np.array_equal(h.nodes(), want_nodes)
    assert gpu.batch_lde_commit([(d, w, n, m, blowup), (d, w, n, m, blowup)])[0] == [h.root, h.root]
    if m > 1:  # two trees over column ranges of one LDE
        split = m // 2
        hs, pre_root, pre_nodes = gpu.coset_lde_split_trees_dev(d, n, m, blowup, w, split)
        assert pre_root == pre_nodes[0].tobytes()
        P = np.uint64(workload.P)
        br = [int(format(i, "0%db" % (n * blowup).bit_length())[:0:-1] or "0", 2) for i in range(n * blowup)]
        rows = np.where(want_lde >= P, want_lde - P, want_lde)[br]
        for nodes, cols in ((pre_nodes, rows[:, :split]), (hs.nodes(), rows[:, split:])):
            L = n * blowup // 2
            for i in sorted({0, 1 % L, L // 2, L - 1}):
                msg = np.ascontiguousarray(cols[2 * i:2 * i + 2]).astype(">u8").tobytes()
                assert nodes[L - 1 + i].tobytes() == ora.keccak256(msg)

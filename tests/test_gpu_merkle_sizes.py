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

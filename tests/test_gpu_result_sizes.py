"""Openings and FRI answers on both sides of the 64 KiB up to which the kernels
write them to host memory themselves, and well past it: each answer as from a
call for its position alone, openings also against the table's own rows and
nodes (bytes, exact)."""
import numpy as np
import pytest

from lambda_vm_amd import workload

pytestmark = pytest.mark.gpu


# one position's answer is 11 * 32 + 16 m bytes at 2^11 leaves: 64 of 1024 bytes
# (m = 42) are exactly 64 KiB
@pytest.mark.parametrize("m,count", [(42, 1), (42, 63), (42, 64), (42, 65), (1, 300), (600, 20)])
def test_openings(gpu, ora, m, count):
    n, blowup = 1 << 11, 2
    h = gpu.coset_lde_dev(gpu.DeviceBuffer.from_array(workload.trace_table(51, m, n, m)), n, m, blowup,
                          gpu.coset_weights_dev(n, 7))
    pos = np.random.default_rng(count).integers(0, n, count).astype(np.uint64)
    paths, rows = h.open(pos)
    lde, nodes = h.download(), h.nodes()
    rev = [int(format(i, "012b")[::-1], 2) for i in range(2 * n)]
    for k, p in enumerate(pos.tolist()):
        assert np.array_equal(rows[k], lde[[rev[2 * p], rev[2 * p + 1]]])
        assert np.array_equal(paths[k], ora.merkle_path(nodes, p))


@pytest.mark.parametrize("count", [1, 30, 40, 200])
def test_fri_answers(gpu, count):
    # the layers of 2^11, 2^10, ... points answer 24 + 32 * (10, 9, ...) bytes a position, 1.9 KB in all
    h = gpu.GpuFri(np.random.default_rng(5).integers(0, workload.P, size=(1 << 12, 3), dtype=np.uint64), 7)
    h.commit_phase(gpu.Transcript(b"sizes"), 2, 1)
    iotas = np.random.default_rng(count).integers(0, 1 << 11, count).astype(np.uint64)
    sym, paths = h.query(iotas)
    for k in sorted({0, count // 2, count - 1}):
        s1, p1 = h.query(iotas[k:k + 1])
        assert np.array_equal(sym[:, k], s1[:, 0])
        assert all(np.array_equal(a[k], b[0]) for a, b in zip(paths, p1))
    for i in range(h.num_layers()):
        ev, nodes = h.layer(i)
        assert np.array_equal(sym[i], ev[(iotas >> np.uint64(i)) ^ np.uint64(1)])
    h.close()


def test_more_openings_than_a_grid_has_blocks(gpu):
    """2^24 positions of a block of 256 threads are 2^32 threads, more than one
    launch takes; a table of four leaves, every answer from its own rows and nodes."""
    m, L, count = 1, 4, (1 << 24) + 5
    h = gpu.coset_lde_dev(gpu.DeviceBuffer.from_array(workload.trace_table(53, m, L, m)), L, m, 2,
                          gpu.coset_weights_dev(L, 7))
    pos = np.random.default_rng(1).integers(0, L, count).astype(np.uint64)
    want_paths, want_rows = h.open(np.arange(L, dtype=np.uint64))
    paths, rows = h.open(pos)
    assert np.array_equal(rows, want_rows[pos]) and np.array_equal(paths, want_paths[pos])


def test_more_queries_than_a_grid_has_blocks(gpu):
    """2^25 queries of a block of 128 threads, on one committed layer of four values."""
    h = gpu.GpuFri(np.random.default_rng(6).integers(0, workload.P, size=(8, 3), dtype=np.uint64), 7)
    h.fold_and_commit_layer([3, 5, 7])
    iotas = np.random.default_rng(2).integers(0, 4, (1 << 25) + 5).astype(np.uint64)
    want_sym, want_paths = h.query(np.arange(4, dtype=np.uint64))
    sym, paths = h.query(iotas)
    assert len(paths) == 1 and np.array_equal(sym[0], want_sym[0][iotas])
    assert np.array_equal(paths[0], want_paths[0][iotas])
    h.close()

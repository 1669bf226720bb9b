"""Host tables in and out through the page-locked ring (512 KiB slots, 8 of
them): below a slot, at its edge, words past it, more slots than the ring has,
a row longer than a slot. Natural-order rows, tree and a second copy out,
against the oracle (whole numbers, exact)."""
import ctypes as C
import threading

import numpy as np
import pytest

from lambda_vm_amd import _native, workload

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


class _Locked:
    """Page-locked memory of the library's own HIP runtime as a uint64 array."""

    def __init__(self, words):
        self.p = C.c_void_p()
        assert _native.lib().hipHostMalloc(C.byref(self.p), C.c_size_t(words * 8), C.c_uint(0)) == 0
        self.a = np.ctypeslib.as_array((C.c_uint64 * words).from_address(self.p.value))

    def free(self):
        assert _native.lib().hipHostFree(self.p) == 0


def _ring_use(gpu, f):
    """Slots that a call moved each way through the ring."""
    gpu.prof_reset()
    gpu.prof_enable(True)
    f()
    gpu.prof_enable(False)
    return tuple(gpu.prof_query(nm)[0] for nm in ("host_ring_in", "host_ring_out"))


def _commit(tr, n, m, blowup, w, out):
    root, h = np.zeros(32, dtype=np.uint8), C.c_void_p()
    _native.call("lvm_coset_lde_row_major_with_merkle_tree_keep", tr, n, m, blowup, w, out,
                 root.ctypes.data_as(_native.u8p), C.byref(h))
    return h


def test_page_locked_and_device_memory_go_past_the_ring(gpu):
    """Tables in memory that the runtime knows are copied directly (page-locked
    results of more than 1 MiB, also at an offset into their allocation), pageable
    ones through the ring, in any mix; rows and roots the same."""
    n, m, blowup = 1 << 12, 33, 2  # 1 MiB and 32 KiB in, twice that out
    tr = workload.trace_table(35, 0, n, m)
    w = gpu.coset_weights_dev(n, 7).to_array(np.uint64, (n,))
    ref, rows = gpu.coset_lde_row_major_with_merkle_tree_keep(tr, n, m, blowup, w)
    words, off = n * blowup * m, 100
    locked = [_Locked(k + off) for k in (n * m, n, words)]
    locked[0].a[off:] = tr.reshape(-1)
    locked[1].a[off:] = w
    ptr = [x.a[off:].ctypes.data_as(_native.u64p) for x in locked]
    out = np.zeros(words, dtype=np.uint64)
    page = [tr.ctypes.data_as(_native.u64p), w.ctypes.data_as(_native.u64p), out.ctypes.data_as(_native.u64p)]
    for mask in range(8):
        a = [(ptr if mask >> i & 1 else page)[i] for i in range(3)]
        res = locked[2].a[off:] if mask & 4 else out
        res[:] = 0
        hs = []
        used = _ring_use(gpu, lambda: hs.append(gpu.GpuLde(_commit(a[0], n, m, blowup, a[1], a[2]).value)))
        assert hs[0].root == ref.root and np.array_equal(res.reshape(-1, m), rows)
        assert used == ((0 if mask & 1 else 3) + (0 if mask & 2 else 1), 0 if mask & 4 else 5), mask
    for p, slots in ((page[2], 5), (ptr[2], 0)):
        assert _ring_use(gpu, lambda: _native.call("lvm_lde_download", ref.h, p)) == (0, slots)
    # device memory in a host table's place
    buf, dtr, dw = gpu.DeviceBuffer(words * 8), gpu.DeviceBuffer.from_array(tr), gpu.DeviceBuffer.from_array(w)
    d = [C.cast(C.c_void_p(b.ptr), _native.u64p) for b in (dtr, dw, buf)]
    hs = []
    assert _ring_use(gpu, lambda: hs.append(gpu.GpuLde(_commit(d[0], n, m, blowup, d[1], d[2]).value))) == (0, 0)
    assert hs[0].root == ref.root and np.array_equal(buf.to_array(np.uint64, (n * blowup, m)), rows)
    for x in locked:
        x.free()


def test_small_page_locked_results(gpu):
    """Up to 1 MiB of page-locked result comes through the ring, a word more directly."""
    for n, m, slots in ((1 << 13, 16, 2), (1 << 13, 17, 0)):  # LDE of 2^13 rows: 1 MiB and 64 KiB more
        tr = workload.trace_table(36, m, n // 2, m)
        h = gpu.coset_lde_dev(gpu.DeviceBuffer.from_array(tr), n // 2, m, 2, gpu.coset_weights_dev(n // 2, 7))
        x = _Locked(n * m)
        p = x.a.ctypes.data_as(_native.u64p)
        assert _ring_use(gpu, lambda: _native.call("lvm_lde_download", h.h, p)) == (0, slots)
        assert np.array_equal(x.a.reshape(n, m), h.download())
        x.free()


@pytest.mark.parametrize("m,slots", [(32, 64), (33, 0)])  # 2^17 rows: 32 MiB, and past it
def test_large_pageable_tables_go_up_directly(gpu, m, slots):
    n = 1 << 17
    tr = workload.trace_table_modp(37, m, n, m)
    w = gpu.coset_weights_dev(n, 7)
    want = gpu.coset_lde_dev(gpu.DeviceBuffer.from_array(tr), n, m, 1, w).root
    hw = w.to_array(np.uint64, (n,))
    p = [a.ctypes.data_as(_native.u64p) for a in (tr, hw)]
    hs = []
    used = _ring_use(gpu, lambda: hs.append(gpu.GpuLde(_commit(p[0], n, m, 1, p[1], None).value)))
    assert used == (slots + 2, 0) and hs[0].root == want  # the weights are two slots

"""Barycentric sums and DEEP at the widths and row counts where the kernels
split their work: column groups of 64 and 16, rows below a block, and trace
terms with zero weights (pruned openings). Canonical values, exact."""
import ctypes as C

import numpy as np
import pytest

from lambda_vm_amd import _native, workload

pytestmark = pytest.mark.gpu
P = np.uint64(workload.P)


def canon(a):
    a = np.asarray(a, dtype=np.uint64)
    return np.where(a >= P, a - P, a)


def bitrev_perm(log_n):
    return np.array([int(format(i, f"0{log_n}b")[::-1], 2) for i in range(1 << log_n)])


@pytest.mark.parametrize("log_n,m,K", [(1, 1, 1), (1, 300, 2), (3, 2, 8), (5, 255, 2), (6, 256, 1), (7, 257, 2),
                                       (10, 127, 3), (11, 128, 2), (12, 4, 2), (13, 85, 4), (9, 520, 1)])
def test_barycentric_widths(gpu, ora, log_n, m, K):
    n, blowup, g = 1 << log_n, 2, 3
    tr = workload.trace_table(51, log_n, n, m)
    h, host = gpu.coset_lde_row_major_with_merkle_tree_keep(tr, n, m, blowup, ora.lde_weights(n, g))
    zs = workload.fp3_values(177 + log_n, K)
    got = gpu.barycentric_base_multi(h, g, zs)
    for k in range(K):
        assert np.array_equal(canon(got[k]), canon(ora.barycentric_base(host, n, blowup, g, zs[k]))), k


@pytest.mark.parametrize("log_n,m,ma,np_,K,pruned", [(1, 1, 0, 0, 1, False), (2, 16, 1, 1, 2, False),
                                                     (5, 17, 6, 2, 2, True), (6, 33, 11, 3, 2, True),
                                                     (7, 48, 5, 2, 3, False), (8, 4, 22, 1, 2, True),
                                                     (4, 15, 0, 6, 4, False), (9, 120, 2, 2, 2, True)])
def test_deep_widths_and_zero_weights(gpu, ora, log_n, m, ma, np_, K, pruned):
    _deep_matches(gpu, ora, log_n, m, ma, np_, K, "pruned" if pruned else "")


# weights by scalar loads: two sums from 2^18 rows on, three from 2^20 with up to 227
# columns; a geometric case has two
@pytest.mark.parametrize("log_n,m,ma,np_,K,kind", [(17, 17, 2, 1, 2, "pruned"), (17, 3, 0, 0, 2, ""),
                                                   (17, 5, 1, 2, 3, "geometric"), (16, 5, 1, 2, 4, "geometric"),
                                                   (17, 6, 1, 0, 4, "geometric"), (19, 3, 1, 1, 3, ""),
                                                   (18, 3, 1, 1, 3, ""), (17, 2, 0, 1, 1, ""), (17, 2, 0, 1, 4, "")])
def test_deep_weights_scalar_and_in_lds(gpu, ora, log_n, m, ma, np_, K, kind):
    _deep_matches(gpu, ora, log_n, m, ma, np_, K, kind)


def _deep_matches(gpu, ora, log_n, m, ma, np_, K, kind):
    n, blowup, g = 1 << log_n, 2, 3
    N = n * blowup
    w = ora.lde_weights(n, g)
    hm, lm = gpu.coset_lde_row_major_with_merkle_tree_keep(workload.trace_table(52, log_n, n, m), n, m, blowup, w)
    ha = la = hp = lp = None
    if ma:
        ta = workload.trace_table(53, log_n, n, 3 * ma)
        ha, la = gpu.coset_lde_ext3_row_major_with_merkle_tree_keep(ta, n, ma, blowup, w)
    if np_:
        tp = workload.trace_table(54, log_n, n, 3 * np_)
        hp, lp = gpu.coset_lde_ext3_row_major_with_merkle_tree_keep(tp, n, np_, blowup, w)
    cols = m + ma
    zp, tood = workload.fp3_values(55, K), workload.fp3_values(56, cols * K)
    gtr = workload.fp3_values(57, cols * K).reshape(cols, K, 3)
    if kind == "pruned":  # only the last column opens at the next rows, as a bus table's
        gtr[:-1, 1:] = 0
    if kind == "geometric":  # gamma^(cols + j(K-1) + k-1), as the transcript's
        powers = gpu.fp3_powers(workload.fp3_values(61, 1)[0], cols * K)
        gtr[:, 0] = powers[:cols]
        gtr[:, 1:] = powers[cols:].reshape(cols, K - 1, 3)
    gtr = gtr.reshape(-1, 3)
    kw = dict(z_parts=workload.fp3_values(58, 1)[0] if np_ else None,
              parts_ood=workload.fp3_values(59, np_) if np_ else None,
              gammas_h=workload.fp3_values(60, np_) if np_ else None)
    got = gpu.deep_composition(hm, g, zp, tood, gtr, aux=ha, parts=hp, **kw).to_array(np.uint64, (N, 3))
    ref = ora.deep_composition(lm, g, zp, tood, gtr, aux=la, parts=lp, **kw)
    assert np.array_equal(canon(got), canon(ref[bitrev_perm(N.bit_length() - 1)]))


# one point of 64 columns, or two where few lanes idle, take one row per wave, the
# others rows side by side: the edges of both and of their column groups, few rows
# and several chunks
@pytest.mark.parametrize("log_n,m,K", [(1, 64, 1), (12, 63, 1), (12, 64, 2), (12, 65, 1), (11, 64, 3), (10, 129, 2),
                                       (9, 65, 2), (10, 96, 2), (10, 95, 2), (6, 129, 1),
                                       (10, 129, 3), (10, 192, 8), (9, 193, 4), (11, 200, 1), (3, 1480, 2),
                                       (16, 64, 2), (17, 17, 3)])
def test_barycentric_groups(gpu, ora, log_n, m, K):
    test_barycentric_widths(gpu, ora, log_n, m, K)


def test_barycentric_scratch_is_small_beside_the_weights(gpu):
    """Device memory of a call on a wide table: the row weights (24 K n bytes) and
    partial sums that stay below them, by the pool's high-water mark."""
    lib, n, m, K = _native.lib(), 1 << 18, 300, 8
    h = gpu.coset_lde_dev(gpu.splitmix_table_dev(n, m, 7, 1), n, m, 1, gpu.coset_weights_dev(n, 7))
    pool, v = C.c_void_p(), C.c_uint64(0)
    assert lib.hipDeviceGetDefaultMemPool(C.byref(pool), 0) == 0
    gpu.trim()
    assert lib.hipMemPoolGetAttribute(pool, 7, C.byref(v)) == 0  # hipMemPoolAttrUsedMemCurrent
    before = v.value
    v = C.c_uint64(0)
    assert lib.hipMemPoolSetAttribute(pool, 8, C.byref(v)) == 0  # hipMemPoolAttrUsedMemHigh
    gpu.barycentric_base_multi(h, 7, workload.fp3_values(9, K))
    assert lib.hipMemPoolGetAttribute(pool, 8, C.byref(v)) == 0
    assert 24 * K * n <= v.value - before <= 2 * 24 * K * n

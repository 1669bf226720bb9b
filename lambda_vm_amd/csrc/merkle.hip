// Keccak-256 Merkle commitment kernels for gfx950.
//
// Leaf layout (crypto/stark/src/prover.rs:895-961, commitment.rs:42, :81-91):
// leaf i = Keccak( BE(canon(row[br(2i)])) || BE(canon(row[br(2i+1)])) ) over
// the committed columns in order; an Fp3 element streams components 0,1,2
// (extensions_goldilocks.rs:497-503). The LDE tables here are stored with
// their rows already in bit-reversed order, so leaf i reads physical rows
// 2i and 2i+1. A big-endian 8-byte element absorbed into a little-endian
// Keccak lane is bswap64(canonical value); 136-byte blocks are 17 lanes.
//
// Tree layout (crypto/crypto/src/merkle_tree/merkle.rs:201-224, utils.rs:
// 68-96): nodes[0..L-1) inner with the root at 0, leaves at [L-1, 2L-1),
// parent(i) = Keccak(node[2i+1] || node[2i+2]).
#include "lvm_internal.hpp"
#include "tree_top.hpp"

namespace lvm {

static_assert(TREE_WIDE_SPAN == TREE_THREADS, "batched launches are sized in leaves and parents per block of the kernels");

// XOR the big-endian encoding of an element into a lane held as 32-bit
// halves: the little-endian lane of BE(v) is bswap64(v), v canonical.
__device__ __forceinline__ void absorb_be(uint32_t &l, uint32_t &h, uint64_t v) {
    l ^= __builtin_bswap32((uint32_t)(v >> 32));
    h ^= __builtin_bswap32((uint32_t)v);
}

// One thread per leaf. Words [w0, w1) of rows 2i and 2i+1 (row stride
// `pitch` words) are absorbed in order, 17 lanes per permutation. CONTIG:
// the committed words are whole rows, so the leaf's data is one contiguous
// run of 2*pitch words. CANON: the words may lie in [p, 2^64) (rows handed in
// by a caller; this library's own LDE rows are canonical).
// VALU-bound (0.95 of the issue rate on wide tables): what counts is
// instructions. The last block masks the words past the message instead of
// branching per word, which had the compiler copy the 50-register state at
// each of 17 joins (1300 cycles, 7 % of a permutation).
template <bool CONTIG, bool CANON>
__device__ __forceinline__ void row_pair_leaf(const uint64_t *__restrict__ rows, uint64_t pitch, uint64_t w0,
                                              uint64_t w1, uint64_t i, uint64_t *__restrict__ leaves) {
    const uint64_t width = w1 - w0;
    const uint64_t total = 2 * width;
    const uint64_t skip = pitch - width;  // row 2i's end to row 2i+1's start
    const gmem_u64 *row = LVM_GLOBAL_CONST(rows) + (2 * i) * pitch + w0;
    auto word = [&](uint64_t e) -> uint64_t {
        const uint64_t v = row[CONTIG ? e : e + (e >= width ? skip : 0)];
        return CANON ? canon(v) : v;
    };
    uint32_t l[25], h[25];
#pragma unroll
    for (int k = 0; k < 25; k++) l[k] = h[k] = 0;
    uint64_t e = 0;
    for (; e + 17 <= total; e += 17) {
#pragma unroll
        for (int j = 0; j < 17; j++) absorb_be(l[j], h[j], word(e + j));
        keccak_f1600_32(l, h);
    }
    const uint32_t rem = (uint32_t)(total - e);  // 0..16 words, then the padding byte
#pragma unroll
    for (int j = 0; j < 17; j++) {
        const bool in = (uint32_t)j < rem;
        const uint64_t v = word(in ? e + j : 0);
        const uint32_t mask = in ? ~0u : 0u;
        l[j] ^= (__builtin_bswap32((uint32_t)(v >> 32)) & mask) | ((uint32_t)j == rem ? 0x01u : 0u);
        h[j] ^= __builtin_bswap32((uint32_t)v) & mask;
    }
    h[16] ^= 0x80000000u;
    keccak_f1600_32_digest<false>(l, h);
    uint64_t *o = leaves + 4 * i;
#pragma unroll
    for (int k = 0; k < 4; k++) o[k] = ((uint64_t)h[k] << 32) | l[k];
}

// Leaves [span*b, span*b + span) of a small table, one permutation per 16
// lanes, and the tree levels above them in the same launch. A table of up to
// LEAF_TOP_LEAVES leaves would fill at most an eighth of the chip's lanes with
// one leaf each, at 7.2 us per absorbed block; nodes is the whole tree.
__device__ __forceinline__ void row_pair_leaf_top(const uint64_t *rows, uint64_t pitch, uint64_t w0, uint64_t w1,
                                                  uint64_t L, uint32_t span, uint64_t b, uint64_t *nodes,
                                                  uint64_t *root) {
    __shared__ TreeTopLds s;
    const TreeTop t(s, root);
    const uint64_t first = (uint64_t)span * b;
    if (t.wave_on(span)) {
        const bool on = t.g < span;
        const uint64_t width = w1 - w0, total = 2 * width, blocks = total / 17 + 1;
        // the leaf's rows 2i and 2i+1; word e of the message is word e of row
        // 2i, or word e - width of row 2i+1 (pitch - width words further on)
        const gmem_u64 *row = LVM_GLOBAL_CONST(rows) + 2 * (first + (on ? t.g : 0)) * pitch + w0;
        const uint64_t skip = pitch - width;
        uint64_t v[5];
        auto fetch = [&](uint64_t blk) {
#pragma unroll
            for (int x = 0; x < 5; x++) {
                const uint32_t i = 5 * t.y + x;
                const uint64_t e = blk * 17 + i;
                v[x] = on && i < 17 && e < total ? row[e + (e >= width ? skip : 0)] : 0;
            }
        };
        uint32_t a[5] = {0, 0, 0, 0, 0};
        fetch(0);
        for (uint64_t blk = 0; blk < blocks; blk++) {
            const bool last = blk + 1 == blocks;
            const uint64_t rem = total - blk * 17;  // first padding word of the last block
#pragma unroll
            for (int x = 0; x < 5; x++) {
                const uint32_t i = 5 * t.y + x;
                const uint64_t c = canon(v[x]);
                a[x] ^= __builtin_bswap32(t.half ? (uint32_t)c : (uint32_t)(c >> 32));
                if (last && i == rem && t.half == 0) a[x] ^= 0x01;
                if (last && i == 16 && t.half == 1) a[x] ^= 0x80000000u;
            }
            if (!last) fetch(blk + 1);
            t.permute(a);
        }
        if (on) t.put(a, nodes, L - 1 + first + t.g, s, 0);
    }
    tree_top_levels(t, s, nodes, L - 1 + first, span, 0);
}

__global__ __launch_bounds__(TREE_THREADS) void leaf_top_kernel(const uint64_t *rows, uint64_t pitch, uint64_t w0,
                                                                uint64_t w1, uint64_t L, uint32_t span,
                                                                uint64_t *nodes, uint64_t *root) {
    row_pair_leaf_top(rows, pitch, w0, w1, L, span, blockIdx.x, nodes, root);
}

template <bool CONTIG, bool CANON>
__global__ __launch_bounds__(256) void keccak_row_pair_leaves_kernel(const uint64_t *__restrict__ rows,
                                                                    uint64_t pitch, uint64_t w0, uint64_t w1,
                                                                    uint64_t num_leaves,
                                                                    uint64_t *__restrict__ leaves) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num_leaves) return;
    row_pair_leaf<CONTIG, CANON>(rows, pitch, w0, w1, i, leaves);
}

// Leaves of several tables in one launch: blocks [prefix[t], prefix[t+1])
// hash table t's leaves, TREE_THREADS per block, or job.span of them with the
// levels above for a small table.
__global__ __launch_bounds__(TREE_THREADS) void keccak_leaves_batched_kernel(const LeafJob *__restrict__ jobs,
                                                                            const uint32_t *__restrict__ prefix,
                                                                            uint32_t count, uint64_t *roots) {
    const uint32_t b = blockIdx.x;
    const uint32_t t = find_slot(prefix, count, b);
    const LeafJob j = jobs[t];
    if (j.span) {
        row_pair_leaf_top(j.rows, j.pitch, 0, j.pitch, j.num_leaves, j.span, b - prefix[t], j.nodes,
                          roots + 4 * j.root);
        return;
    }
    const uint64_t i = (uint64_t)(b - prefix[t]) * TREE_THREADS + threadIdx.x;
    if (i >= j.num_leaves) return;
    row_pair_leaf<true, false>(j.rows, j.pitch, 0, j.pitch, i, j.nodes + 4 * (j.num_leaves - 1));
}

// parent p = Keccak(node[2p+1] || node[2p+2]), one lane per node
__device__ __forceinline__ void merkle_parent(uint64_t *nodes, uint64_t p) {
    const uint64_t *l = nodes + 4 * (2 * p + 1);
    const uint64_t *r = nodes + 4 * (2 * p + 2);
    uint64_t lv[4] = {l[0], l[1], l[2], l[3]}, rv[4] = {r[0], r[1], r[2], r[3]}, o[4];
    keccak_pair_node(lv, rv, o);
    uint64_t *d = nodes + 4 * p;
    d[0] = o[0];
    d[1] = o[1];
    d[2] = o[2];
    d[3] = o[3];
}

// One level of parents [begin, begin+count).
__global__ __launch_bounds__(256) void merkle_level_kernel(uint64_t *nodes, uint64_t begin, uint64_t count) {
    const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= count) return;
    merkle_parent(nodes, begin + k);
}

// Up to 6 tree levels per launch, one permutation per 16 lanes: block b takes
// the 2*span children [cstart + 2*span*b, ...) of one level (span <=
// TREE_TOP_SPAN parents), writes their parents, keeps them in LDS and keeps
// hashing pairs, writing every level it produces to the node array. The
// levels are a serial chain of permutations, so what counts is the latency of
// one: 512 threads hold 32 states (two waves per SIMD at the first level).
// A tree of 2^11 leaves: 98 -> 48 us against one lane per node with its rounds
// unrolled; 2^17 leaves (top of 2^14): 130 -> 62 us.
__device__ __forceinline__ void merkle_top_body(uint64_t *nodes, uint64_t cstart, uint64_t pstart, uint32_t span,
                                                uint64_t b, uint64_t *root) {
    __shared__ TreeTopLds s;
    const TreeTop t(s, root);
    const uint64_t pbase = pstart + (uint64_t)span * b;  // first parent of this block
    if (t.wave_on(span)) {
        const bool on = t.g < span;
        uint32_t a[5];
        coop_load_pair(a, (const gmem_u32 *)nodes + 8 * (cstart + 2 * ((uint64_t)span * b + t.g)), on);
        t.permute(a);
        if (on) t.put(a, nodes, pbase + t.g, s, 0);
    }
    tree_top_levels(t, s, nodes, pbase, span, 0);
}

__global__ __launch_bounds__(TREE_THREADS) void merkle_top_kernel(uint64_t *nodes, uint64_t cstart, uint64_t pstart,
                                                                  uint32_t span, uint64_t *root) {
    merkle_top_body(nodes, cstart, pstart, span, blockIdx.x, root);
}

// One tree step for each of several trees: blocks [prefix[t], prefix[t+1])
// run step t (one wide level, TREE_THREADS parents per block, or a tree top).
__global__ __launch_bounds__(TREE_THREADS) void merkle_steps_batched_kernel(const TreeStep *__restrict__ steps,
                                                                            const uint32_t *__restrict__ prefix,
                                                                            uint32_t count, uint64_t *roots) {
    const uint32_t b = blockIdx.x;
    const uint32_t t = find_slot(prefix, count, b);
    const TreeStep s = steps[t];
    if (s.span > TREE_TOP_SPAN) {
        const uint32_t i = s.span * (b - prefix[t]) + threadIdx.x;
        if (i < s.parents) merkle_parent(s.nodes, s.pstart + i);
    } else
        merkle_top_body(s.nodes, s.cstart, s.pstart, s.span, b - prefix[t], roots + 4 * s.root);
}

size_t padded_leaves(size_t n) {
    size_t p = 1;
    while (p < n) p <<= 1;
    return p;
}

uint64_t keccak_row_pair_leaves(const uint64_t *rows, uint64_t pitch, uint64_t w0, uint64_t w1, uint64_t L,
                                bool canonical, uint8_t *nodes, uint64_t *root_out, hipStream_t st) {
    if (L <= LEAF_TOP_LEAVES) {
        const uint32_t span = leaf_top_span(L);
        hipLaunchKernelGGL(leaf_top_kernel, dim3((unsigned)(L / span)), dim3(TREE_THREADS), 0, st, rows, pitch, w0, w1,
                           L, span, (uint64_t *)nodes, root_out);
        return L / span;
    }
    uint64_t *leaves = (uint64_t *)(nodes + (L - 1) * 32);
    dim3 grid((unsigned)((L + 255) / 256));
    const bool contig = w0 == 0 && w1 == pitch;
    if (contig && canonical)
        hipLaunchKernelGGL((keccak_row_pair_leaves_kernel<true, false>), grid, dim3(256), 0, st, rows, pitch, w0, w1,
                           L, leaves);
    else if (contig)
        hipLaunchKernelGGL((keccak_row_pair_leaves_kernel<true, true>), grid, dim3(256), 0, st, rows, pitch, w0, w1, L,
                           leaves);
    else
        hipLaunchKernelGGL((keccak_row_pair_leaves_kernel<false, true>), grid, dim3(256), 0, st, rows, pitch, w0, w1,
                           L, leaves);
    return L;
}

void merkle_build_inner(uint8_t *nodes_b, uint64_t C, uint64_t *root_out, hipStream_t st) {
    uint64_t *nodes = (uint64_t *)nodes_b;
    // wide levels: one fully parallel launch per level
    while (C > TREE_TOP_CHILDREN) {
        const uint64_t count = C / 2;
        hipLaunchKernelGGL(merkle_level_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, nodes,
                           count - 1, count);
        C = count;
    }
    // narrow top: up to 6 levels per launch through LDS
    while (C > 1) {
        const uint32_t span = (uint32_t)(C / 2 < TREE_TOP_SPAN ? C / 2 : TREE_TOP_SPAN);
        const uint64_t blocks = C / (2 * span);
        hipLaunchKernelGGL(merkle_top_kernel, dim3((unsigned)blocks), dim3(TREE_THREADS), 0, st, nodes, C - 1,
                           C / 2 - 1, span, root_out);
        C = blocks;
    }
}

void launch_leaves_batched(const LeafJob *d_jobs, const uint32_t *d_prefix, uint32_t count, uint32_t blocks,
                           uint64_t *roots, hipStream_t st) {
    if (blocks)
        hipLaunchKernelGGL(keccak_leaves_batched_kernel, dim3(blocks), dim3(TREE_THREADS), 0, st, d_jobs, d_prefix,
                           count, roots);
}

void launch_tree_steps_batched(const TreeStep *d_steps, const uint32_t *d_prefix, uint32_t count, uint32_t blocks,
                               uint64_t *roots, hipStream_t st) {
    if (blocks)
        hipLaunchKernelGGL(merkle_steps_batched_kernel, dim3(blocks), dim3(TREE_THREADS), 0, st, d_steps, d_prefix, count,
                           roots);
}

}  // namespace lvm

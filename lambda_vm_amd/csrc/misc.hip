// Small kernels: field-arithmetic test kernels (crypto/math-cuda/kernels/
// arith.cu semantics), bit-reversed row gathers, Merkle path gathers.
#include "lvm_internal.hpp"

namespace lvm {

__global__ void gl_op_kernel(int op, const uint64_t *a, const uint64_t *b, uint64_t *out, uint64_t n) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint64_t x = a[i], y = b ? b[i] : 0, r;
    switch (op) {
    case 0: r = add(x, y); break;
    case 1: r = sub(x, y); break;
    case 2: r = mul(x, y); break;
    case 3: r = neg(x); break;
    case 4: r = inv(x); break;
    default: r = sqr(x); break;
    }
    out[i] = r;
}

__global__ void fp3_op_kernel(int op, const uint64_t *a, const uint64_t *b, uint64_t *out, uint64_t n) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    fp3 x{a[3 * i], a[3 * i + 1], a[3 * i + 2]};
    fp3 y{0, 0, 0};
    if (b) y = fp3{b[3 * i], b[3 * i + 1], b[3 * i + 2]};
    fp3 r;
    switch (op) {
    case 0: r = f3_add(x, y); break;
    case 1: r = f3_sub(x, y); break;
    case 2: r = f3_mul(x, y); break;
    case 3: r = f3_neg(x); break;
    case 4: r = f3_inv(x); break;
    default: r = f3_sqr(x); break;
    }
    out[3 * i] = r.c0;
    out[3 * i + 1] = r.c1;
    out[3 * i + 2] = r.c2;
}

void launch_gl_op(int op, const uint64_t *a, const uint64_t *b, uint64_t *out, uint64_t n, bool ext3,
                  hipStream_t st) {
    dim3 grid((unsigned)((n + 255) / 256));
    if (ext3)
        hipLaunchKernelGGL(fp3_op_kernel, grid, dim3(256), 0, st, op, a, b, out, n);
    else
        hipLaunchKernelGGL(gl_op_kernel, grid, dim3(256), 0, st, op, a, b, out, n);
}

__global__ void copy_words_kernel(const uint64_t *__restrict__ src, uint64_t *__restrict__ dst, uint64_t count) {
    const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < count) dst[idx] = src[idx];
}

void launch_copy_words(const uint64_t *src, uint64_t *dst, uint64_t count, hipStream_t st) {
    if (!count) return;
    hipLaunchKernelGGL(copy_words_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, src, dst, count);
}

// Words [first, first + count) of the natural-order table (row r = physical row
// bitrev(r), rows of `w` words) to dst[0, count).
__global__ void gather_bitrev_rows_kernel(const uint64_t *__restrict__ src, uint64_t *__restrict__ dst,
                                          uint32_t log_rows, uint64_t w, uint64_t first, uint64_t count) {
    const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= count) return;
    const uint64_t r = (first + idx) / w, c = first + idx - r * w;
    const uint64_t pr = log_rows ? bitrev((uint32_t)r, log_rows) : 0;
    dst[idx] = src[pr * w + c];
}

void launch_gather_bitrev_words(const uint64_t *src, uint64_t *dst, uint32_t log_rows, uint64_t w, uint64_t first,
                                uint64_t count, hipStream_t st) {
    if (!count) return;
    hipLaunchKernelGGL(gather_bitrev_rows_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, src, dst,
                       log_rows, w, first, count);
}

void launch_gather_bitrev_rows(const uint64_t *src, uint64_t *dst, uint64_t rows, uint32_t log_rows, uint64_t w,
                               hipStream_t st) {
    launch_gather_bitrev_words(src, dst, log_rows, w, 0, rows * w, st);
}

// Merkle authentication paths (sibling of each node from the leaf up,
// crypto/crypto/src/merkle_tree/merkle.rs:291-308) and the two opened rows
// per position (physical rows 2*pos and 2*pos+1 of the bit-reversed table).
// One block per position, every path node and row word read at once: level k's
// L >> k nodes start at (L >> k) - 1, so the sibling of leaf p's ancestor there
// is node (L >> k) - 1 + ((p >> k) ^ 1). 30 positions of a 2^21-leaf tree: a
// thread walking its path and rows took 43 us.
__global__ __launch_bounds__(256) void open_kernel(const uint64_t *__restrict__ nodes, uint64_t L,
                                                   const uint64_t *__restrict__ lde, uint64_t w,
                                                   const uint64_t *__restrict__ pos, uint32_t depth, uint64_t *paths,
                                                   uint64_t *rows) {
    const uint64_t q = blockIdx.x, p = pos[q];
    for (uint32_t i = threadIdx.x; i < 4 * depth; i += 256) {
        const uint32_t k = i / 4;
        paths[q * depth * 4 + i] = nodes[4 * ((L >> k) - 1 + ((p >> k) ^ 1)) + i % 4];
    }
    if (rows)
        for (uint64_t j = threadIdx.x; j < 2 * w; j += 256) rows[q * 2 * w + j] = lde[2 * p * w + j];
}

void launch_open(const uint64_t *nodes, uint64_t L, const uint64_t *lde, uint64_t w, const uint64_t *pos,
                 uint64_t count, uint32_t depth, uint64_t *paths, uint64_t *rows, hipStream_t st) {
    // a grid holds fewer than 2^32 threads: launches of at most 2^23 positions
    constexpr uint64_t MOST = 1u << 23;
    for (uint64_t q = 0; q < count; q += MOST) {
        const uint64_t n = count - q < MOST ? count - q : MOST;
        hipLaunchKernelGGL(open_kernel, dim3((unsigned)n), dim3(256), 0, st, nodes, L, lde, w, pos + q, depth,
                           paths + q * depth * 4, rows ? rows + q * 2 * w : nullptr);
    }
}

// Plain 16-byte-vector device copy (grid-stride), the calibration kernel for
// HBM traffic counters.
// One 16-byte element per lane over a full grid (blocks walk the buffer in
// order): 6.2 TB/s on 1 GiB, where a grid-stride loop over 16384 blocks
// measured 4.7 TB/s.
__global__ __launch_bounds__(256) void copy16_kernel(const uint4 *__restrict__ src, uint4 *__restrict__ dst,
                                                     uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

void launch_copy16(void *dst, const void *src, uint64_t n16, hipStream_t st) {
    // launches of at most 2^31 blocks (2^43 bytes) each
    const uint64_t chunk = (uint64_t)256 << 31;
    for (uint64_t off = 0; off < n16; off += chunk) {
        const uint64_t n = n16 - off < chunk ? n16 - off : chunk;
        hipLaunchKernelGGL(copy16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                           (const uint4 *)src + off, (uint4 *)dst + off, n);
    }
}

// w_i = scale * offset^i (the coset weights n^-1 * g^i of
// crypto/stark/src/prover.rs:451-467 with scale = n^-1)
__global__ void coset_weights_kernel(uint64_t n, uint64_t offset, uint64_t scale, uint64_t *out) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = mul(scale, pow(offset, i));
}

void launch_coset_weights(uint64_t n, uint64_t offset, uint64_t scale, uint64_t *out, hipStream_t st) {
    if (!n) return;
    hipLaunchKernelGGL(coset_weights_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, offset, scale,
                       out);
}

// Synthetic table: element (r, c) = SplitMix64 draw r of the stream seeded
// with 0x1A3BDA7A ^ (cfg << 48) ^ (table << 32) ^ c, reduced mod p (draw k is
// mix(seed + (k+1) * 0x9E3779B97F4A7C15)). Row-major n x m.
__global__ void fill_splitmix_kernel(uint64_t *out, uint64_t n, uint64_t m, uint64_t cfg, uint64_t table) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n * m) return;
    const uint64_t r = i / m, c = i % m;
    const uint64_t seed = 0x1A3BDA7Aull ^ (cfg << 48) ^ (table << 32) ^ c;
    uint64_t z = seed + (r + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    out[i] = canon(z);
}

void launch_fill_splitmix(uint64_t *out, uint64_t n, uint64_t m, uint64_t cfg, uint64_t table, hipStream_t st) {
    const uint64_t total = n * m;
    if (!total) return;
    hipLaunchKernelGGL(fill_splitmix_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, out, n, m, cfg,
                       table);
}

}  // namespace lvm

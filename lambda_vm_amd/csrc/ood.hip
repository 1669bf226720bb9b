// Out-of-domain stage kernels for gfx950: Fp3 batch inversion, inverted
// denominators over the LDE coset, barycentric evaluation of resident LDE
// columns at K points, and the DEEP composition codeword.
//
// Coset points: physical row p of a resident LDE table (rows stored in
// bit-reversed order) is the natural LDE index bitrev_N(p), i.e. the point
// x_p = g * w_N^bitrev_N(p). Its first n physical rows are the sub-coset
// g*<w_n> the barycentric formula of crypto/stark/src/trace.rs:831-1110
// reads (natural rows i*B), so those reads are contiguous here.
#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

#include "lvm_internal.hpp"
#include "prof.hpp"

namespace lvm {

__device__ __forceinline__ fp3 ld3(const uint64_t *p) { return fp3{p[0], p[1], p[2]}; }
__device__ __forceinline__ void st3(uint64_t *p, fp3 v) {
    p[0] = v.c0;
    p[1] = v.c1;
    p[2] = v.c2;
}

// Montgomery batch inversion (crypto/math/src/field/element.rs:64-111) with
// interleaved ownership: thread t inverts elements t, t+T, t+2T, ... so each
// wave's loads and stores stay coalesced; one Fp3 inversion per thread.
// `out` holds the running prefix products during the forward sweep.
__global__ __launch_bounds__(256) void batch_inverse_fp3_kernel(const uint64_t *__restrict__ in,
                                                                uint64_t *__restrict__ out, uint64_t n) {
    const uint64_t T = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    fp3 acc = fp3{1, 0, 0};
    uint64_t i = t;
    for (; i < n; i += T) {
        acc = f3_mul(acc, ld3(in + 3 * i));
        st3(out + 3 * i, acc);
    }
    fp3 inv_acc = f3_inv(acc);
    // walk back: out[i] = inv_acc * prefix[i - T]; inv_acc *= in[i]
    uint64_t last = t + ((n - 1 - t) / T) * T;
    for (i = last;; i -= T) {
        if (i >= T) {
            fp3 prev = ld3(out + 3 * (i - T));
            fp3 xi = ld3(in + 3 * i);
            st3(out + 3 * i, f3_mul(inv_acc, prev));
            inv_acc = f3_mul(inv_acc, xi);
        } else {
            st3(out + 3 * i, inv_acc);
            break;
        }
    }
}

// Inverted pole factors over the LDE coset, for K poles z_k in Fp3 and the
// first `rows` physical rows p of an LDE of 2^log_N rows on offset*<w_N>
// (x_p = offset * w_N^bitrev_N(p)):
//   mode 0: out[k * rows + p] = 1 / (x_p - z_k)        (DEEP, XMinusZ)
//   mode 1: out[k * rows + p] = x_p / (z_k - x_p)      (barycentric weights)
// x - z has constant w and w^2 parts (-z1, -z2), so with a0 = x - z0 its norm
// and adjugate in Fp[w]/(w^3 - 2) are cheap base-field polynomials in a0:
//   Norm = a0^3 - 6 z1 z2 a0 - (2 z1^3 + 4 z2^3)
//   adj  = (a0^2 - 2 z1 z2, 2 z2^2 + z1 a0, z1^2 + z2 a0),  1/(x - z) = adj / Norm.
// Each thread owns E rows p = t, t + T, ... (coalesced) and inverts the
// products D(p) = prod_k Norm_k(p) of its rows with one base-field inversion
// (Montgomery's trick, prefixes kept in registers); Norm_k^-1 = D^-1 * prod_{j != k} Norm_j.
// Replaces the Fp3 batch inversion of materialised differences
// (crypto/math-cuda/src/inverse.rs:241-300, crypto/stark/src/trace.rs:900-940).
struct PoleConst {
    uint64_t z0, z1, z2, c1x3, c3, c1, c2, z1s;
};
// rows per thread E: 16 on large domains; 2 on small ones, where the chain of
// E rows (not the grid) sets the kernel's duration

template <int K, int E>
__global__ __launch_bounds__(256) void pole_inverse_kernel(uint64_t *__restrict__ out, uint64_t rows, uint32_t log_N,
                                                           uint64_t offset, const uint64_t *__restrict__ z, int mode,
                                                           const uint64_t *__restrict__ lo,
                                                           const uint64_t *__restrict__ hi) {
    const uint64_t T = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= rows) return;
    PoleConst pc[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        const uint64_t z0 = z[3 * k], z1 = z[3 * k + 1], z2 = z[3 * k + 2];
        const uint64_t z12 = mul(z1, z2), c1 = dbl(z12);
        const uint64_t z1s = sqr(z1), z2s = sqr(z2);
        pc[k] = PoleConst{z0, z1, z2, add(dbl(c1), c1), add(dbl(mul(z1s, z1)), dbl(dbl(mul(z2s, z2)))), c1, dbl(z2s),
                          z1s};
    }
    auto point = [&](uint64_t p) -> uint64_t {
        const uint32_t e = log_N ? (bitrev((uint32_t)p, log_N) << (32 - log_N)) : 0u;
        return mul(offset, mul(lo[e & 0xFFFFu], hi[e >> 16]));
    };
    auto norm = [&](const PoleConst &c, uint64_t x, uint64_t &a0, uint64_t &sq) -> uint64_t {
        a0 = sub(x, c.z0);
        sq = sqr(a0);
        return sub(sub(mul(sq, a0), mul(c.c1x3, a0)), c.c3);
    };
    uint64_t pre[E];
    uint64_t acc = 1;
#pragma unroll
    for (int j = 0; j < E; j++) {
        const uint64_t p = t + (uint64_t)j * T;
        if (p < rows) {
            const uint64_t x = point(p);
            uint64_t d = 1;
#pragma unroll
            for (int k = 0; k < K; k++) {
                uint64_t a0, sq;
                d = mul(d, norm(pc[k], x, a0, sq));
            }
            acc = mul(acc, d);
        }
        pre[j] = acc;
    }
    uint64_t inv_acc = inv(acc);
#pragma unroll
    for (int j = E - 1; j >= 0; j--) {
        const uint64_t p = t + (uint64_t)j * T;
        if (p >= rows) continue;
        const uint64_t x = point(p);
        uint64_t a0[K], sq[K], nk[K];
#pragma unroll
        for (int k = 0; k < K; k++) nk[k] = norm(pc[k], x, a0[k], sq[k]);
        uint64_t d = 1;
#pragma unroll
        for (int k = 0; k < K; k++) d = mul(d, nk[k]);
        uint64_t dinv = j ? mul(inv_acc, pre[j - 1]) : inv_acc;
        inv_acc = mul(inv_acc, d);
        if (mode) dinv = mul(dinv, neg(x));
        // prefix / suffix products of the norms: Norm_k^-1 = D^-1 * pre_k * suf_k
        uint64_t sfx[K];
        sfx[K - 1] = 1;
#pragma unroll
        for (int k = K - 2; k >= 0; k--) sfx[k] = mul(sfx[k + 1], nk[k + 1]);
        uint64_t pfx = dinv;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const uint64_t ni = K > 1 ? mul(pfx, sfx[k]) : pfx;
            if (k + 1 < K) pfx = mul(pfx, nk[k]);
            const PoleConst &c = pc[k];
            const fp3 adj = fp3{sub(sq[k], c.c1), add(c.c2, mul(c.z1, a0[k])), add(c.z1s, mul(c.z2, a0[k]))};
            st3(out + 3 * ((uint64_t)k * rows + p), f3_mul_base(adj, ni));
        }
    }
}

template <int E>
static void launch_pole_inverse_e(uint64_t *out, uint64_t rows, uint32_t log_N, uint64_t offset, const uint64_t *z,
                                  uint32_t K, int mode, const uint64_t *lo, const uint64_t *hi, hipStream_t st) {
    const uint64_t threads = (rows + E - 1) / E;
    const dim3 grid((unsigned)((threads + 255) / 256)), blk(256);
    switch (K) {
    case 1: hipLaunchKernelGGL((pole_inverse_kernel<1, E>), grid, blk, 0, st, out, rows, log_N, offset, z, mode, lo, hi); break;
    case 2: hipLaunchKernelGGL((pole_inverse_kernel<2, E>), grid, blk, 0, st, out, rows, log_N, offset, z, mode, lo, hi); break;
    case 3: hipLaunchKernelGGL((pole_inverse_kernel<3, E>), grid, blk, 0, st, out, rows, log_N, offset, z, mode, lo, hi); break;
    case 4: hipLaunchKernelGGL((pole_inverse_kernel<4, E>), grid, blk, 0, st, out, rows, log_N, offset, z, mode, lo, hi); break;
    case 5: hipLaunchKernelGGL((pole_inverse_kernel<5, E>), grid, blk, 0, st, out, rows, log_N, offset, z, mode, lo, hi); break;
    case 6: hipLaunchKernelGGL((pole_inverse_kernel<6, E>), grid, blk, 0, st, out, rows, log_N, offset, z, mode, lo, hi); break;
    case 7: hipLaunchKernelGGL((pole_inverse_kernel<7, E>), grid, blk, 0, st, out, rows, log_N, offset, z, mode, lo, hi); break;
    default: hipLaunchKernelGGL((pole_inverse_kernel<8, E>), grid, blk, 0, st, out, rows, log_N, offset, z, mode, lo, hi); break;
    }
}

static void launch_pole_inverse(uint64_t *out, uint64_t rows, uint32_t log_N, uint64_t offset, const uint64_t *z,
                                uint32_t K, int mode, const uint64_t *lo, const uint64_t *hi, hipStream_t st) {
    if (!rows) return;
    if (rows >= (1u << 20))
        launch_pole_inverse_e<16>(out, rows, log_N, offset, z, K, mode, lo, hi, st);
    else
        launch_pole_inverse_e<2>(out, rows, log_N, offset, z, K, mode, lo, hi, st);
}

constexpr int BARY_MAX_K = 8;
// partial[chunk][k][c] = sum over the chunk's rows p of lde[p][c] * scale[k][p]
// block: 256 threads over a group of gc adjacent columns and as many rows RB at
// once as fit; grid (chunks of rpb rows, column groups). The three components
// of each point's sum are delayed-reduction dot products (one 128-bit accumulate
// per product, one reduction per thread), loads of U rows issued together; the
// RB partial sums of a column meet in LDS. Two forms:
//  - packed: thread = row * columns + column, so a block's loads are runs of whole
//    rows and no lane idles on a narrow table (with 64 lanes a row, 17 columns
//    used 17 of them); every lane loads its row's scales;
//  - WAVE: a row per wave, 64 columns a group, the scales by scalar loads and as
//    scalar operands: half the registers, one vector load a row instead of 1 + 3 K.
// bary_shape says which, with both measured.
constexpr int BARY_WAVE_MAX_K = 2;

template <int K, bool WAVE>
__global__ __launch_bounds__(256) void bary_partial_kernel(const uint64_t *__restrict__ lde, uint64_t w, uint64_t n,
                                                           uint32_t gc, uint64_t rpb,
                                                           const uint64_t *__restrict__ scale,
                                                           uint64_t *__restrict__ partial) {
    constexpr int U = K <= 2 ? 4 : 2;
    __shared__ uint64_t red[256][3];
    const uint32_t t = threadIdx.x;
    const uint64_t c0 = (uint64_t)blockIdx.y * gc;
    const uint32_t have = w - c0 < gc ? (uint32_t)(w - c0) : gc;
    const uint32_t wc = WAVE ? 64 : have, RB = 256 / wc;
    const uint32_t r = WAVE ? __builtin_amdgcn_readfirstlane(t / 64) : t / wc, c = t - r * wc;
    const uint64_t p0 = (uint64_t)blockIdx.x * rpb, pend = p0 + rpb < n ? p0 + rpb : n;
    acc128 acc[K][3];
#pragma unroll
    for (int k = 0; k < K; k++)
#pragma unroll
        for (int j = 0; j < 3; j++) acc_zero(acc[k][j]);
    if (WAVE ? c < have : r < RB) {
        const gmem_u64 *f = LVM_GLOBAL_CONST(lde) + c0 + c;
        // scales of a wave's row in the constant address space (no kernel in flight
        // writes them): a uniform address becomes a scalar load
        using scale_u64 = std::conditional_t<WAVE, const __attribute__((address_space(4))) uint64_t, const gmem_u64>;
        scale_u64 *sc = (scale_u64 *)scale;
        uint64_t p = p0 + r;
        for (; p + (U - 1) * RB < pend; p += U * RB) {
            uint64_t v[U], s[U][K][3];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint64_t q = p + u * RB;
                v[u] = f[q * w];
#pragma unroll
                for (int k = 0; k < K; k++)
#pragma unroll
                    for (int j = 0; j < 3; j++) s[u][k][j] = sc[3 * (k * n + q) + j];
            }
            __builtin_amdgcn_sched_barrier(0);  // all U rows' loads before the first product
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int k = 0; k < K; k++)
#pragma unroll
                    for (int j = 0; j < 3; j++) {
                        if constexpr (WAVE)
                            acc_mad_uniform(acc[k][j], s[u][k][j], v[u]);
                        else
                            acc_mad(acc[k][j], s[u][k][j], v[u]);
                    }
        }
        for (; p < pend; p += RB) {
            const uint64_t v = f[p * w];
#pragma unroll
            for (int k = 0; k < K; k++)
#pragma unroll
                for (int j = 0; j < 3; j++) acc_mad(acc[k][j], sc[3 * (k * n + p) + j], v);
        }
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        fp3 v = fp3{acc_reduce(acc[k][0]), acc_reduce(acc[k][1]), acc_reduce(acc[k][2])};
        st3(red[t], v);
        for (uint32_t left = RB; left > 1;) {
            const uint32_t half = (left + 1) / 2;
            __syncthreads();
            if (r + half < left) {
                v = f3_add(v, ld3(red[t + half * wc]));
                st3(red[t], v);
            }
            left = half;
        }
        if (r == 0 && c < have) st3(partial + 3 * (((uint64_t)blockIdx.x * K + k) * w + c0 + c), v);
        __syncthreads();  // the sums are rewritten for the next point
    }
}

struct BaryShape {
    bool wave;
    uint32_t gc;               // columns of a group
    uint64_t cgroups, rpb, chunks;
};

// A table of 64 columns or more takes a row per wave for one point, and for two
// where that leaves at most a quarter of the lanes idle (bary_sum of 2^20 rows,
// packed form against this one, K = 1 and 2: 64 columns 174 against 127 us and 231
// against 207; 65 columns 206 against 185 and 288 against 428; 100 columns 295
// against 209 and 430 against 370; 129 columns 419 against 325 and 577 against
// 616; 256 columns 604 against 400 and 858 against 673; 48 columns K = 2 188 against
// 183). Three points run out of scalar registers (256 columns 1165 against 1293).
// Packed groups are all of a row up to 128 columns, then equal groups of at most
// 64, which leave few lanes over (one group of 200 used 200 of 256: K = 4 1827
// against 1240). A chunk is 1024 rows (64 a thread when more than 16 fit side by
// side), less when the grid would have under 1024 blocks: chunks of 64 rows of wide
// tables made the partial sums 16 times as large (2^22 x 300 at eight points 3.8
// GB) and were no faster.
BaryShape bary_shape(uint64_t n, uint64_t w, size_t K) {
    BaryShape b;
    b.wave = w >= 64 && (K == 1 || (K == BARY_WAVE_MAX_K && 4 * w >= 3 * 64 * ((w + 63) / 64)));
    b.cgroups = b.wave || w > 128 ? (w + 63) / 64 : 1;
    b.gc = b.wave ? 64 : (uint32_t)((w + b.cgroups - 1) / b.cgroups);
    const uint64_t RB = 256 / b.gc;
    b.rpb = std::max<uint64_t>(1024, 64 * RB);
    while (b.rpb > 4 * RB && ((n + b.rpb - 1) / b.rpb) * b.cgroups < 1024) b.rpb /= 2;
    b.chunks = (n + b.rpb - 1) / b.rpb;
    return b;
}

template <int K>
static void launch_bary_partial(const BaryShape &b, hipStream_t st, const uint64_t *lde, uint64_t w, uint64_t n,
                                const uint64_t *scale, uint64_t *partial) {
    const dim3 grid((unsigned)b.chunks, (unsigned)b.cgroups);
    if constexpr (K <= BARY_WAVE_MAX_K) {
        if (b.wave) {
            hipLaunchKernelGGL((bary_partial_kernel<K, true>), grid, dim3(256), 0, st, lde, w, n, b.gc, b.rpb, scale,
                               partial);
            return;
        }
    }
    hipLaunchKernelGGL((bary_partial_kernel<K, false>), grid, dim3(256), 0, st, lde, w, n, b.gc, b.rpb, scale, partial);
}

// out[k][c] = vf[k] * sum over chunks of partial[chunk][k][c]; one block per
// output (k, c): its threads sum strided chunks, then a tree in LDS.
__global__ __launch_bounds__(256) void bary_combine_kernel(const uint64_t *partial, uint64_t chunks, uint32_t K,
                                                           uint64_t w, const uint64_t *vf, uint64_t *out) {
    __shared__ uint64_t red[256][3];
    const uint64_t idx = blockIdx.x;
    const uint64_t k = idx / w, c = idx - k * w;
    const uint32_t t = threadIdx.x;
    fp3 s = fp3{0, 0, 0};
    for (uint64_t ch = t; ch < chunks; ch += 256) s = f3_add(s, ld3(partial + 3 * ((ch * K + k) * w + c)));
    red[t][0] = s.c0;
    red[t][1] = s.c1;
    red[t][2] = s.c2;
    for (uint32_t h = 128; h > 0; h >>= 1) {
        __syncthreads();
        if (t < h) {
            fp3 v = f3_add(fp3{red[t][0], red[t][1], red[t][2]}, fp3{red[t + h][0], red[t + h][1], red[t + h][2]});
            red[t][0] = v.c0;
            red[t][1] = v.c1;
            red[t][2] = v.c2;
        }
    }
    if (t == 0) st3(out + 3 * idx, f3_mul(ld3(vf + 3 * k), fp3{red[0][0], red[0][1], red[0][2]}));
}

// DEEP composition at every LDE row (crypto/math-cuda/kernels/deep.cu:1-25,
// crypto/stark/src/prover.rs:2400-2604), in storage (bit-reversed) order:
//   deep[p] = inv_h[p] * (sum_j gh_j * H_j[p] - ch)
//           + sum_k inv_t[k][p] * (sum_j gt_{j,k} * t_j[p] - ct_k)
// where ch = sum_j gh_j * H_j(z^P) and ct_k = sum_j gt_{j,k} * t_j(z_k) are
// computed once on the host, main columns are base words, aux and parts are
// Fp3 (3 words each).
constexpr int DEEP_MAX_K = 4;
constexpr int DEEP_CHUNK = 16;  // most columns staged per LDS round

// An Fp3 column a = a0 + a1 w + a2 w^2 weighted by g is three base columns
// weighted by g, w g and w^2 g, so every table is a segment of base columns.
struct DeepSegment {
    const uint64_t *rows;
    uint64_t cols;  // words per row
};
struct DeepArgs {
    uint64_t N;
    DeepSegment trace[2], parts;  // main and aux trace words, composition parts words
    const uint64_t *gtr;          // [trace word][KA][3]
    const uint64_t *gh;           // [parts word][3]
    const uint64_t *consts;       // ct_k, then ch
    const uint64_t *rpow;
    const uint64_t *inv_den;      // [pole][N][3]
    uint64_t *out;
};

// block: 256 consecutive physical rows. A chunk of columns of those rows goes
// through LDS with coalesced row-segment loads (the next chunk's loads are
// issued before the current chunk is accumulated); each thread accumulates
// its row's sum_j gt_{j,k} * t_j[p] as 3*KA delayed-reduction dot products.
// The weights are the same for every row: scalar loads and scalar operands, a
// zero weight skipped (a bus table opens one column at its next row, so all its
// other weights of k = 1 are zero), or, LW, beside the columns in LDS
// (launch_deep). KA < K when the trace-term weights are geometric in k past the
// first KA - 1 points (gt_{j,k} = gt_{j,KA-1} * r^(k-KA+1) for every column j,
// which the reference's weights are: gamma^(W + j(K-1) + k - 1) for k >= 1,
// crypto/stark/src/prover.rs:2400-2460): then sum_j gt_{j,k} t_j = r^(k-KA+1) *
// sum_j gt_{j,KA-1} t_j, and rpow[k] holds r^(k-KA+1).
template <int K, int KA, bool LW>
__global__ __launch_bounds__(256) void deep_kernel(DeepArgs a) {
    __shared__ uint64_t tile[256][DEEP_CHUNK + 1];
    __shared__ uint64_t sw[LW ? DEEP_CHUNK * 3 * KA : 1];
    const uint32_t t = threadIdx.x;
    const uint64_t N = a.N, r0 = (uint64_t)blockIdx.x * 256, p = r0 + t;
    uint64_t nv[DEEP_CHUNK], nw = 0;
    // columns [j0, j0 + cw) of the block's rows: thread t loads column t % 16 of
    // rows t / 16, t / 16 + 16, ... (16 lanes per row segment)
    const uint32_t lc = t & 15, lr = t >> 4;
    const uint32_t rows = N - r0 < 256 ? (uint32_t)(N - r0) : 256u;  // a power of two
    auto fetch = [&](const DeepSegment &s, uint32_t j0, uint32_t cw, const uint64_t *w, uint32_t words) {
        if (LW) nw = t < cw * words ? LVM_GLOBAL_CONST(w)[t] : 0;  // columns past the chunk weigh nothing
        if (lc >= cw || lr >= rows) return;
        const gmem_u64 *src = LVM_GLOBAL_CONST(s.rows) + (r0 + lr) * s.cols + j0 + lc;
        const uint64_t step = 16 * s.cols;
        if (rows == 256) {
#pragma unroll
            for (int q = 0; q < 16; q++) nv[q] = src[q * step];
        } else {
#pragma unroll
            for (int q = 0; q < 16; q++)
                if (16u * q < rows) nv[q] = src[q * step];
        }
    };
    auto stage = [&]() {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 16; q++) tile[lr + 16 * q][lc] = nv[q];
        if (LW && t < DEEP_CHUNK * 3 * KA) sw[t] = nw;
        __syncthreads();
    };
    // acc[k] += w_k * (the thread's value) over the chunk's columns; a column's
    // scalar weights are loaded while the previous one is accumulated
    auto accumulate = [&](auto &acc, const uint64_t *w, uint32_t cw) {
        constexpr int NK = sizeof(acc) / sizeof(acc[0]);
        if constexpr (LW) {
            // eight columns' LDS reads together (2^12 x 600, one sum: 78 us, four 93)
            for (uint32_t c0 = 0; c0 < cw; c0 += 8) {
#pragma unroll
                for (uint32_t cc = c0; cc < c0 + 8; cc++) {
                    const uint64_t v = tile[t][cc];
                    const uint64_t *g = sw + 3 * NK * cc;
#pragma unroll
                    for (int k = 0; k < NK; k++)
#pragma unroll
                        for (int j = 0; j < 3; j++) acc_mad(acc[k][j], g[3 * k + j], v);
                }
            }
            return;
        }
        uint64_t g[3 * NK];
#pragma unroll
        for (int i = 0; i < 3 * NK; i++) g[i] = w[i];
        for (uint32_t cc = 0; cc < cw; cc++) {
            const uint64_t v = tile[t][cc];
            uint64_t cur[3 * NK];
#pragma unroll
            for (int i = 0; i < 3 * NK; i++) cur[i] = g[i];
            w += cc + 1 < cw ? 3 * NK : 0;
#pragma unroll
            for (int i = 0; i < 3 * NK; i++) g[i] = w[i];
#pragma unroll
            for (int k = 0; k < NK; k++) {
                if (cur[3 * k] | cur[3 * k + 1] | cur[3 * k + 2]) {
#pragma unroll
                    for (int j = 0; j < 3; j++) acc_mad_uniform(acc[k][j], cur[3 * k + j], v);
                }
            }
        }
    };
    // equal chunks of at most DEEP_CHUNK columns
    auto width = [](uint64_t cols) -> uint32_t {
        const uint32_t n = (uint32_t)((cols + DEEP_CHUNK - 1) / DEEP_CHUNK);
        return n ? (uint32_t)((cols + n - 1) / n) : 0;
    };
    acc128 acc[KA][3];
#pragma unroll
    for (int k = 0; k < KA; k++)
#pragma unroll
        for (int j = 0; j < 3; j++) acc_zero(acc[k][j]);
    const uint64_t *w = a.gtr;
    for (int sgi = 0; sgi < 2; sgi++) {
        const DeepSegment s = a.trace[sgi];
        const uint32_t cols = (uint32_t)s.cols, cm = width(cols);
        if (!cols) continue;
        fetch(s, 0, cm, w, 3 * KA);
        for (uint32_t j0 = 0; j0 < cols; j0 += cm) {
            const uint32_t cw = cols - j0 < cm ? cols - j0 : cm;
            stage();
            const uint32_t next = j0 + cm;
            if (next < cols) fetch(s, next, cols - next < cm ? cols - next : cm, w + (uint64_t)cw * 3 * KA, 3 * KA);
            accumulate(acc, w, cw);
            w += (uint64_t)cw * 3 * KA;
        }
    }
    fp3 tk[K];
#pragma unroll
    for (int k = 0; k < KA; k++) tk[k] = fp3{acc_reduce(acc[k][0]), acc_reduce(acc[k][1]), acc_reduce(acc[k][2])};
#pragma unroll
    for (int k = KA; k < K; k++) tk[k] = f3_mul(ld3(a.rpow + 3 * k), tk[KA - 1]);
    fp3 r = fp3{0, 0, 0};
    if (p < N) {
#pragma unroll
        for (int k = 0; k < K; k++)
            r = f3_add(r, f3_mul(ld3(a.inv_den + 3 * (k * N + p)), f3_sub(tk[k], ld3(a.consts + 3 * k))));
    }
    if (a.parts.cols) {
        const uint32_t cols = (uint32_t)a.parts.cols, cm = width(cols);
        acc128 ha[1][3];
#pragma unroll
        for (int j = 0; j < 3; j++) acc_zero(ha[0][j]);
        for (uint32_t j0 = 0; j0 < cols; j0 += cm) {
            const uint32_t cw = cols - j0 < cm ? cols - j0 : cm;
            fetch(a.parts, j0, cw, a.gh + 3 * j0, 3);
            stage();
            accumulate(ha, a.gh + 3 * j0, cw);
        }
        if (p < N) {
            const fp3 hs = fp3{acc_reduce(ha[0][0]), acc_reduce(ha[0][1]), acc_reduce(ha[0][2])};
            r = f3_add(r, f3_mul(ld3(a.inv_den + 3 * (K * N + p)), f3_sub(hs, ld3(a.consts + 3 * K))));
        }
    }
    if (p < N) st3(a.out + 3 * p, r);
}

// Where the weights come from. Scalar loads with scalar operands win where several
// blocks a CU hide their latency, one trip to the L2 per column, and above all
// where weights are zero; with fewer blocks, and where the weights outgrow the scalar
// cache, the chunk's weights through LDS do. deep_rows, scalar against LDS: two
// sums of 2^20 x 200 471 against 488 us (one weight in two zero 394 against 479), of
// 2^18 x 600 366 against 358 (304 against 349), but of 2^17 x 600 279 against 200,
// 2^14 x 64 44 against 24, 2^12 x 1480 731 against 295. One sum and four are never
// better off scalar (2^20 x 64 172 against 162 and 401 against 364); three (weights
// that are not geometric) are from 2^20 rows on with weights that fit the 16 KiB
// cache (64 columns 284 against 304, 200 columns 644 against 651, 400 columns 1446
// against 1166; 2^18 x 200 216 against 177).
template <int K, int KA>
static void launch_deep(hipStream_t st, const DeepArgs &a) {
    const uint64_t blocks = (a.N + 255) / 256, weights = 24 * KA * (a.trace[0].cols + a.trace[1].cols);
    if constexpr (KA == 2 || KA == 3) {
        if (KA == 2 ? blocks >= 1024 : blocks >= 4096 && weights <= (16u << 10)) {
            hipLaunchKernelGGL((deep_kernel<K, KA, false>), dim3((unsigned)blocks), dim3(256), 0, st, a);
            return;
        }
    }
    hipLaunchKernelGGL((deep_kernel<K, KA, true>), dim3((unsigned)blocks), dim3(256), 0, st, a);
}
}  // namespace lvm

using namespace lvm;

namespace {
unsigned log2u(uint64_t x) { return (unsigned)__builtin_ctzll(x); }

struct Scratch {
    std::vector<void *> ptrs;
    ~Scratch() {
        for (void *p : ptrs) lvm_free(p);
    }
    template <class T>
    int get(T **out, size_t bytes) {
        void *p = nullptr;
        hipError_t e = lvm_malloc(&p, bytes ? bytes : 8);
        if (e != hipSuccess) return fail(LVM_ERR_NOMEM, std::string("device allocation failed: ") + hipGetErrorString(e));
        ptrs.push_back(p);
        *out = (T *)p;
        return LVM_OK;
    }
};

#define TRYS(x)                        \
    do {                               \
        int _rc = (x);                 \
        if (_rc != LVM_OK) return _rc; \
    } while (0)

void launch_batch_inverse(const uint64_t *in, uint64_t *out, uint64_t n, hipStream_t st) {
    if (!n) return;
    // ~64 elements per thread amortise the one inversion each thread performs
    uint64_t threads = (n + 63) / 64;
    if (threads < 256) threads = n < 256 ? n : 256;
    uint64_t blocks = (threads + 255) / 256;
    hipLaunchKernelGGL(batch_inverse_fp3_kernel, dim3((unsigned)blocks), dim3(256), 0, st, in, out, n);
}

// host Fp3 helpers
struct H3 {
    uint64_t c[3];
};
H3 h3mul(H3 a, H3 b) {
    fp3 r = f3_mul(fp3{a.c[0], a.c[1], a.c[2]}, fp3{b.c[0], b.c[1], b.c[2]});
    return H3{{r.c0, r.c1, r.c2}};
}
}  // namespace

extern "C" {

int lvm_batch_inverse_ext3_dev(const uint64_t *dev_in, uint64_t *dev_out, size_t n) {
    if ((!dev_in || !dev_out) && n) return fail(LVM_ERR_ARG, "null argument");
    if (dev_in == dev_out && n) return fail(LVM_ERR_ARG, "in and out must differ");
    Device *d = device_state();
    if (!d) return LVM_ERR_DEVICE;
    if (take_injected_fault()) return fail(LVM_ERR_INJECTED, "injected fault");
    {
        ProfScope ps("batch_inverse", thread_stream(d));
        launch_batch_inverse(dev_in, dev_out, n, thread_stream(d));
    }
    LVM_HIP(hipGetLastError());
    LVM_HIP(hipStreamSynchronize(thread_stream(d)));
    return LVM_OK;
}

int lvm_batch_inverse_ext3(const uint64_t *in, uint64_t *out, size_t n) {
    if ((!in || !out) && n) return fail(LVM_ERR_ARG, "null argument");
    if (!n) return LVM_OK;
    Device *d = device_state();
    if (!d) return LVM_ERR_DEVICE;
    Scratch s;
    uint64_t *di, *dout;
    TRYS(s.get(&di, n * 24));
    TRYS(s.get(&dout, n * 24));
    LVM_HIP(hipMemcpyAsync(di, in, n * 24, hipMemcpyHostToDevice, thread_stream(d)));
    int rc = lvm_batch_inverse_ext3_dev(di, dout, n);
    if (rc) return rc;
    LVM_HIP(hipMemcpyAsync(out, dout, n * 24, hipMemcpyDeviceToHost, thread_stream(d)));
    LVM_HIP(hipStreamSynchronize(thread_stream(d)));
    return LVM_OK;
}

int lvm_barycentric_base_multi(const lvm_lde *h, uint64_t coset_offset, const uint64_t *z, size_t K, uint64_t *out) {
    if (!h || !z || !out || K == 0) return fail(LVM_ERR_ARG, "bad barycentric arguments");
    if (K > (size_t)BARY_MAX_K) return fail(LVM_ERR_ARG, "at most 8 evaluation points per call");
    Device *d = device_state();
    if (!d) return LVM_ERR_DEVICE;
    if (take_injected_fault()) return fail(LVM_ERR_INJECTED, "injected fault");
    hipStream_t st = thread_stream(d);
    const uint64_t n = h->n, w = h->w;
    const unsigned logN = log2u(h->N);
    Scratch s;
    uint64_t *dz, *scale, *partial, *vfd, *dout = nullptr;
    const BaryShape shape = bary_shape(n, w, K);
    const uint64_t chunks = shape.chunks;
    TRYS(s.get(&dz, 2 * K * 24));  // the points, then their vanishing factors
    vfd = dz + 3 * K;
    TRYS(s.get(&scale, K * n * 24));
    TRYS(s.get(&partial, chunks * K * w * 24));
    const size_t obytes = K * w * 24;
    const bool direct = obytes <= STAGE_RESULT;  // the combine kernel writes to mapped host memory
    if (!direct) TRYS(s.get(&dout, obytes));
    // vanishing factors n^-1 * g^-n * (z_k^n - g^n) (trace.rs:900-905)
    std::vector<uint64_t> zv(6 * K);
    std::memcpy(zv.data(), z, K * 24);
    uint64_t *vf = zv.data() + 3 * K;
    const uint64_t gn = pow(coset_offset, n), nig = mul(inv((uint64_t)n), inv(gn));
    for (size_t k = 0; k < K; k++) {
        fp3 zn = f3_pow(fp3{z[3 * k], z[3 * k + 1], z[3 * k + 2]}, n);
        fp3 v = f3_mul_base(fp3{sub(zn.c0, gn), zn.c1, zn.c2}, nig);
        vf[3 * k] = v.c0;
        vf[3 * k + 1] = v.c1;
        vf[3 * k + 2] = v.c2;
    }
    StageScope ss(st);
    LVM_HIP(stage_upload(dz, zv.data(), 2 * K * 24, st));
    if (direct) LVM_HIP(stage_result(out, obytes, nullptr, 0, st, (void **)&dout, nullptr));
    {
        ProfScope ps("bary_denoms", st);
        // scale[k][p] = x_p / (z_k - x_p)
        launch_pole_inverse(scale, n, logN, coset_offset, dz, (uint32_t)K, 1, d->tb.fwd_lo, d->tb.fwd_hi, st);
    }
    {
        ProfScope ps("bary_sum", st);
        switch (K) {
        case 1: launch_bary_partial<1>(shape, st, h->lde, w, n, scale, partial); break;
        case 2: launch_bary_partial<2>(shape, st, h->lde, w, n, scale, partial); break;
        case 3: launch_bary_partial<3>(shape, st, h->lde, w, n, scale, partial); break;
        case 4: launch_bary_partial<4>(shape, st, h->lde, w, n, scale, partial); break;
        case 5: launch_bary_partial<5>(shape, st, h->lde, w, n, scale, partial); break;
        case 6: launch_bary_partial<6>(shape, st, h->lde, w, n, scale, partial); break;
        case 7: launch_bary_partial<7>(shape, st, h->lde, w, n, scale, partial); break;
        default: launch_bary_partial<8>(shape, st, h->lde, w, n, scale, partial); break;
        }
        hipLaunchKernelGGL(bary_combine_kernel, dim3((unsigned)(K * w)), dim3(256), 0, st, partial, chunks,
                           (uint32_t)K, w, vfd, dout);
    }
    LVM_HIP(hipGetLastError());
    if (!direct) LVM_HIP(stage_download(out, dout, obytes, st));
    LVM_HIP(stage_sync(st));
    return LVM_OK;
}

int lvm_deep_composition(const lvm_lde *main, const lvm_lde *aux, const lvm_lde *parts, uint64_t coset_offset,
                         const uint64_t *z_points, size_t K, const uint64_t *z_parts, const uint64_t *trace_ood,
                         const uint64_t *parts_ood, const uint64_t *gammas_tr, const uint64_t *gammas_h,
                         uint64_t *dev_out) {
    if (!main || !z_points || !trace_ood || !gammas_tr || !dev_out) return fail(LVM_ERR_ARG, "null argument");
    if (K == 0 || K > (size_t)DEEP_MAX_K) return fail(LVM_ERR_ARG, "1..4 trace evaluation points");
    if ((aux && (aux->N != main->N || aux->w % 3)) || (parts && (parts->N != main->N || parts->w % 3)))
        return fail(LVM_ERR_ARG, "aux/parts tables must share the LDE domain and hold Fp3 columns");
    if (parts && (!z_parts || !parts_ood || !gammas_h)) return fail(LVM_ERR_ARG, "parts need z^P, their OOD values and gammas");
    Device *d = device_state();
    if (!d) return LVM_ERR_DEVICE;
    if (take_injected_fault()) return fail(LVM_ERR_INJECTED, "injected fault");
    hipStream_t st = thread_stream(d);
    const uint64_t N = main->N, wm = main->w, wa = aux ? aux->w / 3 : 0, np = parts ? parts->w / 3 : 0;
    const uint64_t cols = wm + wa;
    const uint32_t npoles = (uint32_t)K + (parts ? 1 : 0);
    // host constants: ct_k = sum_j gt_{j,k} t_j(z_k), ch = sum_j gh_j H_j(z^P)
    std::vector<uint64_t> consts(3 * (K + 1), 0), poles(3 * npoles);
    for (size_t k = 0; k < K; k++) {
        H3 acc{{0, 0, 0}};
        for (uint64_t j = 0; j < cols; j++) {
            const uint64_t *g = gammas_tr + 3 * (j * K + k), *t = trace_ood + 3 * (j * K + k);
            H3 pr = h3mul(H3{{g[0], g[1], g[2]}}, H3{{t[0], t[1], t[2]}});
            for (int c = 0; c < 3; c++) acc.c[c] = add(acc.c[c], pr.c[c]);
        }
        std::memcpy(&consts[3 * k], acc.c, 24);
        std::memcpy(&poles[3 * k], z_points + 3 * k, 24);
    }
    if (parts) {
        H3 acc{{0, 0, 0}};
        for (uint64_t j = 0; j < np; j++) {
            H3 pr = h3mul(H3{{gammas_h[3 * j], gammas_h[3 * j + 1], gammas_h[3 * j + 2]}},
                          H3{{parts_ood[3 * j], parts_ood[3 * j + 1], parts_ood[3 * j + 2]}});
            for (int c = 0; c < 3; c++) acc.c[c] = add(acc.c[c], pr.c[c]);
        }
        std::memcpy(&consts[3 * K], acc.c, 24);
        std::memcpy(&poles[3 * K], z_parts, 24);
    }
    // geometric trace-term weights past k = 1: gt_{j,k} = gt_{j,k-1} * r for all j, k >= 2
    std::vector<uint64_t> rp(3 * K, 0);
    bool geo = K > 2;
    if (geo) {
        const H3 g01{{gammas_tr[3], gammas_tr[4], gammas_tr[5]}}, g02{{gammas_tr[6], gammas_tr[7], gammas_tr[8]}};
        if (canon(g01.c[0]) == 0 && canon(g01.c[1]) == 0 && canon(g01.c[2]) == 0) {
            geo = false;
        } else {
            const fp3 ri = f3_inv(fp3{g01.c[0], g01.c[1], g01.c[2]});
            const H3 r = h3mul(g02, H3{{ri.c0, ri.c1, ri.c2}});
            H3 pw{{1, 0, 0}};
            for (size_t k = 2; k < K; k++) {
                pw = h3mul(pw, r);
                std::memcpy(&rp[3 * k], pw.c, 24);
            }
            for (uint64_t j = 0; j < cols && geo; j++)
                for (size_t k = 2; k < K && geo; k++) {
                    const uint64_t *a = gammas_tr + 3 * (j * K + k - 1), *b = gammas_tr + 3 * (j * K + k);
                    const H3 want = h3mul(H3{{a[0], a[1], a[2]}}, r);
                    for (int c = 0; c < 3; c++) geo = geo && canon(want.c[c]) == canon(b[c]);
                }
        }
    }
    // the weights by base word: an Fp3 column's three words weigh g, w g, w^2 g
    const uint32_t KA = geo ? 2 : (uint32_t)K;
    const uint64_t words = wm + 3 * wa;
    std::vector<uint64_t> wt(3 * KA * words), wh(9 * np);
    auto times_w = [](const uint64_t *g, uint64_t *o) {  // w g (w^3 = 2)
        const uint64_t g0 = g[0], g1 = g[1], g2 = g[2];
        o[0] = dbl(g2);
        o[1] = g0;
        o[2] = g1;
    };
    for (uint64_t j = 0; j < cols; j++)
        for (uint32_t k = 0; k < KA; k++) {
            const uint64_t *g = gammas_tr + 3 * (j * K + k);
            const uint64_t w0 = j < wm ? j : wm + 3 * (j - wm);
            std::memcpy(&wt[3 * (w0 * KA + k)], g, 24);
            if (j >= wm) {
                times_w(&wt[3 * (w0 * KA + k)], &wt[3 * ((w0 + 1) * KA + k)]);
                times_w(&wt[3 * ((w0 + 1) * KA + k)], &wt[3 * ((w0 + 2) * KA + k)]);
            }
        }
    for (uint64_t j = 0; j < np; j++) {
        std::memcpy(&wh[9 * j], gammas_h + 3 * j, 24);
        times_w(&wh[9 * j], &wh[9 * j + 3]);
        times_w(&wh[9 * j + 3], &wh[9 * j + 6]);
    }
    Scratch s;
    uint64_t *inv_den, *dargs;
    TRYS(s.get(&inv_den, (uint64_t)npoles * N * 24));
    // poles, consts, powers and weights in one upload
    std::vector<uint64_t> blob;
    auto put = [&](const void *p, size_t bytes) {
        const size_t at = blob.size();
        blob.resize(at + (bytes + 7) / 8);
        if (bytes) std::memcpy(&blob[at], p, bytes);
        return at;
    };
    const size_t o_poles = put(poles.data(), npoles * 24), o_consts = put(consts.data(), (K + 1) * 24), o_rp = put(rp.data(), K * 24);
    const size_t o_wt = put(wt.data(), wt.size() * 8), o_wh = put(wh.data(), wh.size() * 8);
    TRYS(s.get(&dargs, blob.size() * 8));
    StageScope ss(st);
    LVM_HIP(stage_upload(dargs, blob.data(), blob.size() * 8, st));
    {
        ProfScope ps("deep_denoms", st);
        // 1 / (x - z) (XMinusZ, crypto/math-cuda/src/inverse.rs:241-300)
        launch_pole_inverse(inv_den, N, log2u(N), coset_offset, dargs + o_poles, npoles, 0, d->tb.fwd_lo, d->tb.fwd_hi, st);
    }
    {
        ProfScope ps("deep_rows", st);
        const DeepArgs a{N,
                         {{main->lde, wm}, {aux ? aux->lde : nullptr, 3 * wa}},
                         {parts ? parts->lde : nullptr, 3 * np},
                         dargs + o_wt, dargs + o_wh, dargs + o_consts,
                         dargs + o_rp, inv_den, dev_out};
        switch (K * 2 + (geo ? 1 : 0)) {
        case 2: launch_deep<1, 1>(st, a); break;
        case 4: launch_deep<2, 2>(st, a); break;
        case 6: launch_deep<3, 3>(st, a); break;
        case 7: launch_deep<3, 2>(st, a); break;
        case 8: launch_deep<4, 4>(st, a); break;
        default: launch_deep<4, 2>(st, a); break;
        }
    }
    LVM_HIP(hipGetLastError());
    LVM_HIP(stage_sync(st));
    return LVM_OK;
}

}  // extern "C"

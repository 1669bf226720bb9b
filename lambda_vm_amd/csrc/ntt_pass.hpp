// The NTT pass kernels (layout, passes and remaps described in ntt.hip).
#pragma once
#include <type_traits>

#include "lvm_internal.hpp"

namespace lvm {

// w_{2^32}^e via the two-level table (canonical)
__device__ __forceinline__ uint64_t tw32(const uint64_t *lo, const uint64_t *hi, uint32_t e) {
    return cmul(LVM_GLOBAL_CONST(lo)[e & 0xFFFFu], LVM_GLOBAL_CONST(hi)[e >> 16]);
}

// bit reversal of i over `bits` bits, for compile-time indices
constexpr uint32_t bitrev_small(uint32_t i, int bits) {
    uint32_t r = 0;
    for (int b = 0; b < bits; b++) r |= ((i >> b) & 1u) << (bits - 1 - b);
    return r;
}

// log2 of w_R as a power of two (w_R = w_16^(16/R)), forward and inverse
constexpr int log2_root(int R, bool inverse) { return ((inverse ? 36 : 156) * (16 / R)) % 192; }

constexpr uint64_t cmod_mul(uint64_t a, uint64_t b) { return (uint64_t)(((unsigned __int128)a * b) % P); }
constexpr uint64_t cmod_pow(uint64_t a, uint64_t e) {
    uint64_t r = 1;
    while (e) {
        if (e & 1) r = cmod_mul(r, a);
        a = cmod_mul(a, a);
        e >>= 1;
    }
    return r;
}
// w_16 = w_{2^32}^(2^28) of the field's root of unity, and its inverse
static_assert(cmod_pow(1753635133440165772ull, 1ull << 28) == cmod_pow(2, 156), "forward w_16 is 2^156");
static_assert(cmod_mul(cmod_pow(2, 156), cmod_pow(2, 36)) == 1, "inverse w_16 is 2^36");

// DIF butterfly (u, v) -> (u + v, (u - v) * 2^T); where the cheaper form of
// the power of two computes -2^T, the subtraction is swapped instead
template <int T>
__device__ __forceinline__ void bfly_pow2(uint64_t &u, uint64_t &v) {
    const uint64_t a = u, b = v;
    u = cadd(a, b);
    if constexpr (T % 192 == 0)
        v = csub(a, b);
    else if constexpr (pow2_negates<T>())
        v = cmul_pow2_form<T>(csub(b, a));
    else
        v = cmul_pow2_form<T>(csub(a, b));
}

template <int R, int LOGW, int H, int I>
__device__ __forceinline__ void dif_stage(uint64_t *x) {
    if constexpr (I < R) {
        if constexpr ((I & H) == 0) bfly_pow2<(LOGW * ((I & (H - 1)) * (R / (2 * H)))) % 192>(x[I], x[I + H]);
        dif_stage<R, LOGW, H, I + 1>(x);
    }
}

// In-register radix-2 DIF DFT of size R <= 16 with root 2^LOGW: natural
// input order, bit-reversed output order, canonical values.
template <int R, int LOGW, int H = R / 2>
__device__ __forceinline__ void dif_small(uint64_t *x) {
    if constexpr (H >= 1) {
        dif_stage<R, LOGW, H, 0>(x);
        dif_small<R, LOGW, H / 2>(x);
    }
}

template <int R>
__device__ __forceinline__ void dft_small(uint64_t *x, bool inverse) {
    if (inverse)
        dif_small<R, log2_root(R, true)>(x);
    else
        dif_small<R, log2_root(R, false)>(x);
}

// ---- tiling ----
constexpr int PASS_C = 16, PASS_T = 256;  // words and threads per tile; 32-word tiles of 512 threads measured slower

// n / d with inv = udiv_inv(d)
__device__ __forceinline__ uint32_t udiv(uint32_t n, uint32_t d, uint32_t inv) {
    const uint32_t q = __umulhi(n, inv);
    return n - q * d >= d ? q + 1 : q;
}

// Body of one pass for block `block` of the table's tiles.
//
// Tiles: run-major windows of PASS_C words. A run is the S rows of one block (run =
// S*m words, below 2^31), lane c of window w takes word w*16 + c, i.e. row jlo =
// word / m and column word % m. In the last pass (S = 1) of a table of at most 8
// columns a tile packs `units` = 16 / m whole runs side by side. NJ: rows a window
// can span, each with factors of its own in LDS (1 for m a multiple of 16, 2 for
// most m, 4 for m >= 4); 0: more than 4 (m < 4), every lane forms its factors
// itself.
// COSET: the first pass of a coset expansion (bit-reversed input rows,
// pre-multiplied, several cosets from one read).
template <int LOG_R1, int LOG_R2, bool COSET, int NJ>
__device__ __forceinline__ void ntt_pass_body(const PassArgs &a, uint32_t block) {
    constexpr int R1 = 1 << LOG_R1, R2 = 1 << LOG_R2, R = R1 * R2, LOG_R = LOG_R1 + LOG_R2;
    constexpr int C = PASS_C, NT = PASS_T;
    // TPC = min(R1, R2) threads per column; each holds R / TPC elements in
    // both rounds: D1 = R2 / TPC size-R1 DFTs in round 1, D2 = R1 / TPC
    // size-R2 DFTs in round 2 (for R1 != R2 no thread idles in either round)
    constexpr int TPC = R1 < R2 ? R1 : R2;
    constexpr int D1 = R2 / TPC, D2 = R1 / TPC;
    constexpr int TILES = NT / (C * TPC);
    constexpr int NL = NJ ? NJ : 1;  // factor tables in LDS
    static_assert(TILES >= 1 && D1 * R1 == D2 * R2, "tile shape");

    __shared__ uint64_t s_data[TILES][R * C];
    __shared__ uint64_t s_pre[COSET && NJ ? TILES : 1][NL][COSET && NJ ? R : 1];
    __shared__ uint64_t s_post[NJ ? TILES : 1][NL][NJ ? R : 1];
    __shared__ uint64_t s_tw[R];

    const int tid = threadIdx.x;
    const int c = tid % C;
    const int tc = (tid / C) % TPC;
    const int tl = tid / (C * TPC);
    // the cosets of a small table are shared out over copies of its blocks
    const uint32_t cg = COSET ? block / a.blocks : 0;
    const uint32_t tile = (block - cg * a.blocks) * TILES + tl;
    const bool t_ok = tile < a.tiles;

    const uint32_t log_s = a.log_s;
    // unit: the tile's run; jb: its window's first row, jl: the lane's row past it
    const uint32_t unit = t_ok ? udiv(tile, a.wins, a.win_inv) : 0;
    const uint32_t w0 = t_ok ? (tile - unit * a.wins) * C : 0;
    bool c_ok = t_ok && w0 + c < a.run;
    const uint32_t word = c_ok ? w0 + c : w0;  // a lane past the run reads its window's first word
    uint64_t blk;
    uint32_t jb, jlo, col, nj = 1;
    if (NJ && a.units > 1) {
        const uint32_t u = udiv(word, a.m, a.m_inv);
        blk = (uint64_t)unit * a.units + u;
        c_ok = c_ok && blk < a.total_groups;
        if (!c_ok) blk = 0;
        jb = jlo = 0;
        col = word - u * a.m;
    } else {
        blk = unit;
        jb = udiv(w0, a.m, a.m_inv);
        jlo = udiv(word, a.m, a.m_inv);
        col = word - jlo * a.m;
        if (NJ > 1) nj = udiv(w0 + C - 1 < a.run ? w0 + C - 1 : a.run - 1, a.m, a.m_inv) - jb + 1;
    }
    const uint32_t jl = NJ > 1 ? jlo - jb : 0;
    const uint64_t rowb = blk << a.log_msub;  // logical row of t = 0, j = 0
    const uint64_t row0 = rowb + jlo;

    // position t holds frequency k1 = bitrev_R(t): w_M^(j*k1)
    auto post_factor = [&](uint32_t j, uint32_t t) -> uint64_t {
        return tw32(a.tw_lo, a.tw_hi, (uint32_t)(((uint64_t)j * bitrev(t, LOG_R)) << (32 - a.log_msub)));
    };
    // weights[row] * w_N^(coset*row)
    auto pre_factor = [&](uint32_t coset, uint64_t lrow) -> uint64_t {
        return cmul(LVM_GLOBAL_CONST(a.weights)[lrow],
                    tw32(a.shift_lo, a.shift_hi, (uint32_t)(((uint64_t)coset * lrow) << (32 - a.shift_log))));
    };

    // inner twiddles w_R^e = w_256^(e*256/R), e < R
    for (int e = tid; e < R; e += NT) s_tw[e] = LVM_GLOBAL_CONST(a.tw_r)[e << (8 - LOG_R)];
    const int tin = tid % (C * TPC);
    // per-tile post-twiddle factors, shared by the words of a row
    if (NJ && log_s && t_ok) {
        for (uint32_t e = tin; e < R * nj; e += C * TPC) s_post[tl][e >> LOG_R][e & (R - 1)] = post_factor(jb + (e >> LOG_R), e & (R - 1));
    }

    uint64_t x[R1 > R2 ? R1 : R2];
    uint64_t xin[D1][R1];
    // Input element (d, i) of a thread is t = t0 + R2*i with t0 = tc + TPC*d,
    // logical row rowA + ((TPC*d + R2*i) << log_s) with rowA = row0 + (tc << log_s):
    // disjoint bit fields, so with bit-reversed input rows (over in_bitrev_bits
    // = log_msub bits) the physical row is bitrev(rowA) + bitrev_R(TPC*d + R2*i)
    // << (bits - log_s - LOG_R). Either way a per-thread base plus a uniform
    // stride per element, and the loads are issued back to back.
    const uint64_t rowA = row0 + ((uint64_t)tc << log_s);
    const uint64_t physA = COSET ? (uint64_t)bitrev((uint32_t)rowA, a.in_bitrev_bits) : rowA;
    const gmem_u64 *src = LVM_GLOBAL_CONST(a.in) + physA * a.in_pitch + col;
    const uint64_t in_step = (uint64_t)a.in_pitch << (COSET ? a.in_bitrev_bits - log_s - LOG_R : log_s);
#pragma unroll
    for (int d = 0; d < D1; d++) {
#pragma unroll
        for (int i = 0; i < R1; i++) {
            const uint32_t u = (uint32_t)(TPC * d + R2 * i);
            const uint64_t sel = COSET ? bitrev_small(u, LOG_R) : u;
            xin[d][i] = src[sel * in_step];
        }
    }

    const uint32_t ncos = COSET ? a.cosets_per_block : 1u;
    for (uint32_t ci = 0; ci < ncos; ci++) {
    const uint32_t coset = cg * ncos + ci;
    if constexpr (COSET && NJ) {
        if (t_ok) {
            for (uint32_t e = tin; e < R * nj; e += C * TPC)
                s_pre[tl][e >> LOG_R][e & (R - 1)] = pre_factor(coset, rowb + jb + (e >> LOG_R) + ((uint64_t)(e & (R - 1)) << log_s));
        }
    }
    __syncthreads();

    // ---- round 1: size-R1 DFTs over t = t0 + R2*i, then w_R^(t0*k_a) ----
#pragma unroll
    for (int d = 0; d < D1; d++) {
        const int t0 = tc + TPC * d;
#pragma unroll
        for (int i = 0; i < R1; i++) {
            if constexpr (COSET)
                x[i] = cmul(xin[d][i], NJ ? s_pre[tl][jl][t0 + R2 * i]
                                          : pre_factor(coset, row0 + ((uint64_t)(t0 + R2 * i) << log_s)));
            else
                x[i] = a.in_canonical ? xin[d][i] : ccanon(xin[d][i]);
        }
        dft_small<R1>(x, a.inverse);
        // position i holds frequency k_a = bitrev_R1(i)
        if constexpr (R2 > 1) {
#pragma unroll
            for (int i = 1; i < R1; i++) x[i] = cmul(x[i], s_tw[t0 * (int)bitrev_small(i, LOG_R1)]);
        }
#pragma unroll
        for (int i = 0; i < R1; i++) s_data[tl][(t0 + R2 * i) * C + c] = x[i];
    }
    __syncthreads();

    // ---- round 2: size-R2 DFTs over t0 at t = R2*t1 + t0 ----
    const uint64_t obase = COSET ? (uint64_t)bitrev(coset, a.coset_bits) * a.out_coset_rows : 0;
    // output q = R2*t1 + i is row obase + row0 + (q << log_s): a base and a uniform stride
    gmem_u64 *dst = LVM_GLOBAL(a.out) + (obase + row0 + ((uint64_t)(R2 * tc) << log_s)) * a.out_pitch + col;
    const uint64_t out_step = (uint64_t)a.out_pitch << log_s;
#pragma unroll
    for (int d = 0; d < D2; d++) {
        const int t1 = tc + TPC * d;
#pragma unroll
        for (int i = 0; i < R2; i++) x[i] = s_data[tl][(R2 * t1 + i) * C + c];
        dft_small<R2>(x, a.inverse);
        if (c_ok) {
#pragma unroll
            for (int i = 0; i < R2; i++) {
                uint64_t v = x[i];
                if (log_s) v = cmul(v, NJ ? s_post[tl][jl][R2 * t1 + i] : post_factor(jlo, R2 * t1 + i));
                dst[(R2 * TPC * d + i) * out_step] = v;
            }
        }
    }
    if constexpr (COSET) __syncthreads();  // the LDS tile and factors are rewritten by the next coset
    }
}

// Calls f with the compile-time radices of a pass of 2^r points.
template <class F>
static void with_radix(int r, F &&f) {
    switch (r) {
    case 1: f(std::integral_constant<int, 1>(), std::integral_constant<int, 0>()); break;
    case 2: f(std::integral_constant<int, 1>(), std::integral_constant<int, 1>()); break;
    case 3: f(std::integral_constant<int, 2>(), std::integral_constant<int, 1>()); break;
    case 4: f(std::integral_constant<int, 2>(), std::integral_constant<int, 2>()); break;
    case 5: f(std::integral_constant<int, 3>(), std::integral_constant<int, 2>()); break;
    case 6: f(std::integral_constant<int, 3>(), std::integral_constant<int, 3>()); break;
    case 7: f(std::integral_constant<int, 4>(), std::integral_constant<int, 3>()); break;
    case 8: f(std::integral_constant<int, 4>(), std::integral_constant<int, 4>()); break;
    default: break;
    }
}

// Calls f with NJ for a pass whose windows span `rows` rows.
template <class F>
static void with_rows(uint32_t rows, F &&f) {
    if (rows == 1)
        f(std::integral_constant<int, 1>());
    else if (rows == 2)
        f(std::integral_constant<int, 2>());
    else if (rows <= 4)
        f(std::integral_constant<int, 4>());
    else
        f(std::integral_constant<int, 0>());
}

}  // namespace lvm

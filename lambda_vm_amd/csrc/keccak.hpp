// Keccak-f[1600] (FIPS 202 section 3: theta, rho, pi, chi, iota; 24 rounds)
// for gfx950. Each 64-bit lane is held as two 32-bit VGPRs (lo, hi):
//  - column parities and theta use v_bitop3_b32 as a 3-input XOR (LUT 0x96),
//    and the theta term D[x] is folded into the per-lane XOR (A ^ C[x-1] ^
//    rot(C[x+1], 1) is one 3-input XOR per half). v_xor_b32 alone issues every
//    2.9 cycles per wave against 4.7 for v_bitop3_b32, but not in this mix:
//    parities of two-input XORs measured slower (row-pair leaves of 2^24 x 64:
//    8.27 against 7.7-7.9 ms), D[x] formed first and XORed in the same;
//  - a 64-bit rotate is two v_alignbit_b32 (funnel shifts of the halves);
//  - chi, a ^ (~b & c), is one v_bitop3_b32 per half (LUT 0xD2 for
//    operands (a, b, c), i.e. f(0xF0, 0xCC, 0xAA)).
// ~180 VALU instructions per round. Keccak-256 framing (rate 136 bytes, pad
// 0x01 ... 0x80, little-endian lanes) is what the reference's Merkle leaves,
// nodes and transcript use (crypto/crypto/src/hash/platform_keccak.rs:
// 124-125, sha3 0.10.8; crypto/math-cuda/kernels/keccak.cu:114-138 states the
// same framing).
#pragma once
#include "field.hpp"

namespace lvm {

__constant__ static const uint32_t KECCAK_RC_LO[24] = {
    0x00000001u, 0x00008082u, 0x0000808au, 0x80008000u, 0x0000808bu, 0x80000001u, 0x80008081u, 0x00008009u,
    0x0000008au, 0x00000088u, 0x80008009u, 0x8000000au, 0x8000808bu, 0x0000008bu, 0x00008089u, 0x00008003u,
    0x00008002u, 0x00000080u, 0x0000800au, 0x8000000au, 0x80008081u, 0x00008080u, 0x80000001u, 0x80008008u};
__constant__ static const uint32_t KECCAK_RC_HI[24] = {
    0x00000000u, 0x00000000u, 0x80000000u, 0x80000000u, 0x00000000u, 0x00000000u, 0x80000000u, 0x80000000u,
    0x00000000u, 0x00000000u, 0x00000000u, 0x00000000u, 0x00000000u, 0x80000000u, 0x80000000u, 0x80000000u,
    0x80000000u, 0x80000000u, 0x00000000u, 0x80000000u, 0x80000000u, 0x80000000u, 0x00000000u, 0x80000000u};

__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
    // lanes known to be zero (the first round of a one-block message) drop out
    if (__builtin_constant_p(a) && a == 0) return b ^ c;
    if (__builtin_constant_p(b) && b == 0) return a ^ c;
    if (__builtin_constant_p(c) && c == 0) return a ^ b;
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}
// a ^ (~b & c)
__device__ __forceinline__ uint32_t chi(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0xD2);
}

// rotate the 64-bit value (hi, lo) left by N, 0 <= N < 64
template <int N>
__device__ __forceinline__ void rotl(uint32_t hi, uint32_t lo, uint32_t &oh, uint32_t &ol) {
    if constexpr (N == 0) {
        oh = hi;
        ol = lo;
    } else if constexpr (N == 32) {
        oh = lo;
        ol = hi;
    } else if constexpr (N < 32) {
        oh = __builtin_amdgcn_alignbit(hi, lo, 32 - N);
        ol = __builtin_amdgcn_alignbit(lo, hi, 32 - N);
    } else {
        oh = __builtin_amdgcn_alignbit(lo, hi, 64 - N);
        ol = __builtin_amdgcn_alignbit(hi, lo, 64 - N);
    }
}

// C[x] and rot(C[x], 1) of theta
__device__ __forceinline__ void theta_c(const uint32_t l[25], const uint32_t h[25], uint32_t Cl[5], uint32_t Ch[5],
                                        uint32_t Rl[5], uint32_t Rh[5]) {
#pragma unroll
    for (int x = 0; x < 5; x++) {
        Cl[x] = xor3(xor3(l[x], l[x + 5], l[x + 10]), l[x + 15], l[x + 20]);
        Ch[x] = xor3(xor3(h[x], h[x + 5], h[x + 10]), h[x + 15], h[x + 20]);
    }
#pragma unroll
    for (int x = 0; x < 5; x++) rotl<1>(Ch[x], Cl[x], Rh[x], Rl[x]);
}

// B[dst] = rot(A[src] ^ C[x-1] ^ rot(C[x+1], 1), R) where x = src % 5
#define LVM_KB(dst, src, R)                                                                      \
    rotl<R>(xor3(h[src], Ch[((src) + 4) % 5], Rh[((src) + 1) % 5]),                             \
            xor3(l[src], Cl[((src) + 4) % 5], Rl[((src) + 1) % 5]), bh[dst], bl[dst])

// one round (theta, rho, pi, chi, iota) on the 32-bit halves
__device__ __forceinline__ void keccak_round_32(uint32_t l[25], uint32_t h[25], int round) {
    uint32_t Cl[5], Ch[5], Rl[5], Rh[5];
    theta_c(l, h, Cl, Ch, Rl, Rh);
    uint32_t bl[25], bh[25];
    // theta + rho + pi: B[y, 2x+3y] = rot(A[x,y] ^ D[x], r[x,y]), lane index x + 5y
    LVM_KB(0, 0, 0);
    LVM_KB(10, 1, 1);
    LVM_KB(20, 2, 62);
    LVM_KB(5, 3, 28);
    LVM_KB(15, 4, 27);
    LVM_KB(16, 5, 36);
    LVM_KB(1, 6, 44);
    LVM_KB(11, 7, 6);
    LVM_KB(21, 8, 55);
    LVM_KB(6, 9, 20);
    LVM_KB(7, 10, 3);
    LVM_KB(17, 11, 10);
    LVM_KB(2, 12, 43);
    LVM_KB(12, 13, 25);
    LVM_KB(22, 14, 39);
    LVM_KB(23, 15, 41);
    LVM_KB(8, 16, 45);
    LVM_KB(18, 17, 15);
    LVM_KB(3, 18, 21);
    LVM_KB(13, 19, 8);
    LVM_KB(14, 20, 18);
    LVM_KB(24, 21, 2);
    LVM_KB(9, 22, 61);
    LVM_KB(19, 23, 56);
    LVM_KB(4, 24, 14);
    // chi
#pragma unroll
    for (int y = 0; y < 25; y += 5) {
#pragma unroll
        for (int x = 0; x < 5; x++) {
            l[y + x] = chi(bl[y + x], bl[y + (x + 1) % 5], bl[y + (x + 2) % 5]);
            h[y + x] = chi(bh[y + x], bh[y + (x + 1) % 5], bh[y + (x + 2) % 5]);
        }
    }
    // iota
    l[0] ^= KECCAK_RC_LO[round];
    h[0] ^= KECCAK_RC_HI[round];
}

// The last round as far as a 32-byte digest needs it: row 0 of its B, lanes 0..3.
__device__ __forceinline__ void keccak_last_round_digest(uint32_t l[25], uint32_t h[25]) {
    uint32_t Cl[5], Ch[5], Rl[5], Rh[5];
    theta_c(l, h, Cl, Ch, Rl, Rh);
    uint32_t bl[5], bh[5];
    LVM_KB(0, 0, 0);
    LVM_KB(1, 6, 44);
    LVM_KB(2, 12, 43);
    LVM_KB(3, 18, 21);
    LVM_KB(4, 24, 14);
#pragma unroll
    for (int x = 0; x < 4; x++) {
        l[x] = chi(bl[x], bl[(x + 1) % 5], bl[(x + 2) % 5]);
        h[x] = chi(bh[x], bh[(x + 1) % 5], bh[(x + 2) % 5]);
    }
    l[0] ^= KECCAK_RC_LO[23];
    h[0] ^= KECCAK_RC_HI[23];
}
#undef LVM_KB

// The 24 rounds as a loop (one copy of the round body keeps the code small).
__device__ __forceinline__ void keccak_f1600_32(uint32_t l[25], uint32_t h[25]) {
#pragma unroll 1
    for (int round = 0; round < 24; round++) keccak_round_32(l, h, round);
}

// The permutation that ends a Keccak-256: only lanes 0..3 (the digest) come
// out, the last round's other lanes are not formed. FIRST: the first round is
// a copy of its own, for states whose zero lanes are known at compile time
// (one-block messages). Together 3.5 % of a permutation.
template <bool FIRST>
__device__ __forceinline__ void keccak_f1600_32_digest(uint32_t l[25], uint32_t h[25]) {
    if constexpr (FIRST) keccak_round_32(l, h, 0);
#pragma unroll 1
    for (int round = FIRST ? 1 : 0; round < 23; round++) keccak_round_32(l, h, round);
    keccak_last_round_digest(l, h);
}

// Keccak-256 of exactly two 32-byte nodes (one permutation): lanes 0..7 hold
// left || right, pad byte 0x01 at lane 8, 0x80 at the top of lane 16.
__device__ __forceinline__ void keccak_pair_node(const uint64_t lft[4], const uint64_t rgt[4], uint64_t out[4]) {
    uint32_t l[25], h[25];
#pragma unroll
    for (int i = 0; i < 25; i++) l[i] = h[i] = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        l[i] = (uint32_t)lft[i];
        h[i] = (uint32_t)(lft[i] >> 32);
        l[4 + i] = (uint32_t)rgt[i];
        h[4 + i] = (uint32_t)(rgt[i] >> 32);
    }
    l[8] = 0x01;
    h[16] = 0x80000000u;
    keccak_f1600_32_digest<true>(l, h);
#pragma unroll
    for (int i = 0; i < 4; i++) out[i] = ((uint64_t)h[i] << 32) | l[i];
}

// ---- one permutation over 16 lanes ----
//
// A single Keccak-f on one lane is a serial chain of ~4300 VALU instructions,
// each taking its wave's issue slot for four cycles whatever the number of
// active lanes: 7.2 us, which every level of a tree top pays with the chip
// idle. Here a 16-lane DPP row holds one state: lane (y, half) = bits 0..2 and
// bit 3 of the lane number holds the 32-bit halves of row y, x = 0..4 in five
// registers (lanes y = 5..7 hold zero). Per round:
//  - column parities: XOR over the 8 lanes of a half, three DPP steps (zero
//    lanes do not contribute);
//  - theta, and rho as one funnel shift per word with the other half (lane ^ 8)
//    brought by a row rotate; a rotation by 0 or by 32..63 lands in the other
//    half, which the next step's addresses undo;
//  - pi through LDS: every lane stores its five words and reads the five of its
//    new row (row stride 65 words: the reads of a 32-lane half-wave hit
//    distinct banks);
//  - chi is local to the lane.
// About 55 instructions and one LDS round trip per round, four states a wave.
struct CoopKeccak {
    uint32_t sh[5];   // rho: funnel shift of word x
    uint32_t rd[5];   // pi: LDS word of the new row's word x
    uint32_t wr;      // LDS word of word 0 (word x at wr + COOP_ROW * x)
    uint32_t m_lo, m_hi;  // iota: all ones in the lane holding that half of word 0
};
constexpr uint32_t COOP_ROW = 65;
constexpr uint32_t COOP_ZERO = 5 * COOP_ROW;       // a word that stays zero
constexpr uint32_t COOP_WORDS = COOP_ZERO + 1;     // LDS words per wave

// rotation of lane (x, y), index x + 5y
constexpr uint32_t KECCAK_RHO[25] = {0,  1,  62, 28, 27, 36, 44, 6,  55, 20, 3,  10, 43,
                                     25, 39, 41, 45, 15, 21, 8,  18, 2,  61, 56, 14};
constexpr uint64_t rho_of_column(int x) {  // y = 0..4, six bits each
    uint64_t v = 0;
    for (int y = 0; y < 5; y++) v |= (uint64_t)KECCAK_RHO[x + 5 * y] << (6 * y);
    return v;
}
constexpr uint64_t rho_of_row(int y) {  // x = 0..4, six bits each
    uint64_t v = 0;
    for (int x = 0; x < 5; x++) v |= (uint64_t)KECCAK_RHO[x + 5 * y] << (6 * x);
    return v;
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
constexpr int DPP_XOR1 = 0xB1, DPP_XOR2 = 0x4E, DPP_HALF_MIRROR = 0x141, DPP_ROR8 = 0x128;

// Lane constants, and the wave's zero word (call with the wave converged).
__device__ __forceinline__ void coop_setup(CoopKeccak &k, uint32_t *ws) {
    const uint32_t lane = threadIdx.x & 63, y = lane & 7, half = (lane >> 3) & 1, base = lane & 48;
#pragma unroll
    for (int x = 0; x < 5; x++) {
        const uint32_t n = (uint32_t)(rho_of_column(x) >> (6 * y)) & 63u;
        k.sh[x] = (64u - n) & 31u;
    }
#pragma unroll
    for (int X = 0; X < 5; X++) {
        // B[X, Y] comes from lane row X, word x = 3Y + X mod 5
        const uint32_t x = (3 * y + X) % 5;
        const uint32_t n = (uint32_t)(rho_of_row(X) >> (6 * x)) & 63u;
        const uint32_t swap = (n == 0 || n >= 32) ? 1u : 0u;
        k.rd[X] = y < 5 ? x * COOP_ROW + base + ((half ^ swap) << 3) + X : COOP_ZERO;
    }
    k.wr = lane;
    k.m_lo = (y == 0 && half == 0) ? ~0u : 0u;
    k.m_hi = (y == 0 && half == 1) ? ~0u : 0u;
    if (lane == 0) ws[COOP_ZERO] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Keccak-f of the four states of the wave (a[x] of lane (y, half) as above);
// ws: the wave's COOP_WORDS words of LDS. Every lane of the wave takes part.
__device__ __forceinline__ void keccak_f1600_coop(uint32_t a[5], const CoopKeccak &k, uint32_t *ws) {
#pragma unroll
    for (int round = 0; round < 24; round++) {
        uint32_t c[5], r[5];
#pragma unroll
        for (int x = 0; x < 5; x++) c[x] = a[x] ^ dpp<DPP_XOR1>(a[x]);
#pragma unroll
        for (int x = 0; x < 5; x++) c[x] ^= dpp<DPP_XOR2>(c[x]);
#pragma unroll
        for (int x = 0; x < 5; x++) c[x] ^= dpp<DPP_HALF_MIRROR>(c[x]);
#pragma unroll
        for (int x = 0; x < 5; x++) r[x] = __builtin_amdgcn_alignbit(c[x], dpp<DPP_ROR8>(c[x]), 31);
#pragma unroll
        for (int x = 0; x < 5; x++) a[x] = xor3(a[x], c[(x + 4) % 5], r[(x + 1) % 5]);
#pragma unroll
        for (int x = 0; x < 5; x++)
            ws[k.wr + COOP_ROW * x] = __builtin_amdgcn_alignbit(a[x], dpp<DPP_ROR8>(a[x]), k.sh[x]);
        // one wave's LDS accesses stay in order: no wait, only no reordering
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        uint32_t b[5];
#pragma unroll
        for (int x = 0; x < 5; x++) b[x] = ws[k.rd[x]];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int x = 0; x < 5; x++) a[x] = chi(b[x], b[(x + 1) % 5], b[(x + 2) % 5]);
        // a ^ (constant & mask)
        a[0] = __builtin_amdgcn_bitop3_b32(a[0], KECCAK_RC_LO[round], k.m_lo, 0x78);
        a[0] = __builtin_amdgcn_bitop3_b32(a[0], KECCAK_RC_HI[round], k.m_hi, 0x78);
    }
}

// The state of Keccak-256 over two 32-byte nodes (one permutation): `src` is
// the 16 words left || right, read only by lanes with `on`.
template <class Ptr>
__device__ __forceinline__ void coop_load_pair(uint32_t a[5], Ptr src, bool on) {
    const uint32_t lane = threadIdx.x & 63, y = lane & 7, half = (lane >> 3) & 1;
#pragma unroll
    for (int x = 0; x < 5; x++) {
        const uint32_t i = 5 * y + x;  // 64-bit lane of the state
        uint32_t v = 0;
        if (on && i < 8) v = src[2 * i + half];
        if (i == 8 && half == 0) v = 0x01;
        if (i == 16 && half == 1) v = 0x80000000u;
        a[x] = v;
    }
}

}  // namespace lvm

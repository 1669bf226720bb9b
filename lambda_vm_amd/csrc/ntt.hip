// Batched row-major Goldilocks NTT passes for gfx950.
//
// Layout: a table is row-major (row r holds the `m` columns of trace row r,
// `pitch` u64 apart), exactly the reference's host layout
// (crypto/math/src/polynomial.rs:527-597, crypto/math-cuda/src/lde.rs:674).
// Every column is transformed independently; a workgroup tile covers 16
// adjacent words of a run, so each row touch is one 128-byte segment and the
// twiddles of a tile are computed once and shared by its words. In a pass with
// row stride S the S rows of a block are one run of S*m contiguous words, cut
// into windows of 16: a window may span several rows (each has its own twiddle
// factors), but no lane idles on a table whose width is not a multiple of 16
// and every segment starts on a cache line. Against windows within one row:
// commitments of 2^19 x 83 2.33 -> 2.09 ms and of 14 ragged tables 21.68 ->
// 20.15 ms, a proof of eight VM tables of 4 to 26 columns 76.0 -> 72.5 ms.
//
// A size-2^L DIF transform is split into passes. A pass with sub-transform
// size R = R1*R2 and row stride S works on blocks of M = R*S rows:
//   Y[k1] = sum_t x[blk*M + t*S + j] * w_R^(t*k1)          (size-R DFT over t)
//   out[blk*M + bitrev_R(k1)*S + j] = Y[k1] * w_M^(j*k1)   (post twiddle)
// after which every M/R... block of S contiguous rows is an independent
// size-S DFT (the four-step identity). Chaining passes down to S = 1 leaves
// the full DFT in bit-reversed row order. Inside a pass the first log2(R1)
// radix-2 stages run in registers on elements spaced R2 apart, the tile is
// exchanged through LDS, and the last log2(R2) stages run in registers on
// R2 contiguous elements.
//
// Inside a pass the size-R DFT uses the four-step form: round 1 is a size-R1
// DFT over t = t0 + R2*i followed by the inner twiddle w_R^(t0*k_a), round 2
// a size-R2 DFT over t0. Both small DFTs (R1, R2 <= 16) are radix-2 DIF
// whose twiddles are roots of unity of order <= 16, all of the form +-2^s
// in this field (forward w_16 = 2^156, inverse w_16 = 2^36), so they are
// shifts and a reduction, chosen at compile time; a negative sign swaps the
// butterfly's subtraction. Values are kept canonical from the load on, which
// makes each add and sub one conditional correction (field.hpp cadd/csub).
//
// Optional input remaps make the same kernel serve the coset LDE:
//  - input rows may be read at bitrev(logical row) (the coefficient buffer
//    produced by the inverse transform is in bit-reversed order);
//  - element j may be pre-multiplied by weights[j] * w_N^(coset*j)
//    (LDE weights n^-1*g^j, crypto/stark/src/prover.rs:451-467, times the
//    coset shift that turns one size-N transform into B size-n ones);
//  - output rows may be offset per coset by bitrev_B(coset)*n.
#include "ntt_pass.hpp"
#include "prof.hpp"

namespace lvm {

// one-dimensional grid, the windows of a run adjacent, XCD-contiguous
// (neighbouring windows share cache lines where rows are not a multiple of 16
// words)
template <int LOG_R1, int LOG_R2, bool COSET, int NJ>
__global__ __launch_bounds__(PASS_T) void ntt_pass_kernel(PassArgs a) {
    ntt_pass_body<LOG_R1, LOG_R2, COSET, NJ>(a, xcd_contiguous(blockIdx.x, gridDim.x));
}

// threads per column of a pass of 2^r points: min(R1, R2) of with_radix's split
static uint32_t pass_tiles_per_block(int r) { return PASS_T / (PASS_C << (r / 2)); }

// floor(2^32 / d), the multiplier of udiv
static uint32_t udiv_inv(uint32_t d) { return d == 1 ? ~0u : (uint32_t)((1ull << 32) / d); }

// Fills the tiling fields of a pass of 2^r points (every other field set) and
// returns its blocks. cosets: those a coset pass produces; all from one block,
// which reads its tile once, unless the table is so small that its blocks
// leave most of the chip idle (2^10 x 8 commitment: 141 -> 111 us).
uint32_t pass_tiling(int r, uint32_t cosets, PassArgs &a) {
    const uint64_t S = 1ull << a.log_s, words = S * a.m;
    a.units = a.log_s == 0 && a.m <= PASS_C / 2 ? PASS_C / a.m : 1;
    a.run = (uint32_t)words * a.units;  // words < 2^31 (plan_passes)
    a.wins = (uint32_t)(((uint64_t)a.run + PASS_C - 1) / PASS_C);
    a.win_inv = udiv_inv(a.wins);
    a.m_inv = udiv_inv(a.m);
    const uint64_t runs = ((a.total_groups >> a.log_s) + a.units - 1) / a.units;
    a.tiles = (uint32_t)(runs * a.wins);
    const uint32_t per = pass_tiles_per_block(r);
    a.blocks = (a.tiles + per - 1) / per;
    // rows a window spans: its first word lies at most m - gcd(16, m) into a row
    uint32_t g = PASS_C;
    while (a.m % g) g /= 2;
    a.rows = a.log_s ? 1 + (a.m - g + PASS_C - 1) / a.m : 1;
    if (a.rows > S) a.rows = (uint32_t)S;
    const uint32_t copies = a.blocks < COSET_SPLIT_BLOCKS ? cosets : 1;
    a.cosets_per_block = cosets / copies;
    return a.blocks * copies;
}

static void launch_pass(int r, const PassArgs &a0, uint32_t cosets, hipStream_t st, const char *name) {
    ProfScope ps(name, st);
    PassArgs a = a0;
    const uint32_t blocks = pass_tiling(r, cosets, a);
    with_radix(r, [&](auto A, auto B) {
        with_rows(a.rows, [&](auto NJ) {
            if (a.weights)
                hipLaunchKernelGGL((ntt_pass_kernel<A(), B(), true, NJ()>), dim3(blocks), dim3(PASS_T), 0, st, a);
            else
                hipLaunchKernelGGL((ntt_pass_kernel<A(), B(), false, NJ()>), dim3(blocks), dim3(PASS_T), 0, st, a);
        });
    });
}

// Pass plans per log2 size: default splits log n into passes of at most 8
// bits, largest first; set_ntt_plan installs a measured split.
static int g_plan[33][8];
static int g_plan_len[33];

// A pass indexes a run, the S*m words of a block's rows, with 31 bits; the first
// pass has the longest. An installed split whose first radix is too small for
// that (tables of tens of GB) gives way to the default, whose runs are n*m/256 words,
// below 2^31 for every table that fits the device's memory.
int plan_passes(unsigned log_n, uint32_t m, int *r) {
    if (log_n <= 32 && g_plan_len[log_n] > 0 && ((uint64_t)m << (log_n - g_plan[log_n][0])) < (1ull << 31)) {
        for (int i = 0; i < g_plan_len[log_n]; i++) r[i] = g_plan[log_n][i];
        return g_plan_len[log_n];
    }
    int np = 0;
    unsigned left = log_n;
    while (left > 0) {
        unsigned take = left > 8 ? 8 : left;
        r[np++] = (int)take;
        left -= take;
    }
    return np;
}

bool set_ntt_plan(unsigned log_n, const int *r, int np) {
    if (log_n > 32 || np < 0 || np > 8) return false;
    int sum = 0;
    for (int i = 0; i < np; i++) {
        if (r[i] < 1 || r[i] > 8) return false;
        sum += r[i];
    }
    if (np > 0 && sum != (int)log_n) return false;
    for (int i = 0; i < np; i++) g_plan[log_n][i] = r[i];
    g_plan_len[log_n] = np;  // 0 restores the default split
    return true;
}

// The pass sequence of one table's coset LDE (inverse transform of the
// trace, then the coset expansion), as the argument blocks the single-table
// path launches: radix in r_out, arguments (tiling included) in a_out, blocks in blocks_out.
int lde_pass_list(const uint64_t *trace, uint32_t m, unsigned log_n, unsigned log_blowup, const uint64_t *weights,
                  uint64_t *coef, uint64_t *lde, const Tables &tb, int *r_out, PassArgs *a_out, uint32_t *blocks_out) {
    int r[8];
    const int np = plan_passes(log_n, m, r);
    if (np == 0) return -1;
    int k = 0;
    unsigned done = 0;
    for (int p = 0; p < np; p++) {
        PassArgs a{};
        a.in = p == 0 ? trace : coef;
        a.out = coef;
        a.in_pitch = a.out_pitch = m;
        a.m = m;
        a.log_msub = log_n - done;
        a.log_s = log_n - done - r[p];
        a.total_groups = (1ull << log_n) >> r[p];
        a.tw_lo = tb.inv_lo;
        a.tw_hi = tb.inv_hi;
        a.tw_r = tb.inv_r;
        a.inverse = 1;
        a.in_canonical = p > 0;
        r_out[k] = r[p];
        blocks_out[k] = pass_tiling(r[p], 1, a);
        a_out[k++] = a;
        done += r[p];
    }
    const uint32_t B = 1u << log_blowup;
    done = 0;
    for (int p = 0; p < np; p++) {
        PassArgs a{};
        a.in = p == 0 ? coef : lde;
        a.out = lde;
        a.in_pitch = a.out_pitch = m;
        a.m = m;
        a.log_msub = log_n - done;
        a.log_s = log_n - done - r[p];
        a.tw_lo = tb.fwd_lo;
        a.tw_hi = tb.fwd_hi;
        a.tw_r = tb.fwd_r;
        a.in_canonical = 1;
        if (p == 0) {
            a.in_bitrev_bits = log_n;
            a.total_groups = (1ull << log_n) >> r[0];
            a.out_coset_rows = 1ull << log_n;
            a.coset_bits = log_blowup;
            a.shift_log = log_n + log_blowup;
            a.weights = weights;
            a.shift_lo = tb.fwd_lo;
            a.shift_hi = tb.fwd_hi;
        } else {
            a.total_groups = ((uint64_t)B << log_n) >> r[p];
        }
        r_out[k] = r[p];
        blocks_out[k] = pass_tiling(r[p], p == 0 ? B : 1, a);
        a_out[k++] = a;
        done += r[p];
    }
    return k;
}

// In-place DIF passes over `rows` rows of `buf` (independent size-2^log_n
// problems stacked), starting at pass index `first`.
static const char *PASS_NAMES[2][4] = {{"ntt_fwd_pass0", "ntt_fwd_pass1", "ntt_fwd_pass2", "ntt_fwd_pass3"},
                                       {"ntt_inv_pass0", "ntt_inv_pass1", "ntt_inv_pass2", "ntt_inv_pass3"}};

static void run_passes(uint64_t *buf, uint32_t pitch, uint32_t m, size_t rows, unsigned log_n, int first,
                       const int *r, int np, const Tables &tb, bool inverse, hipStream_t st) {
    unsigned done = 0;
    for (int p = 0; p < first; p++) done += r[p];
    for (int p = first; p < np; p++) {
        PassArgs a{};
        a.in = buf;
        a.out = buf;
        a.in_pitch = a.out_pitch = pitch;
        a.m = m;
        a.log_msub = log_n - done;
        a.log_s = log_n - done - r[p];
        a.total_groups = rows >> r[p];
        a.tw_lo = inverse ? tb.inv_lo : tb.fwd_lo;
        a.tw_hi = inverse ? tb.inv_hi : tb.fwd_hi;
        a.tw_r = inverse ? tb.inv_r : tb.fwd_r;
        a.inverse = inverse ? 1u : 0u;
        a.in_canonical = 1;
        launch_pass(r[p], a, 1, st, PASS_NAMES[inverse][p < 3 ? p : 3]);
        done += r[p];
    }
}

// Unnormalised inverse DFT of each column of a natural-order row-major
// table; output rows are in bit-reversed order.
void ntt_inverse_rows(const uint64_t *in, uint32_t in_pitch, uint64_t *out, uint32_t out_pitch, uint32_t m,
                      unsigned log_n, const Tables &tb, hipStream_t st) {
    int r[8];
    int np = plan_passes(log_n, m, r);
    if (np == 0) {
        (void)hipMemcpy2DAsync(out, out_pitch * 8, in, in_pitch * 8, m * 8, 1, hipMemcpyDeviceToDevice, st);
        return;
    }
    PassArgs a{};
    a.in = in;
    a.out = out;
    a.in_pitch = in_pitch;
    a.out_pitch = out_pitch;
    a.m = m;
    a.log_msub = log_n;
    a.log_s = log_n - r[0];
    a.total_groups = (1ull << log_n) >> r[0];
    a.tw_lo = tb.inv_lo;
    a.tw_hi = tb.inv_hi;
    a.tw_r = tb.inv_r;
    a.inverse = 1;
    launch_pass(r[0], a, 1, st, PASS_NAMES[1][0]);
    run_passes(out, out_pitch, m, 1ull << log_n, log_n, 1, r, np, tb, true, st);
}

// Forward DFT of each column (natural in, bit-reversed out).
void ntt_forward_rows(const uint64_t *in, uint32_t in_pitch, uint64_t *out, uint32_t out_pitch, uint32_t m,
                      unsigned log_n, const Tables &tb, hipStream_t st) {
    int r[8];
    int np = plan_passes(log_n, m, r);
    if (np == 0) {
        (void)hipMemcpy2DAsync(out, out_pitch * 8, in, in_pitch * 8, m * 8, 1, hipMemcpyDeviceToDevice, st);
        return;
    }
    PassArgs a{};
    a.in = in;
    a.out = out;
    a.in_pitch = in_pitch;
    a.out_pitch = out_pitch;
    a.m = m;
    a.log_msub = log_n;
    a.log_s = log_n - r[0];
    a.total_groups = (1ull << log_n) >> r[0];
    a.tw_lo = tb.fwd_lo;
    a.tw_hi = tb.fwd_hi;
    a.tw_r = tb.fwd_r;
    launch_pass(r[0], a, 1, st, PASS_NAMES[0][0]);
    run_passes(out, out_pitch, m, 1ull << log_n, log_n, 1, r, np, tb, false, st);
}

// Coset LDE expansion: coefficient table `coef` (n rows, bit-reversed order,
// unnormalised iDFT of the trace) -> `lde` (n*B rows, bit-reversed order over
// log2(n*B) bits) of the evaluations on offset*<w_N> (offset folded into weights).
// log_n >= 1 (every entry point rejects tables of fewer than two rows); returns
// LVM_ERR_ARG without writing `lde` for a size that has no pass plan.
int ntt_coset_expand(const uint64_t *coef, uint32_t coef_pitch, uint64_t *lde, uint32_t lde_pitch, uint32_t m,
                      unsigned log_n, unsigned log_blowup, const uint64_t *weights, const Tables &tb,
                      hipStream_t st) {
    int r[8];
    int np = plan_passes(log_n, m, r);
    if (np == 0) return LVM_ERR_ARG;
    const uint32_t B = 1u << log_blowup;
    PassArgs a{};
    a.in = coef;
    a.out = lde;
    a.in_pitch = coef_pitch;
    a.out_pitch = lde_pitch;
    a.m = m;
    a.log_msub = log_n;
    a.log_s = log_n - r[0];
    a.in_bitrev_bits = log_n;
    a.total_groups = (1ull << log_n) >> r[0];
    a.out_coset_rows = 1ull << log_n;
    a.coset_bits = log_blowup;
    a.shift_log = log_n + log_blowup;
    a.weights = weights;
    a.in_canonical = 1;
    a.tw_lo = tb.fwd_lo;
    a.tw_hi = tb.fwd_hi;
    a.shift_lo = tb.fwd_lo;
    a.shift_hi = tb.fwd_hi;
    a.tw_r = tb.fwd_r;
    launch_pass(r[0], a, B, st, "ntt_coset_pass0");
    run_passes(lde, lde_pitch, m, (size_t)B << log_n, log_n, 1, r, np, tb, false, st);
    return LVM_OK;
}

}  // namespace lvm

// Proof-of-work nonce search on gfx950 (crypto/stark/src/grinding.rs; the
// reference's GPU search is crypto/math-cuda/src/grinding.rs:29
// `generate_nonce_gpu`).
//
//   inner = Keccak(PREFIX || seed || g)             (grinding.rs:84-93, host)
//   nonce valid iff BE u64 of Keccak(inner || BE(nonce))[0..8] < 2^(64-g)
//                                                   (grinding.rs:66-80)
// The result is the smallest valid nonce, the deterministic answer of the
// reference's sequential search. One thread per candidate; the 40-byte
// message fits one Keccak-f (lanes 0-3 the inner digest, lane 4 the nonce,
// padding in lanes 5 and 16). Batches of candidates are searched in
// increasing order; a wave lowers one word of device memory, `best`, to its
// smallest hit, and a wave whose candidates all lie above `best` leaves at
// once: no smaller hit can be lost, and once one is found the rest of the
// batch costs its dispatch alone.
//
// The expected search is 2^g candidates, VALU-bound (one permutation each,
// 2^24 take 1.7 ms). A batch holds 2^(g+2), so that one batch in fifty misses
// (e^-4), bounded below by one block per CU and above by 2^24. Mean over 24
// seeds, batches of 2^24 searched in full before: g = 16 1.74 -> 0.058 ms,
// g = 20 1.67 -> 0.16 ms, g = 22 1.81 -> 0.54 ms.
//
// lvm_generate_nonce_noalloc runs the same kernels with `best` in a fixed
// device word (`scratch` below), so a search allocates no memory.
#include <cstring>
#include <mutex>
#include <string>

#include "keccak.hpp"
#include "lvm_internal.hpp"
#include "prof.hpp"

namespace lvm {

void host_keccak256(const uint8_t *p, size_t n, uint8_t out[32]);

constexpr int GRIND_BLOCK = 256;

// candidates per launch
uint64_t grind_batch(unsigned g) { return 1ull << (g + 2 < 16 ? 16 : g + 2 > 24 ? 24 : g + 2); }

// the inner digest as four little-endian lanes, passed by value
struct GrindDigest {
    uint64_t w[4];
};

// `best` of the allocation-free search. Host code never names it outside
// HIP_SYMBOL(): kernels get its device address from g_scratch_dev.
static __device__ __align__(256) uint64_t scratch[1];

__global__ void grind_start_kernel(uint64_t *best) { *best = ~0ull; }

__global__ __launch_bounds__(GRIND_BLOCK) void grind_kernel(GrindDigest inner, uint64_t base, uint64_t count,
                                                            uint64_t limit, uint64_t *best) {
    const uint64_t i = (uint64_t)blockIdx.x * GRIND_BLOCK + threadIdx.x;
    const uint64_t nonce = base + i;
    // one load per wave, and one answer for it
    const uint64_t seen = __hip_atomic_load(best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t cur = ((uint64_t)__builtin_amdgcn_readfirstlane((uint32_t)(seen >> 32)) << 32) |
                         (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)seen);
    if (cur < nonce - (threadIdx.x & 63)) return;
    bool hit = false;
    if (i < count) {
        uint32_t l[25], h[25];
#pragma unroll
        for (int k = 0; k < 25; k++) l[k] = h[k] = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint64_t v = inner.w[k];
            l[k] = (uint32_t)v;
            h[k] = (uint32_t)(v >> 32);
        }
        // BE(nonce) as a little-endian lane is bswap64(nonce)
        const uint64_t nb = bswap64(nonce);
        l[4] = (uint32_t)nb;
        h[4] = (uint32_t)(nb >> 32);
        l[5] = 0x01;           // byte 40: first padding byte
        h[16] = 0x80000000u;   // byte 135: last padding byte
        keccak_f1600_32_digest<true>(l, h);
        const uint64_t lane0 = ((uint64_t)h[0] << 32) | l[0];
        hit = bswap64(lane0) < limit;
    }
    // the wave's smallest hit is its lowest lane's
    const uint64_t mask = __ballot(hit);
    if (hit && (mask & ((1ull << (threadIdx.x & 63)) - 1)) == 0)
        __hip_atomic_fetch_min(best, nonce, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

namespace {
constexpr int GRIND_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
uint64_t *g_scratch_dev[GRIND_MAX_DEVICES];  // device address of `scratch` per device, set by grind_scratch_setup

// Keccak(PREFIX || seed || g) as little-endian lanes (grinding.rs:84-93)
GrindDigest inner_digest(const uint8_t seed[32], uint8_t grinding_factor) {
    static const uint8_t PREFIX[8] = {0x01, 0x23, 0x45, 0x67, 0x89, 0xab, 0xcd, 0xed};
    uint8_t msg[41], inner_b[32];
    std::memcpy(msg, PREFIX, 8);
    std::memcpy(msg + 8, seed, 32);
    msg[40] = grinding_factor;
    host_keccak256(msg, 41, inner_b);
    GrindDigest dg;
    std::memcpy(dg.w, inner_b, 32);
    return dg;
}
}  // namespace

// Resolves the device address of `scratch` on the current device (called by
// lvm_init with `device` current; once per device).
int grind_scratch_setup(int device) {
    if (device < 0 || device >= GRIND_MAX_DEVICES) return fail(LVM_ERR_ARG, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_dev[device]) return LVM_OK;
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
        return fail(LVM_ERR_DEVICE, std::string("address of the nonce-search scratch: ") + hipGetErrorString(e));
    g_scratch_dev[device] = (uint64_t *)p;
    return LVM_OK;
}

}  // namespace lvm

extern "C" int lvm_generate_nonce(const uint8_t seed[32], uint8_t grinding_factor, uint64_t max_nonce,
                                  uint64_t *nonce_out) {
    using namespace lvm;
    if (!seed || !nonce_out) return fail(LVM_ERR_ARG, "null argument");
    if (grinding_factor < 1 || grinding_factor > 64) return fail(LVM_ERR_ARG, "grinding factor must be 1..64");
    Device *d = device_state();
    if (!d) return LVM_ERR_DEVICE;
    hipStream_t st = lib_stream();
    const GrindDigest inner = inner_digest(seed, grinding_factor);
    const uint64_t limit = grinding_factor == 64 ? 1 : (1ull << (64 - grinding_factor));
    const uint64_t batch = grind_batch(grinding_factor);
    uint64_t *d_best = nullptr;
    if (lvm_malloc(&d_best, 8) != hipSuccess)
        return fail(LVM_ERR_NOMEM, "device allocation for the nonce search failed");
    StageScope ss(st);
    hipError_t e = hipSuccess;
    uint64_t best = ~0ull;
    hipLaunchKernelGGL(grind_start_kernel, dim3(1), dim3(1), 0, st, d_best);
    for (uint64_t base = 0; e == hipSuccess && base < max_nonce; base += batch) {
        const uint64_t count = max_nonce - base < batch ? max_nonce - base : batch;
        {
            ProfScope ps("grinding", st);
            hipLaunchKernelGGL(grind_kernel, dim3((unsigned)((count + GRIND_BLOCK - 1) / GRIND_BLOCK)),
                               dim3(GRIND_BLOCK), 0, st, inner, base, count, limit, d_best);
        }
        e = hipGetLastError();
        if (e == hipSuccess) e = stage_download(&best, d_best, 8, st);
        if (e == hipSuccess) e = stage_sync(st);
        if (e != hipSuccess || best != ~0ull) break;
        if (base + batch < base) break;  // wrapped
    }
    lvm_free(d_best);
    if (e != hipSuccess) return fail(LVM_ERR_DEVICE, std::string("nonce search failed: ") + hipGetErrorString(e));
    if (best == ~0ull) return fail(LVM_ERR_STATE, "no valid nonce below the search limit");
    *nonce_out = best;
    return LVM_OK;
}

// The same search with no allocation: `best` in the device's `scratch` word;
// one 8-byte copy per batch to the host. Needs
// lvm_init on this device first (it resolves the scratch address). Calls that
// overlap on one device share its scratch and race.
extern "C" int lvm_generate_nonce_noalloc(const uint8_t seed[32], uint8_t grinding_factor, uint64_t max_nonce,
                                          uint64_t *nonce_out) {
    using namespace lvm;
    if (!seed || !nonce_out) return fail(LVM_ERR_ARG, "null argument");
    if (grinding_factor < 1 || grinding_factor > 64) return fail(LVM_ERR_ARG, "grinding factor must be 1..64");
    int id = 0;
    if (hipGetDevice(&id) != hipSuccess) return fail(LVM_ERR_DEVICE, "hipGetDevice failed (no GPU visible?)");
    uint64_t *sc = nullptr;
    if (id >= 0 && id < GRIND_MAX_DEVICES) {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        sc = g_scratch_dev[id];
    }
    if (!sc) return fail(LVM_ERR_STATE, "nonce-search scratch not set up on this device: call lvm_init first");
    Device *d = device_state();  // initialised by lvm_init: no allocation here
    if (!d) return LVM_ERR_DEVICE;
    hipStream_t st = thread_stream_if_any(d);
    const GrindDigest inner = inner_digest(seed, grinding_factor);
    const uint64_t limit = grinding_factor == 64 ? 1 : (1ull << (64 - grinding_factor));
    hipError_t e = hipSuccess;
    uint64_t best = ~0ull;
    const uint64_t batch = grind_batch(grinding_factor);
    hipLaunchKernelGGL(grind_start_kernel, dim3(1), dim3(1), 0, st, sc);
    for (uint64_t base = 0; base < max_nonce; base += batch) {
        const uint64_t count = max_nonce - base < batch ? max_nonce - base : batch;
        hipLaunchKernelGGL(grind_kernel, dim3((unsigned)((count + GRIND_BLOCK - 1) / GRIND_BLOCK)), dim3(GRIND_BLOCK),
                           0, st, inner, base, count, limit, sc);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipMemcpyAsync(&best, sc, 8, hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess || best != ~0ull) break;
        if (base + batch < base) break;  // wrapped
    }
    if (e != hipSuccess) return fail(LVM_ERR_DEVICE, std::string("nonce search failed: ") + hipGetErrorString(e));
    if (best == ~0ull) return fail(LVM_ERR_STATE, "no valid nonce below the search limit");
    *nonce_out = best;
    return LVM_OK;
}

// Block-level Merkle hashing with one permutation per 16 lanes (keccak.hpp
// CoopKeccak): the levels above a block's nodes, kept in LDS between levels.
#pragma once
#include "keccak.hpp"
#include "lvm_internal.hpp"

namespace lvm {

constexpr uint32_t TREE_THREADS = 512;  // TREE_TOP_SPAN states of 16 lanes
static_assert(TREE_THREADS == 16 * TREE_TOP_SPAN, "one state per 16 lanes");

struct TreeTopLds {
    uint32_t pi[TREE_THREADS / 64][COOP_WORDS];
    uint32_t dig[2][TREE_TOP_SPAN][8];
};

// A thread's place in the block and its lane constants.
struct TreeTop {
    CoopKeccak k;
    uint32_t *ws;
    uint32_t g, y, half;
    uint64_t *root;  // nullable: where node 0 goes too
    __device__ __forceinline__ TreeTop(TreeTopLds &s, uint64_t *root_out) : root(root_out) {
        ws = s.pi[threadIdx.x >> 6];
        coop_setup(k, ws);
        g = threadIdx.x >> 4;
        y = threadIdx.x & 7;
        half = (threadIdx.x >> 3) & 1;
    }
    // whether this wave holds any of the first cnt states (uniform per wave)
    __device__ __forceinline__ bool wave_on(uint32_t cnt) const { return (threadIdx.x >> 6) * 4 < cnt; }
    __device__ __forceinline__ void permute(uint32_t a[5]) const { keccak_f1600_coop(a, k, ws); }
    // digest of state g to node `node` and to s.dig[buf][g]
    __device__ __forceinline__ void put(const uint32_t a[5], uint64_t *nodes, uint64_t node, TreeTopLds &s,
                                        uint32_t buf) const {
        if (y != 0) return;
        gmem_u32 *d = (gmem_u32 *)nodes + 8 * node;
#pragma unroll
        for (int x = 0; x < 4; x++) {
            d[2 * x + half] = a[x];
            s.dig[buf][g][2 * x + half] = a[x];
        }
        if (node == 0 && root) {
            gmem_u32 *r = (gmem_u32 *)root;
#pragma unroll
            for (int x = 0; x < 4; x++) r[2 * x + half] = a[x];
        }
    }
};

// The levels above `cnt` nodes [base, base + cnt) of a block (cnt a power of
// two <= TREE_TOP_SPAN; their digests in s.dig[buf]) up to the node above them
// all, every level written to the node array. Every thread of the block calls it.
__device__ __forceinline__ void tree_top_levels(const TreeTop &t, TreeTopLds &s, uint64_t *nodes, uint64_t base,
                                                uint32_t cnt, uint32_t buf) {
    while (cnt > 1) {
        __syncthreads();
        cnt >>= 1;
        base = (base - 1) / 2;  // the parent of node x is (x - 1) / 2; a block's nodes stay contiguous
        if (t.wave_on(cnt)) {
            const bool on = t.g < cnt;
            uint32_t a[5];
            coop_load_pair(a, s.dig[buf][2 * (on ? t.g : 0)], on);
            t.permute(a);
            if (on) t.put(a, nodes, base + t.g, s, buf ^ 1);
        }
        buf ^= 1;
    }
}

}  // namespace lvm

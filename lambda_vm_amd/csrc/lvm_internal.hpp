// Internal declarations shared by the HIP translation units of liblvm_gpu.
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include <stdint.h>
#include <stddef.h>
#include <functional>
#include <string>
#include <vector>

#include "field.hpp"
#include "lvm_gpu.h"

// Resident LDE table + Merkle tree behind the opaque `lvm_lde` handle.
struct lvm_lde {
    int device;
    uint64_t *lde;  // N rows x w words, rows in bit-reversed order
    size_t n, N, w, blowup;
    uint8_t *nodes;  // (2L-1) x 32 bytes, root first
    size_t L;
    uint8_t root[32];
};

namespace lvm {

// Device twiddle tables (built once per device by the library).
//  *_lo[x] = w^x, *_hi[x] = w^(x * 2^16) for w the primitive 2^32-th root of
//  unity of crypto/math/src/field/goldilocks.rs:540 (fwd) or its inverse (inv);
//  *_r[e] = w_256^e (e < 128).
struct Tables {
    uint64_t *fwd_lo, *fwd_hi, *inv_lo, *inv_hi, *fwd_r, *inv_r;
};

// status codes of the C ABI (LVM_OK, LVM_ERR_*) come from lvm_gpu.h

void set_error(const std::string &msg);
int fail(int code, const std::string &msg);

// per-device library state
struct Device {
    int id = -1;
    hipStream_t stream = nullptr;  // the first host thread's library stream
    std::atomic<bool> stream_claimed{false};
    Tables tb{};
};
Device *device_state();  // current device's state, initialised on first use; null on failure
// The calling host thread's library stream on device d: every thread that
// calls the library gets its own (default priority, non-blocking), so tables
// proved from several threads overlap on the GPU. Streams outlive their
// threads (an ending thread's stream is drained and reused by a later one). Work handed from one
// thread to another is complete when the producing call returns (every
// entry point that yields a handle or host data synchronises its stream).
hipStream_t thread_stream(Device *d);
// The calling thread's library stream if it already has one, else the
// device's first stream; creates nothing (for the allocation-free entry point).
hipStream_t thread_stream_if_any(Device *d);
// Resolves the per-device address of the nonce search's fixed scratch array
// (grinding.hip); lvm_init calls it with the device current.
int grind_scratch_setup(int device);

// fault injection for the fallback tests (never set in production)
bool take_injected_fault();

// Device allocations (context.cpp): a cache of freed blocks in size classes
// over the stream-ordered pool. A freed block is reused at once on the stream
// that freed it, and on another stream once the event recorded at its release
// has completed; the driver pool is only touched on a cache miss (its frees
// cost 0.1-0.3 ms of host time each when many blocks are live). When the
// device runs out, the cache is returned to the pool and the allocation retried.
hipStream_t lib_stream();
hipError_t lvm_malloc_bytes(void **p, size_t bytes);
hipError_t lvm_free(void *p);
void lvm_release_cached();
template <class T>
inline hipError_t lvm_malloc(T **p, size_t bytes) {
    return lvm_malloc_bytes((void **)p, bytes);
}

// Small host<->device transfers through a per-thread pinned staging area: a
// copy of pageable memory is staged by the runtime at tens of microseconds
// each, a copy of pinned memory is a plain DMA. stage_upload copies the host
// data into the area at the call and queues the DMA; stage_download queues the
// DMA into the area and the bytes reach dst_host at stage_sync, which
// synchronises the stream. A StageScope around an entry point drops (after a
// stream synchronisation) the downloads it queued but never delivered, so an
// early error return leaves nothing pending. Transfers above 4 MiB go direct.
hipError_t stage_upload(void *dst_dev, const void *src_host, size_t bytes, hipStream_t st);
hipError_t stage_download(void *dst_host, const void *src_dev, size_t bytes, hipStream_t st);
hipError_t stage_sync(hipStream_t st);
// Room in the area for one or two results that kernels queued next on `st`
// write themselves (page-locked memory is mapped): the bytes reach the
// destinations at stage_sync, without a copy's launch. For results of up to
// STAGE_RESULT bytes, written once. No other stage_* call may come between this
// one and the last of those kernels' launches (it could drain the area).
constexpr size_t STAGE_RESULT = 64 << 10;
hipError_t stage_result(void *dst_a, size_t bytes_a, void *dst_b, size_t bytes_b, hipStream_t st, void **a, void **b);
// Transfers of whole tables between pageable host memory and the device, in
// slots of a page-locked ring that the calling thread keeps: the host copies
// one slot while the device moves another. The device side is a kernel that reads
// or writes the slot itself (the memory is mapped): queuing a DMA copy costs the
// host some 25 us a slot against 4 for a launch, and a download's rows are
// reordered on their way out. download() queues every slot
// and delivers all but the last ones; finish() delivers those, so what is
// queued on the stream in between runs beside the host's copies. One ring
// object per call and thread at a time. ready() is false when the ring is not
// wanted or cannot be allocated: the caller then copies directly.
//
// What goes through the ring: pageable memory. Memory that the runtime knows
// (page-locked, managed, a device's own) is copied directly, at the link's rate
// and with no work of the host's. 2^20 x 128 at blowup 2 from and to page-locked
// memory: 1 GiB up and its commitment 53.1 ms through the ring, 27.0 ms
// directly; the 2 GiB LDE down 100 ms against 38.4. Only page-locked results of up
// to RING_LOCKED_OUT come through it, as a copy's launch costs more than they
// (16 KiB 16 us against 26, 512 KiB 35 against 40, 1 MiB 51 against 50, 2 MiB 111
// against 69). Pageable tables of more than RING_MOST_IN go up directly too: the
// runtime pins large pageable memory in place, which beats one thread's copies
// (commitments from 16 MiB 812 us against 780 through the ring, 32 MiB 1573 against
// 1602, 128 MiB 5.4 ms against 6.3, 512 MiB 21.6 against 25.0). On the way down
// the ring stays ahead at every size (1 GiB 56.7 ms against 60.5).
bool ring_takes_upload(const void *src, size_t bytes);
bool ring_takes_download(const void *dst, size_t bytes);
constexpr size_t RING_MOST_IN = 32u << 20;
constexpr size_t RING_LOCKED_OUT = 1u << 20;
constexpr size_t RING_SLOT = 512u << 10, RING_SLOTS = 8;
class HostRing {
  public:
    HostRing(hipStream_t st, bool wanted);
    ~HostRing();
    bool ready() const { return buf_ != nullptr; }
    hipError_t upload(uint64_t *dst_dev, const uint64_t *src_host, size_t words);
    // produce(slot, off, n): queue on the stream the kernel that writes bytes
    // [off, off + n) of the result to `slot`
    using Produce = std::function<void(void *slot, size_t off, size_t n)>;
    hipError_t download(void *dst_host, size_t bytes, const Produce &produce);
    hipError_t finish();

  private:
    hipError_t deliver_oldest();
    hipStream_t st_;
    uint8_t *buf_ = nullptr;
    hipEvent_t ev_[RING_SLOTS] = {};
    uint64_t head_ = 0, tail_ = 0;  // slots queued and slots whose event was waited for
    uint8_t *dst_[RING_SLOTS] = {};  // where a slot's bytes go (nullptr: an upload)
    size_t len_[RING_SLOTS] = {};
};
struct StageScope {
    explicit StageScope(hipStream_t st);
    ~StageScope();
    hipStream_t st;
    size_t mark;
};

#define LVM_HIP(expr)                                                                                   \
    do {                                                                                                \
        hipError_t _e = (expr);                                                                         \
        if (_e != hipSuccess) return ::lvm::fail(LVM_ERR_DEVICE, std::string(#expr) + ": " +    \
                                                   hipGetErrorString(_e));                              \
    } while (0)

// ---- NTT (ntt.hip) ----
// Arguments of one NTT pass over one table (layout and remaps described in ntt.hip).
struct PassArgs {
    const uint64_t *in;
    uint64_t *out;
    uint32_t in_pitch, out_pitch;  // row strides in u64
    uint32_t m;                    // number of columns
    uint32_t log_msub;             // log2 of M (sub-problem rows at this pass)
    uint32_t log_s;                // log2 of the row stride S
    uint32_t in_bitrev_bits;       // 0: natural input rows; else bitrev over this many bits
    uint64_t total_groups;         // rows_logical / R
    uint64_t out_coset_rows;       // rows per coset block in `out` (n); 0 = single block
    uint32_t coset_bits;           // log2(blowup) for the per-coset output offset
    uint32_t shift_log;            // log2 N of the coset shift w_N^(coset*j); 0 = none
    const uint64_t *weights;       // nullable pre-multiply weights[logical row]
    const uint64_t *tw_lo;         // w_{2^32}^(+-x), x < 2^16
    const uint64_t *tw_hi;         // w_{2^32}^(+-x*2^16), x < 2^16
    const uint64_t *shift_lo;      // forward tables for the coset shift
    const uint64_t *shift_hi;
    const uint64_t *tw_r;          // w_256^(+-e), e < 256
    uint32_t cosets_per_block;     // cosets produced per block
    uint32_t inverse;              // 1: inverse transform (tw_* hold inverse powers)
    uint32_t in_canonical;         // 1: input values are below p (an earlier pass wrote them)
    // tiling (pass_tiling): runs of `run` words in `wins` windows of 16
    uint32_t run, wins, tiles;
    uint32_t win_inv, m_inv;       // udiv multipliers of wins and m
    uint32_t blocks;               // blocks that cover the tiles once
    uint32_t rows;                 // rows a window can span
    uint32_t units;                // runs packed into a tile (last pass of a narrow table), else 1
};
// A coset pass of fewer blocks than this has its cosets shared out over copies
// of them (each reads the tile again).
constexpr uint32_t COSET_SPLIT_BLOCKS = 512;

void ntt_inverse_rows(const uint64_t *in, uint32_t in_pitch, uint64_t *out, uint32_t out_pitch, uint32_t m,
                      unsigned log_n, const Tables &tb, hipStream_t st);
void ntt_forward_rows(const uint64_t *in, uint32_t in_pitch, uint64_t *out, uint32_t out_pitch, uint32_t m,
                      unsigned log_n, const Tables &tb, hipStream_t st);
int ntt_coset_expand(const uint64_t *coef, uint32_t coef_pitch, uint64_t *lde, uint32_t lde_pitch, uint32_t m,
                      unsigned log_n, unsigned log_blowup, const uint64_t *weights, const Tables &tb,
                      hipStream_t st);

// ---- Keccak / Merkle (merkle.hip) ----
// Row-pair leaves over words [w0, w1) of each row of a row-major table whose
// rows are already stored in bit-reversed order: leaf i hashes rows 2i, 2i+1,
// into node L-1+i of the tree. Small tables' blocks go on to the levels above
// their leaves; returns the nodes C of the topmost level written, which lie at
// [C-1, 2C-1): what merkle_build_inner goes on from. canonical: every word is
// known to be below p (the NTT's output). root_out (nullable, here and below):
// where the block that hashes the root writes it too.
uint64_t keccak_row_pair_leaves(const uint64_t *rows, uint64_t pitch, uint64_t w0, uint64_t w1, uint64_t L,
                                bool canonical, uint8_t *nodes, uint64_t *root_out, hipStream_t st);
// the levels above the C nodes (a power of two) at [C-1, 2C-1) of a tree
void merkle_build_inner(uint8_t *nodes, uint64_t C, uint64_t *root_out, hipStream_t st);

size_t padded_leaves(size_t n);

// ---- composition (compose.hip) ----
// degree-2 split of N bit-reversed Fp3 composition values into N/2
// natural-order rows [H0 | H1]
void launch_d2_split(const uint64_t *hb, unsigned log_N, uint64_t coset_offset, const Tables &tb, uint64_t *halves,
                     hipStream_t st);
// three or more composition parts: natural rows t of the P part coefficient
// columns (Fp3, scaled for evaluation on the coset) from the bit-reversed
// unnormalised inverse DFT `coef` of the N composition values; P <= 8
void launch_parts_scatter(const uint64_t *coef, unsigned log_N, uint32_t P, const uint64_t *wt,
                          const uint64_t *offset_inv_pows, uint64_t *out, hipStream_t st);

// ---- work lists over several tables (batched stages) ----
// Work-list slot of block b: the t with prefix[t] <= b < prefix[t+1]
// (prefix ascending, prefix[0] = 0), by binary search over `count` slots.
// Workgroups are dispatched to the 8 XCDs round-robin by block index, and
// each XCD has its own L2. This bijection on [0, nb) gives XCD x the
// contiguous logical range [x*q, (x+1)*q) (q = nb / 8; the nb % 8 tail blocks
// keep their index), so neighbouring logical tiles that share cache lines
// (the column groups of one row tile) are served by one L2.
__device__ __forceinline__ uint32_t xcd_contiguous(uint32_t b, uint32_t nb) {
    const uint32_t q = nb >> 3;
    return b < (q << 3) ? (b & 7u) * q + (b >> 3) : b;
}

__device__ __forceinline__ uint32_t find_slot(const uint32_t *__restrict__ prefix, uint32_t count, uint32_t b) {
    uint32_t lo = 0, hi = count - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) / 2;
        if (prefix[mid] <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}
int plan_passes(unsigned log_n, uint32_t m, int *r);  // radices of a size-2^log_n transform of m columns
bool set_ntt_plan(unsigned log_n, const int *r, int np);  // np = 0 restores the default
void launch_pass_batched(int r, bool coset, uint32_t rows, const PassArgs *d_args, const uint32_t *d_prefix,
                         uint32_t count, uint32_t blocks, hipStream_t st);
// One table's coset-LDE pass sequence (inverse passes into `coef`, then the
// coset expansion into `lde`); returns the number of passes.
int lde_pass_list(const uint64_t *trace, uint32_t m, unsigned log_n, unsigned log_blowup, const uint64_t *weights,
                  uint64_t *coef, uint64_t *lde, const Tables &tb, int *r_out, PassArgs *a_out, uint32_t *blocks_out);

struct LeafJob {
    const uint64_t *rows;  // bit-reversed row-major LDE, `pitch` words per row
    uint64_t pitch;
    uint64_t num_leaves;
    uint64_t *nodes;       // the table's tree
    uint32_t span;         // leaves per block of a small table (leaf_top_span), 0: TREE_WIDE_SPAN of them, no levels
    uint32_t root;         // the table's slot in the launch's root array
};
struct TreeStep {
    uint64_t *nodes;
    uint64_t cstart, pstart;  // first child / first parent index of the level
    uint32_t span;            // parents per block at the first level
    uint32_t parents;         // parents of the first level
    uint32_t root;            // the tree's slot in the launch's root array
    uint32_t pad;
};
// Trees of more children than this have their level hashed one node per lane;
// below, the step is a tree top: blocks of TREE_TOP_SPAN parents, all their
// levels, one permutation per 16 lanes (merkle.hip). In a launch over several
// trees the tops' children together stay within TREE_TOP_BATCH (tree_steps).
constexpr uint64_t TREE_TOP_CHILDREN = 1u << 14;
constexpr uint32_t TREE_TOP_SPAN = 32;
constexpr uint64_t TREE_TOP_BATCH = 1u << 15;
constexpr uint32_t TREE_WIDE_SPAN = 512;  // leaves, or parents of a wide level, per block of a batched launch
// Trees of at most this many leaves hash them one permutation per 16 lanes
// too, TREE_TOP_SPAN leaves per block, and the levels above in the same launch,
// when such trees have at most LEAF_TOP_BATCH leaves together (leaf_top_spans).
constexpr uint64_t LEAF_TOP_LEAVES = 1u << 13;
constexpr uint64_t LEAF_TOP_BATCH = 1u << 15;
inline uint32_t leaf_top_span(uint64_t L) { return (uint32_t)(L < TREE_TOP_SPAN ? L : TREE_TOP_SPAN); }
std::vector<uint32_t> leaf_top_spans(const std::vector<uint64_t> &leaves);  // per table of one launch (batch.cpp)
// roots: 32-byte slots, written by the blocks that hash a root
void launch_leaves_batched(const LeafJob *d_jobs, const uint32_t *d_prefix, uint32_t count, uint32_t blocks,
                           uint64_t *roots, hipStream_t st);
void launch_tree_steps_batched(const TreeStep *d_steps, const uint32_t *d_prefix, uint32_t count, uint32_t blocks,
                               uint64_t *roots, hipStream_t st);
// One FRI fold of each of count codewords in shared launches (fri.hip);
// zetas: count x 3; roots_out (count x 32) when committing.
int fri_fold_batch(lvm_fri *const *fs, size_t count, const uint64_t *zetas, bool commit, uint8_t *roots_out);
// What is left of a tree: the levels above its C nodes (a power of two) at [C-1, 2C-1).
struct TreeAt {
    uint8_t *nodes;
    uint64_t C;
    uint32_t root;  // the tree's slot in the launch's root array
};
// The launches that build several trees: for each, its steps (in the trees' order) and their blocks.
std::vector<std::vector<std::pair<TreeStep, uint32_t>>> tree_steps(std::vector<TreeAt> trees);

// Constraint programs (compose.hip interpreter, compose_jit.cpp compiled form).
struct CompArgs;
// Node computing each constraint (given, or the last writer of a pinned root slot).
bool root_nodes_of(const lvm_program *pg, std::vector<uint32_t> &root_node);
bool jit_enabled();
// Boundary constraints of a composition grouped by step, steps in
// first-seen order (the order of CompArgs::b_col).
struct BoundarySteps {
    uint32_t num_steps = 0;
    std::vector<uint32_t> step_off;  // num_steps + 1
    std::vector<uint32_t> col, is_aux;
    std::vector<uint64_t> step_row;  // trace row of each step
};
// false when there are more than COMP_MAX_STEPS distinct steps (mod trace_rows)
bool boundary_steps_of(const uint32_t *b_col, const uint32_t *b_is_aux, const uint64_t *b_step, size_t num_boundary,
                       uint64_t trace_rows, BoundarySteps &bs, std::vector<uint32_t> *order);
// Compiles the program's kernel (or finds it compiled); false when the
// generator does not take the program or the compile fails.
bool jit_prepare(const lvm_program *pg, const std::vector<uint32_t> &root_node, const uint32_t *root_group, int mode);
// Launches the compiled kernel on the current device; false on failure.
bool jit_launch(const lvm_program *pg, const std::vector<uint32_t> &root_node, const uint32_t *root_group, int mode,
                CompArgs &args, uint64_t blocks, hipStream_t st);
// The composition (mode 0) of several tables' programs as one kernel: compile
// (cached per program set), then launch with table t's arguments at d_args[t]
// and its blocks [d_prefix[t], d_prefix[t+1]) (128 natural rows each).
bool jit_prepare_batch(const std::vector<const lvm_program *> &pgs, const std::vector<std::vector<uint32_t>> &root_nodes,
                       const std::vector<const uint32_t *> &root_groups);
bool jit_launch_batch(const std::vector<const lvm_program *> &pgs, const std::vector<std::vector<uint32_t>> &root_nodes,
                      const std::vector<const uint32_t *> &root_groups, const CompArgs *d_args,
                      const uint32_t *d_prefix, uint32_t count, uint64_t blocks, hipStream_t st);
}  // namespace lvm

// FRI commit phase on gfx950: every layer stays in HBM (codeword + Merkle
// tree) and only the 32-byte root crosses to the host per layer, where the
// transcript turns it into the next challenge.
//
// Fold (crypto/stark/src/fri/fri_functions.rs:15-29), codeword in bit-reversed
// order, pairs (2j, 2j+1) conjugate:
//     out[j] = (lo + hi) + inv_tw[j] * (zeta * (lo - hi))
// with inv_tw[j] = 1 / (g_l * w_{N_l}^bitrev(j)) on layer l (offset g_l =
// g^(2^l), length N_l): the reference builds these by batch inversion and
// squares them per layer (fri_functions.rs:37-61); here each thread forms its
// twiddle as g_l^-1 * w_{N_l}^-bitrev(j) from the two-level root table.
// One thread produces folded elements 2j and 2j+1 and hashes them into leaf
// j = Keccak(BE24(e[2j]) || BE24(e[2j+1])) (field_element_vector.rs:129-134)
// in the same pass, so a committed layer is one read of its parent codeword.
#include <cstring>
#include <vector>

#include "lvm_internal.hpp"
#include "prof.hpp"
#include "tree_top.hpp"

namespace lvm {

__device__ __forceinline__ fp3 ld3(const uint64_t *p) { return fp3{p[0], p[1], p[2]}; }
__device__ __forceinline__ void st3(uint64_t *p, fp3 v) {
    p[0] = v.c0;
    p[1] = v.c1;
    p[2] = v.c2;
}

// One fold of a codeword of 2*half Fp3 values into `out` (half values);
// `nodes` (nullable) is the layer's tree, whose half/2 leaves are hashed in the
// same pass; span > 0: a small layer, span leaves per block and the levels above.
struct FoldJob {
    const uint64_t *in;
    uint64_t *out;
    uint64_t *nodes;
    uint64_t half;
    uint64_t z0, z1, z2;
    uint64_t ginv;  // inverse of the codeword's coset offset
    uint32_t log_half;
    uint32_t span;
    uint32_t root;  // the layer tree's slot in the launch's root array
    uint32_t pad;
};

__device__ __forceinline__ fp3 fold_one(const uint64_t *in, uint64_t j, fp3 zeta, uint64_t ginv, uint32_t log_half,
                                        const uint64_t *ilo, const uint64_t *ihi) {
    fp3 lo = ld3(in + 6 * j), hi = ld3(in + 6 * j + 3);
    fp3 sum = f3_add(lo, hi);
    fp3 diff = f3_sub(lo, hi);
    // w_{N_l}^-bitrev(j) = w_{2^32}^-(bitrev(j) << (32 - log N_l)), log N_l = log_half + 1
    uint32_t e = log_half ? (bitrev((uint32_t)j, log_half) << (31 - log_half)) : 0u;
    uint64_t tw = mul(ginv, mul(ilo[e & 0xFFFFu], ihi[e >> 16]));
    return f3_add(sum, f3_mul_base(f3_mul(zeta, diff), tw));
}

// Thread t of one fold: out has half elements; the leaves (with nodes) are
// half/2 digests, padded_leaves(half/2) = half/2.
__device__ __forceinline__ void fri_fold_body(const FoldJob &j, uint64_t t, const uint64_t *ilo,
                                              const uint64_t *ihi) {
    const uint64_t *__restrict__ in = j.in;
    uint64_t *__restrict__ out = j.out;
    const uint64_t half = j.half, ginv = j.ginv;
    uint64_t *__restrict__ leaves = j.nodes ? j.nodes + 4 * (half / 2 - 1) : nullptr;
    const uint32_t log_half = j.log_half;
    const fp3 zeta{j.z0, j.z1, j.z2};
    if (leaves) {
        // thread t: folded elements 2t, 2t+1 and leaf t
        if (2 * t >= half) return;
        fp3 a = fold_one(in, 2 * t, zeta, ginv, log_half, ilo, ihi);
        fp3 b = fold_one(in, 2 * t + 1, zeta, ginv, log_half, ilo, ihi);
        st3(out + 6 * t, a);
        st3(out + 6 * t + 3, b);
        uint32_t l[25], h[25];
#pragma unroll
        for (int k = 0; k < 25; k++) l[k] = h[k] = 0;
        const uint64_t v[6] = {a.c0, a.c1, a.c2, b.c0, b.c1, b.c2};
#pragma unroll
        for (int k = 0; k < 6; k++) {
            uint64_t c = canon(v[k]);
            l[k] = __builtin_bswap32((uint32_t)(c >> 32));
            h[k] = __builtin_bswap32((uint32_t)c);
        }
        l[6] = 0x01;
        h[16] = 0x80000000u;
        keccak_f1600_32_digest<true>(l, h);
        uint64_t *o = leaves + 4 * t;
#pragma unroll
        for (int k = 0; k < 4; k++) o[k] = ((uint64_t)h[k] << 32) | l[k];
    } else {
        if (t >= half) return;
        st3(out + 3 * t, fold_one(in, t, zeta, ginv, log_half, ilo, ihi));
    }
}

// Block b of a small layer: its span leaves' 2*span folded elements, one per
// thread, then leaves and the tree levels above them, one permutation per 16
// lanes. A layer of up to LEAF_TOP_LEAVES leaves has too few to fill the chip
// with one leaf per lane; what its tree costs is the chain of permutations.
__device__ __forceinline__ void fri_fold_top(const FoldJob &j, uint64_t b, const uint64_t *ilo, const uint64_t *ihi,
                                             uint64_t *roots) {
    __shared__ TreeTopLds s;
    __shared__ uint64_t s_val[TREE_TOP_SPAN][6];  // a leaf's two elements, canonical
    const TreeTop t(s, roots + 4 * j.root);
    const uint64_t first = (uint64_t)j.span * b, L = j.half / 2;
    if (threadIdx.x < 2 * j.span) {
        const uint64_t e = 2 * first + threadIdx.x;
        const fp3 v = fold_one(j.in, e, fp3{j.z0, j.z1, j.z2}, j.ginv, j.log_half, ilo, ihi);
        st3(j.out + 3 * e, v);
        uint64_t *o = &s_val[threadIdx.x >> 1][3 * (threadIdx.x & 1)];
        o[0] = canon(v.c0);
        o[1] = canon(v.c1);
        o[2] = canon(v.c2);
    }
    __syncthreads();
    if (t.wave_on(j.span)) {
        const bool on = t.g < j.span;
        uint32_t a[5];
#pragma unroll
        for (int x = 0; x < 5; x++) {
            const uint32_t i = 5 * t.y + x;
            a[x] = 0;
            if (on && i < 6) {
                const uint64_t c = s_val[t.g][i];
                a[x] = __builtin_bswap32(t.half ? (uint32_t)c : (uint32_t)(c >> 32));
            }
            if (i == 6 && t.half == 0) a[x] = 0x01;
            if (i == 16 && t.half == 1) a[x] = 0x80000000u;
        }
        t.permute(a);
        if (on) t.put(a, j.nodes, L - 1 + first + t.g, s, 0);
    }
    tree_top_levels(t, s, j.nodes, L - 1 + first, j.span, 0);
}

// blocks of one fold: threads per block and how many
constexpr uint32_t FOLD_THREADS = TREE_THREADS;
inline uint64_t fold_blocks(const FoldJob &j) {
    if (j.span) return j.half / 2 / j.span;
    return ((j.nodes ? j.half / 2 : j.half) + FOLD_THREADS - 1) / FOLD_THREADS;
}

__device__ __forceinline__ void fri_fold_block(const FoldJob &j, uint64_t b, const uint64_t *ilo,
                                               const uint64_t *ihi, uint64_t *roots) {
    if (j.span)
        fri_fold_top(j, b, ilo, ihi, roots);
    else
        fri_fold_body(j, b * FOLD_THREADS + threadIdx.x, ilo, ihi);
}

__global__ __launch_bounds__(FOLD_THREADS) void fri_fold_kernel(FoldJob j, const uint64_t *ilo, const uint64_t *ihi,
                                                                uint64_t *roots) {
    fri_fold_block(j, blockIdx.x, ilo, ihi, roots);
}

// The same fold for several codewords in one launch: blocks [prefix[t],
// prefix[t+1]) run jobs[t].
__global__ __launch_bounds__(FOLD_THREADS) void fri_fold_batched_kernel(const FoldJob *__restrict__ jobs,
                                                                        const uint32_t *__restrict__ prefix,
                                                                        uint32_t count, const uint64_t *ilo,
                                                                        const uint64_t *ihi, uint64_t *roots) {
    const uint32_t b = blockIdx.x;
    const uint32_t t = find_slot(prefix, count, b);
    const FoldJob j = jobs[t];
    fri_fold_block(j, b - prefix[t], ilo, ihi, roots);
}

// Symmetric evaluations and authentication paths of every layer for every
// query (crypto/stark/src/fri/mod.rs:153-205): index_l = iota >> l, eval_sym =
// e_l[index_l ^ 1], path of leaf index_l >> 1. Block (query, layer), all words
// read at once (level k's L >> k nodes start at (L >> k) - 1); 13 launches of 30
// threads walking a path each took 12 us apiece.
struct QueryLayer {
    const uint64_t *evals, *nodes;
    uint64_t L;
    uint64_t paths_off;  // words before the layer's paths
    uint32_t depth;
    uint32_t pad;
};
__global__ __launch_bounds__(128) void fri_query_kernel(const QueryLayer *__restrict__ layers,
                                                        const uint64_t *__restrict__ iotas, uint64_t first,
                                                        uint64_t count, uint64_t *sym_out, uint64_t *paths_out) {
    const uint64_t q = first + blockIdx.x;
    const uint32_t li = blockIdx.y;
    const QueryLayer l = layers[li];
    const uint64_t idx = iotas[q] >> li, p = idx >> 1;
    if (threadIdx.x < 3) sym_out[(li * count + q) * 3 + threadIdx.x] = l.evals[3 * (idx ^ 1) + threadIdx.x];
    for (uint32_t i = threadIdx.x; i < 4 * l.depth; i += 128) {
        const uint32_t k = i / 4;
        paths_out[l.paths_off + q * l.depth * 4 + i] = l.nodes[4 * ((l.L >> k) - 1 + ((p >> k) ^ 1)) + i % 4];
    }
}

}  // namespace lvm

using namespace lvm;

struct FriLayer {
    uint64_t *evals = nullptr;  // len Fp3
    uint64_t len = 0;
    uint8_t *nodes = nullptr;   // (2L-1) x 32
    uint64_t L = 0;
    uint8_t root[32];
};

struct lvm_fri {
    int device;
    uint64_t *cur = nullptr;  // current codeword (owned unless it is a committed layer's buffer)
    bool cur_owned = true;
    uint64_t len = 0;
    uint64_t offset = 0;  // coset offset of the current codeword
    std::vector<FriLayer> layers;
};

namespace {
bool is_pow2(uint64_t x) { return x && !(x & (x - 1)); }
unsigned log2u(uint64_t x) { return (unsigned)__builtin_ctzll(x); }

void free_fri(lvm_fri *f) {
    if (f->cur && f->cur_owned) lvm_free(f->cur);
    for (auto &l : f->layers) {
        lvm_free(l.evals);
        lvm_free(l.nodes);
    }
    delete f;
}
}  // namespace

extern "C" {

int lvm_fri_new(const uint64_t *evals, size_t len, uint64_t coset_offset, int evals_on_device, lvm_fri **out) {
    if (!evals || !out || !is_pow2(len) || len < 2) return fail(LVM_ERR_ARG, "FRI codeword length must be a power of two >= 2");
    if (log2u(len) > 32) return fail(LVM_ERR_ARG, "FRI codeword exceeds 2^32");
    if (canon(coset_offset) == 0) return fail(LVM_ERR_ARG, "coset offset must be non-zero");
    Device *d = device_state();
    if (!d) return LVM_ERR_DEVICE;
    if (take_injected_fault()) return fail(LVM_ERR_INJECTED, "injected fault");
    lvm_fri *f = new lvm_fri();
    f->device = d->id;
    f->len = len;
    f->offset = coset_offset;
    if (evals_on_device == 2) {
        // adopt a library allocation (lvm_dev_alloc) without copying it
        f->cur = (uint64_t *)evals;
        *out = f;
        return LVM_OK;
    }
    if (lvm_malloc(&f->cur, len * 24) != hipSuccess) {
        delete f;
        return fail(LVM_ERR_NOMEM, "FRI codeword allocation failed");
    }
    hipError_t e = hipMemcpyAsync(f->cur, evals, len * 24, evals_on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice,
                                  thread_stream(d));
    if (e == hipSuccess) e = hipStreamSynchronize(thread_stream(d));
    if (e != hipSuccess) {
        free_fri(f);
        return fail(LVM_ERR_DEVICE, std::string("FRI upload: ") + hipGetErrorString(e));
    }
    *out = f;
    return LVM_OK;
}

static int fri_fold_impl(lvm_fri *f, const uint64_t zeta[3], bool commit, uint8_t root_out[32]) {
    if (!f || !zeta) return fail(LVM_ERR_ARG, "null argument");
    if (f->len < 2) return fail(LVM_ERR_STATE, "codeword already folded to one element");
    if (commit && f->len < 4) return fail(LVM_ERR_STATE, "a committed layer needs at least two folded elements");
    Device *d = device_state();
    if (!d) return LVM_ERR_DEVICE;
    if (take_injected_fault()) return fail(LVM_ERR_INJECTED, "injected fault");
    hipStream_t st = thread_stream(d);
    const uint64_t half = f->len / 2;
    uint64_t *out = nullptr;
    LVM_HIP(lvm_malloc(&out, half * 24));
    FriLayer layer;
    if (commit) {
        layer.L = padded_leaves(half / 2);
        if (lvm_malloc(&layer.nodes, (2 * layer.L - 1) * 32) != hipSuccess) {
            lvm_free(out);
            return fail(LVM_ERR_NOMEM, "FRI tree allocation failed");
        }
    }
    const uint64_t ginv = inv(f->offset);
    const uint32_t log_half = log2u(half);
    const uint32_t span = commit ? leaf_top_spans({layer.L})[0] : 0;
    StageScope ss(st);
    void *root = nullptr;
    hipError_t e = commit ? stage_result(layer.root, 32, nullptr, 0, st, &root, nullptr) : hipSuccess;
    if (e == hipSuccess) {
        ProfScope ps(commit ? "fri_fold_leaves" : "fri_fold", st);
        const FoldJob j{f->cur, out, (uint64_t *)layer.nodes, half, zeta[0], zeta[1], zeta[2], ginv, log_half, span,
                        0, 0};
        hipLaunchKernelGGL(fri_fold_kernel, dim3((unsigned)fold_blocks(j)), dim3(FOLD_THREADS), 0, st, j,
                           d->tb.inv_lo, d->tb.inv_hi, (uint64_t *)root);
    }
    if (e == hipSuccess && commit) {
        ProfScope ps("fri_merkle", st);
        merkle_build_inner(layer.nodes, span ? layer.L / span : layer.L, (uint64_t *)root, st);
    }
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = stage_sync(st);
    if (e != hipSuccess) {
        lvm_free(out);
        if (layer.nodes) lvm_free(layer.nodes);
        return fail(LVM_ERR_DEVICE, std::string("FRI fold: ") + hipGetErrorString(e));
    }
    if (f->cur_owned) lvm_free(f->cur);
    f->cur = out;
    f->len = half;
    f->offset = sqr(f->offset);
    if (commit) {
        layer.evals = out;
        layer.len = half;
        f->cur_owned = false;
        f->layers.push_back(layer);
        if (root_out) std::memcpy(root_out, layer.root, 32);
    } else {
        f->cur_owned = true;
    }
    return LVM_OK;
}

}  // extern "C"

namespace lvm {

// One fold of every codeword fs[0..count) (zeta t at zetas[3t]) on the
// calling thread's stream: one work-list launch for the folds (and their
// leaves), one launch per tree step over all layer trees, roots written to
// mapped host memory. Each state then holds what fri_fold_impl would leave. On a device
// error no state changes.
int fri_fold_batch(lvm_fri *const *fs, size_t count, const uint64_t *zetas, bool commit, uint8_t *roots_out) {
    if (!fs || !zetas || (commit && !roots_out)) return fail(LVM_ERR_ARG, "null argument");
    if (count == 0) return LVM_OK;
    Device *d = device_state();
    if (!d) return LVM_ERR_DEVICE;
    for (size_t t = 0; t < count; t++) {
        if (!fs[t]) return fail(LVM_ERR_ARG, "null FRI state");
        if (fs[t]->device != d->id) return fail(LVM_ERR_ARG, "FRI states of another device");
        if (fs[t]->len < (commit ? 4u : 2u)) return fail(LVM_ERR_STATE, "codeword too short for this fold");
    }
    if (take_injected_fault()) return fail(LVM_ERR_INJECTED, "injected fault");
    hipStream_t st = thread_stream(d);
    std::vector<uint64_t *> outs(count, nullptr);
    std::vector<FriLayer> layers(count);
    uint8_t *arena = nullptr;
    auto release = [&]() {
        for (size_t t = 0; t < count; t++) {
            lvm_free(outs[t]);
            lvm_free(layers[t].nodes);
        }
        lvm_free(arena);
    };
    // descriptors: fold jobs + block prefix, then per tree step the steps + prefix
    std::vector<FoldJob> jobs(count);
    std::vector<uint32_t> prefix(1, 0);
    uint64_t total = 0;
    std::vector<uint64_t> leaves(count, 0);
    for (size_t t = 0; commit && t < count; t++) leaves[t] = padded_leaves(fs[t]->len / 4);
    const std::vector<uint32_t> spans = leaf_top_spans(leaves);
    std::vector<TreeAt> trees;
    for (size_t t = 0; t < count; t++) {
        lvm_fri *f = fs[t];
        const uint64_t half = f->len / 2;
        if (lvm_malloc(&outs[t], half * 24) != hipSuccess) {
            release();
            return fail(LVM_ERR_NOMEM, "FRI layer allocation failed");
        }
        if (commit) {
            layers[t].L = leaves[t];
            if (lvm_malloc(&layers[t].nodes, (2 * layers[t].L - 1) * 32) != hipSuccess) {
                release();
                return fail(LVM_ERR_NOMEM, "FRI tree allocation failed");
            }
            trees.push_back({layers[t].nodes, spans[t] ? leaves[t] / spans[t] : leaves[t], (uint32_t)t});
        }
        jobs[t] = FoldJob{f->cur, outs[t], (uint64_t *)layers[t].nodes, half, zetas[3 * t], zetas[3 * t + 1],
                          zetas[3 * t + 2], inv(f->offset), log2u(half), commit ? spans[t] : 0, (uint32_t)t, 0};
        total += fold_blocks(jobs[t]);
        if (total >= (1ull << 31)) {
            release();
            return fail(LVM_ERR_ARG, "batched fold exceeds 2^31 blocks");
        }
        prefix.push_back((uint32_t)total);
    }
    std::vector<uint8_t> blob;
    auto put = [&](const void *p, size_t bytes) {
        const size_t off = (blob.size() + 15) & ~(size_t)15;
        blob.resize(off + bytes);
        std::memcpy(blob.data() + off, p, bytes);
        return off;
    };
    const size_t o_jobs = put(jobs.data(), count * sizeof(FoldJob));
    const size_t o_prefix = put(prefix.data(), prefix.size() * 4);
    struct StepLaunch {
        size_t steps_off, prefix_off;
        uint32_t count, blocks;
    };
    std::vector<StepLaunch> steps_l;
    for (const auto &launch : tree_steps(trees)) {
        std::vector<TreeStep> steps;
        std::vector<uint32_t> sp(1, 0);
        uint64_t sb = 0;
        for (const auto &step : launch) {
            steps.push_back(step.first);
            sb += step.second;
            sp.push_back((uint32_t)sb);
        }
        steps_l.push_back({put(steps.data(), steps.size() * sizeof(TreeStep)), put(sp.data(), sp.size() * 4),
                           (uint32_t)steps.size(), (uint32_t)sb});
    }
    if (lvm_malloc(&arena, blob.size()) != hipSuccess) {
        release();
        return fail(LVM_ERR_NOMEM, "FRI descriptor allocation failed");
    }
    StageScope ss(st);
    hipError_t e = stage_upload(arena, blob.data(), blob.size(), st);
    void *roots = nullptr;
    if (e == hipSuccess && commit) e = stage_result(roots_out, count * 32, nullptr, 0, st, &roots, nullptr);
    if (e == hipSuccess) {
        ProfScope ps(commit ? "fri_fold_leaves" : "fri_fold", st);
        hipLaunchKernelGGL(fri_fold_batched_kernel, dim3((unsigned)total), dim3(FOLD_THREADS), 0, st,
                           (const FoldJob *)(arena + o_jobs), (const uint32_t *)(arena + o_prefix), (uint32_t)count,
                           d->tb.inv_lo, d->tb.inv_hi, (uint64_t *)roots);
    }
    if (e == hipSuccess && commit) {
        ProfScope ps("fri_merkle", st);
        for (const StepLaunch &l : steps_l)
            launch_tree_steps_batched((const TreeStep *)(arena + l.steps_off), (const uint32_t *)(arena + l.prefix_off),
                                      l.count, l.blocks, (uint64_t *)roots, st);
    }
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = stage_sync(st);
    if (e != hipSuccess) {
        release();
        return fail(LVM_ERR_DEVICE, std::string("batched FRI fold: ") + hipGetErrorString(e));
    }
    lvm_free(arena);
    for (size_t t = 0; t < count; t++) {
        lvm_fri *f = fs[t];
        if (f->cur_owned) lvm_free(f->cur);
        f->cur = outs[t];
        f->len /= 2;
        f->offset = sqr(f->offset);
        if (commit) {
            FriLayer &l = layers[t];
            std::memcpy(l.root, roots_out + 32 * t, 32);
            l.evals = outs[t];
            l.len = f->len;
            f->cur_owned = false;
            f->layers.push_back(l);
        } else {
            f->cur_owned = true;
        }
    }
    return LVM_OK;
}

}  // namespace lvm

extern "C" {

int lvm_fri_fold_and_commit_layer(lvm_fri *f, const uint64_t zeta[3], uint8_t root_out[32]) {
    return fri_fold_impl(f, zeta, true, root_out);
}

int lvm_fri_fold(lvm_fri *f, const uint64_t zeta[3]) { return fri_fold_impl(f, zeta, false, nullptr); }

int lvm_fri_current(const lvm_fri *f, uint64_t *host_out, size_t *len, uint64_t *offset) {
    if (!f) return fail(LVM_ERR_ARG, "null handle");
    if (len) *len = f->len;
    if (offset) *offset = f->offset;
    if (!host_out) return LVM_OK;
    Device *d = device_state();
    if (!d) return LVM_ERR_DEVICE;
    StageScope ss(thread_stream(d));
    LVM_HIP(stage_download(host_out, f->cur, f->len * 24, thread_stream(d)));
    LVM_HIP(stage_sync(thread_stream(d)));
    return LVM_OK;
}

int lvm_fri_num_layers(const lvm_fri *f, size_t *count) {
    if (!f || !count) return fail(LVM_ERR_ARG, "null argument");
    *count = f->layers.size();
    return LVM_OK;
}

int lvm_fri_layer(const lvm_fri *f, size_t layer, uint64_t *evals_out, uint8_t *nodes_out, size_t *len) {
    if (!f || layer >= f->layers.size()) return fail(LVM_ERR_ARG, "bad layer index");
    const FriLayer &l = f->layers[layer];
    if (len) *len = l.len;
    Device *d = device_state();
    if (!d) return LVM_ERR_DEVICE;
    if (evals_out) LVM_HIP(hipMemcpyAsync(evals_out, l.evals, l.len * 24, hipMemcpyDeviceToHost, thread_stream(d)));
    if (nodes_out) LVM_HIP(hipMemcpyAsync(nodes_out, l.nodes, (2 * l.L - 1) * 32, hipMemcpyDeviceToHost, thread_stream(d)));
    LVM_HIP(hipStreamSynchronize(thread_stream(d)));
    return LVM_OK;
}

int lvm_fri_query(const lvm_fri *f, const uint64_t *iotas, size_t count, uint64_t *evals_sym_out, uint8_t *paths_out) {
    if (!f || (count && (!iotas || !evals_sym_out || !paths_out))) return fail(LVM_ERR_ARG, "null argument");
    if (count == 0 || f->layers.empty()) return LVM_OK;
    const uint64_t len0 = f->layers[0].len * 2;
    for (size_t i = 0; i < count; i++)
        if (iotas[i] >= len0 / 2) return fail(LVM_ERR_ARG, "query index out of range");
    Device *d = device_state();
    if (!d) return LVM_ERR_DEVICE;
    hipStream_t st = thread_stream(d);
    // per layer: count sym evals (3 u64) and count paths (depth_l x 32 bytes);
    // the layers' descriptors and the indexes go up in one blob
    const size_t layers = f->layers.size();
    std::vector<uint64_t> blob((layers * sizeof(QueryLayer)) / 8 + count);
    QueryLayer *ql = (QueryLayer *)blob.data();
    size_t path_words = 0;
    for (size_t li = 0; li < layers; li++) {
        const FriLayer &l = f->layers[li];
        ql[li] = QueryLayer{l.evals, (const uint64_t *)l.nodes, l.L, path_words, log2u(l.L), 0};
        path_words += count * log2u(l.L) * 4;
    }
    std::memcpy(blob.data() + layers * sizeof(QueryLayer) / 8, iotas, count * 8);
    const size_t sbytes = layers * count * 24, pbytes = path_words * 8;
    // small answers go to mapped host memory from the kernel, larger ones by copy
    const bool direct = sbytes + pbytes <= STAGE_RESULT;
    // released on every exit (stream-ordered: a block is reused on this stream
    // only after the work queued before its release)
    struct Owned {
        uint64_t *p = nullptr;
        ~Owned() {
            if (p) lvm_free(p);
        }
    } dblob, dsym, dpaths;
    LVM_HIP(lvm_malloc(&dblob.p, blob.size() * 8));
    if (!direct) {
        LVM_HIP(lvm_malloc(&dsym.p, sbytes));
        LVM_HIP(lvm_malloc(&dpaths.p, pbytes ? pbytes : 8));
    }
    StageScope ss(st);
    LVM_HIP(stage_upload(dblob.p, blob.data(), blob.size() * 8, st));
    void *sym = dsym.p, *paths = dpaths.p;
    if (direct) LVM_HIP(stage_result(evals_sym_out, sbytes, paths_out, pbytes, st, &sym, &paths));
    // a grid row holds fewer than 2^32 threads: launches of at most 2^24 queries
    constexpr uint64_t MOST = 1u << 24;
    for (uint64_t q = 0; q < count; q += MOST)
        hipLaunchKernelGGL(fri_query_kernel, dim3((unsigned)(count - q < MOST ? count - q : MOST), (unsigned)layers),
                           dim3(128), 0, st, (const QueryLayer *)dblob.p,
                           dblob.p + layers * sizeof(QueryLayer) / 8, q, (uint64_t)count, (uint64_t *)sym,
                           (uint64_t *)paths);
    LVM_HIP(hipGetLastError());
    if (!direct) {
        LVM_HIP(stage_download(evals_sym_out, dsym.p, sbytes, st));
        if (pbytes) LVM_HIP(stage_download(paths_out, dpaths.p, pbytes, st));
    }
    LVM_HIP(stage_sync(st));
    return LVM_OK;
}

int lvm_fri_release(lvm_fri *f) {
    if (!f) return LVM_OK;
    Device *d = device_state();
    if (d) hipStreamSynchronize(thread_stream(d));
    free_fri(f);
    return LVM_OK;
}

}  // extern "C"

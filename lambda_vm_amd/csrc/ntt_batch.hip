// Work-list launches of the NTT passes: one pass shape over several tables
// (the kernels are those of ntt_pass.hpp, their arguments read from memory).
#include "ntt_pass.hpp"

namespace lvm {

// `args[t]` is table t's pass, blocks [prefix[t], prefix[t+1]) are its tiles,
// windows of a run adjacent, XCD-contiguous.
template <int LOG_R1, int LOG_R2, bool COSET, int NJ>
__global__ __launch_bounds__(PASS_T) void ntt_pass_batched_kernel(const PassArgs *__restrict__ args,
                                                                  const uint32_t *__restrict__ prefix,
                                                                  uint32_t count) {
    const uint32_t b = xcd_contiguous(blockIdx.x, gridDim.x);
    const uint32_t t = find_slot(prefix, count, b);
    const PassArgs a = args[t];
    ntt_pass_body<LOG_R1, LOG_R2, COSET, NJ>(a, b - prefix[t]);
}

void launch_pass_batched(int r, bool coset, uint32_t rows, const PassArgs *d_args, const uint32_t *d_prefix,
                         uint32_t count, uint32_t blocks, hipStream_t st) {
    if (blocks == 0) return;
    with_radix(r, [&](auto A, auto B) {
        with_rows(rows, [&](auto NJ) {
            if (coset)
                hipLaunchKernelGGL((ntt_pass_batched_kernel<A(), B(), true, NJ()>), dim3(blocks), dim3(PASS_T), 0, st,
                                   d_args, d_prefix, count);
            else
                hipLaunchKernelGGL((ntt_pass_batched_kernel<A(), B(), false, NJ()>), dim3(blocks), dim3(PASS_T), 0, st,
                                   d_args, d_prefix, count);
        });
    });
}

}  // namespace lvm

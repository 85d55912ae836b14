// The prefill GEMM's kernels with bf16 activations (a file per type, so that they build side by side).
#include "hm_gemm_kernel.hpp"

hipError_t hm::launch_gemm_bf16(const GemmArgs &a, int group, bool fused, int cfg, dim3 grid, hipStream_t s) {
    return launch_t<BF16>(a, group, fused, cfg, grid, s, AllTiles{});
}

hipError_t hm::launch_gemm_bf16_large_scales(const GemmArgs &a, int group, bool fused, dim3 grid, hipStream_t s) {
    return launch_t<BF16Large>(a, group, fused, kLargeScaleTile, grid, s, std::integer_sequence<int, kLargeScaleTile>{});
}

// The prefill GEMM's kernels with fp16 activations (a file per type, so that they build side by side).
#include "hm_gemm_kernel.hpp"

hipError_t hm::launch_gemm_f16(const GemmArgs &a, int group, bool fused, int cfg, dim3 grid, hipStream_t s) {
    return launch_t<F16>(a, group, fused, cfg, grid, s, AllTiles{});
}

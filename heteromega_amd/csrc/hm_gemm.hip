// Prefill W4A16 GEMM (M > 16): launch planning. The kernels are in hm_gemm_kernel.hpp.
#include "hm_gemm.hpp"

#include <algorithm>
#include <cmath>

namespace hm {
namespace {

// K splits and K groups change the order of an output element's sum. Calls of more than kFreeRows rows whose 128 x 128
// tiles fill the CUs (long K: 1.25 times the CUs) take neither: a row block, a column range or a concatenated matrix computed
// alone gives the bits of the whole call where both calls are of this kind.
constexpr int64_t kFreeRows = 256;
constexpr int64_t kLongK = 64; // K tiles
constexpr int64_t kMaxSplits = 12;

bool may_split(int64_t m, int64_t cols, int64_t kt, int64_t cus) {
    const int64_t tiles = (m + 127) / 128 * (cols / 128);
    return m <= kFreeRows || tiles < cus || (kt >= kLongK && 4 * tiles < 5 * cus);
}

// Estimated time of a launch in us: what a CU's workgroups take one after the other (each run of `its` K tiles at a cost
// per tile that grows with the rows, plus what filling the pipeline and writing the tile cost), beside the time the weights
// take to stream, plus the launch, the exchange between K groups and the split sum. The constants are fitted to launches
// measured on three MI355X. Checked by timing every shape it weighs (26398 launches for 324 calls: gate_up, down
// and Q/K/V of Llama-3.2-1B, Llama-3-8B and Qwen2.5-14B, 17 to 2048 rows, fp16 and bf16): the one it picks takes 0.7% longer
// than the fastest on average, up to 3% in 295 of the calls, 1.16 times at worst. Over 1040 random calls (512 to 14336
// columns and K) it takes 0.76 of the time of the three shapes and the rules by grid size that it replaced (0.72 at 17 to 40
// rows, 0.85 past 520); 16 calls are over 2% slower, nearly all of K up to 1152, where the fit has no shapes, and at worst
// 7808 x 6272 at 49 rows, groups of 32, 20.8 -> 23.4 us.
double launch_us(const GemmTile &t, int64_t wgs, int64_t its, int64_t cus, double weight_mb, double partial_mb) {
    const double rounds = static_cast<double>((wgs + cus - 1) / cus);
    const double rb = t.rbw, n = static_cast<double>(its);
    double fixed, busy;
    if (t.wn * t.wk == 4) { // four waves of eight row blocks, two workgroups per CU (alone on its CU one is faster)
        const double pairs = std::floor(rounds / 2), single = rounds - 2 * pairs;
        fixed = 0.5;
        busy = pairs * (n * 1.68 + 0.35 * rb) + single * (n * 1.02 + 0.35 * rb);
    } else {
        const double per = t.wn == 2 ? 0.40 + 0.225 * rb : t.wn == 4 ? 0.49 + (t.kpb == 0 ? 0.149 : 0.157) * rb : 0.75 + 0.103 * rb;
        fixed = t.wn == 2 ? 3.2 : t.wn == 4 ? 2.9 : 0.6;
        busy = rounds * (n * per + 0.35 * rb);
    }
    const double stream = weight_mb / 5.3;
    return fixed + std::sqrt(busy * busy + stream * stream) + (partial_mb > 0 ? 3.0 + 0.36 * partial_mb : 0.0);
}

GemmPlan plan_uncached(int64_t m, int64_t cols, int64_t kt, int64_t cus, bool large_scales) {
    const bool free = may_split(m, cols, kt, cus);
    const double weight_mb = static_cast<double>(kt * 128 * cols) * 0.535e-6; // nibbles and records
    GemmPlan best;
    double best_us = 0;
    for (int i = 0; i < kGemmTileCount; ++i) {
        const GemmTile &t = kGemmTiles[i];
        if (cols % t.cols() != 0 || (!free && t.wk > 1) || (large_scales && i != kLargeScaleTile)) {
            continue;
        }
        const int64_t tiles_m = (m + t.rows() - 1) / t.rows(), tiles_n = cols / t.cols();
        for (int64_t s = 1; s <= (free ? kMaxSplits : 1); ++s) {
            // At least two K tiles per run of a K group, four of a lone one (but one run of any length); partials within
            // their bound.
            const size_t partial = s > 1 ? static_cast<size_t>(s * m * cols) * sizeof(float) : 0;
            if ((s * t.wk > 1 && kt < s * (t.wk > 1 ? 2 * t.wk : 4)) || partial > kGemmPartialMax) {
                break;
            }
            const double us = launch_us(t, tiles_m * tiles_n * s, (kt + s * t.wk - 1) / (s * t.wk), cus, weight_mb, static_cast<double>(partial) * 1e-6);
            if (best.cfg < 0 || us < best_us) {
                best_us = us;
                best.cfg = i;
                best.tiles_m = tiles_m;
                best.tiles_n = tiles_n;
                best.splits = s;
                best.partial_bytes = partial;
            }
        }
    }
    return best;
}

} // namespace

// The last plans of this host thread, by shape: planning weighs up to about two hundred launches (some 2 us), and each
// call plans twice.
GemmPlan plan_gemm(const GemmCall &c) {
    struct Entry {
        int64_t m = 0, cols = 0, kt = 0, cus = 0;
        bool large_scales = false;
        GemmPlan plan;
    };
    constexpr size_t kEntries = 64;
    thread_local Entry cache[kEntries];
    const int64_t cus = device_topology().cus;
    const int64_t cols = c.fused ? 2 * c.n : c.n;
    const uint64_t h = (static_cast<uint64_t>(c.m) * 0x9E3779B97F4A7C15ull) ^ (static_cast<uint64_t>(cols) * 0xC2B2AE3D27D4EB4Full) ^
                       (static_cast<uint64_t>(c.kt_count) * 0x165667B19E3779F9ull);
    Entry &e = cache[(h >> 32) % kEntries];
    if (e.m != c.m || e.cols != cols || e.kt != c.kt_count || e.cus != cus || e.large_scales != c.w.large_scales) {
        e.plan = plan_uncached(c.m, cols, c.kt_count, cus, c.w.large_scales);
        e.large_scales = c.w.large_scales;
        e.m = c.m;
        e.cols = cols;
        e.kt = c.kt_count;
        e.cus = cus;
    }
    return e.plan;
}

// For tests, which choose their shapes by the launch that they get: the plan of m rows, cols columns (fused: gate and up) and
// kt K tiles on `cus` CUs as {tile, its row blocks, waves over columns, K groups, LDS buffers, K tiles per barrier, K splits,
// bytes of partials}. Host code only, and not part of the C ABI.
extern "C" void hm_gemm_plan_of(int64_t m, int64_t cols, int64_t kt, int64_t cus, int32_t large_scales, int64_t out[8]) {
    const GemmPlan p = plan_uncached(m, cols, kt, cus, large_scales != 0);
    const GemmTile t = p.cfg < 0 ? GemmTile{} : kGemmTiles[p.cfg];
    const int64_t v[8] = {p.cfg, t.rbw, t.wn, t.wk, t.depth, t.kpb, p.splits, static_cast<int64_t>(p.partial_bytes)};
    std::copy(v, v + 8, out);
}

size_t gemm_partial_bound(int64_t m, int64_t cols, int64_t kt) {
    return kt < 4 ? 0 : std::min(kGemmPartialMax, static_cast<size_t>(std::min(kMaxSplits, kt / 2) * m * cols) * sizeof(float));
}

hipError_t launch_gemm(const GemmCall &c, hipStream_t stream) {
    const GemmPlan p = plan_gemm(c);
    if (p.cfg < 0) {
        return hipErrorInvalidValue; // columns that no tile divides: the entry points admit multiples of 128 only
    }
    GemmArgs a;
    a.quant = reinterpret_cast<const uint4 *>(c.w.quant);
    a.meta = c.w.meta;
    a.x = c.x;
    a.y = c.y;
    a.partial = p.splits > 1 ? c.partial : nullptr;
    a.ldx = c.ldx;
    a.ldy = c.ldy;
    a.kt_pitch = static_cast<int>(c.w.kt_pitch());
    a.kt_begin = static_cast<int>(c.kt_begin);
    a.kt_count = static_cast<int>(c.kt_count);
    a.splits = static_cast<int>(p.splits);
    a.strip_begin = static_cast<int>(c.strip_begin);
    a.m = static_cast<int>(c.m);
    a.ncols = static_cast<int>(c.fused ? 2 * c.n : c.n);
    a.tiles_m = static_cast<int>(p.tiles_m);
    a.tiles_n = static_cast<int>(p.tiles_n);
    a.accumulate = c.accumulate && !c.fused ? 1 : 0;
    // Tile order: bands of 4 row tiles, column-major inside a band, so the 32 workgroups resident on one XCD
    // hold about 4 row blocks x 8 column blocks: 4 x 32 KiB of activations and 8 x 16 KiB of weights per K tile
    // through its L2, against 32 + 32 x 16 KiB in row-major order. Measured (same bits): Llama-3-8B layer at
    // M = 512 / 1024 / 2048 -2.2 / -1.7 / -1.7%, Qwen2.5-14B at M = 1024 / 2048 -1.7%; bands of 2 gained 1.2-1.4%,
    // of 8 and 16 less or nothing.
    a.group_m = 4;
    a.xcds = device_topology().xcds;
    const dim3 grid(static_cast<unsigned>(p.tiles_m * p.tiles_n), static_cast<unsigned>(p.splits));
    const int group = static_cast<int>(c.w.group);
    const hipError_t e = c.w.dtype == HM_FP16 ? launch_gemm_f16(a, group, c.fused, p.cfg, grid, stream)
                         : c.w.large_scales   ? launch_gemm_bf16_large_scales(a, group, c.fused, grid, stream)
                                              : launch_gemm_bf16(a, group, c.fused, p.cfg, grid, stream);
    if (e != hipSuccess || p.splits == 1) {
        return e;
    }
    return launch_sum_splits(c.partial, c.y, c.ldy, c.m, a.ncols, static_cast<int>(p.splits), c.fused, c.w.dtype, stream, c.accumulate);
}

} // namespace hm

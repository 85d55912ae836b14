// Prefill W4A16 GEMM on the strip layout: v_mfma_f32_16x16x32 with the weights dequantized in registers.
//
// The B operand of v_mfma_f32_16x16x32 (lane l: column l % 16, K 8 (l / 16) .. + 7 of a 32-K step) is the
// strip layout itself (hm_device.hpp): one 16-byte load per lane brings a strip tile's four 32-K steps. So
// each wave loads the nibbles of its own strips straight from memory into registers (no LDS, and no other
// wave dequantizes the same columns), turns each step's dword into (q - z) * s in the activation type, and
// multiplies it with activation fragments read from LDS. The weight rounding to fp16 / bf16 happens once per
// weight, as in the reference GEMM (src/hipkernels/w4a16_gemm_packed.cu:491-497); accumulation is fp32.
//
// Workgroup = WN waves side by side over a 16 RBW x (16 NSW WN) output tile, times WK groups of such waves that take
// WK runs of the K range and add their sums in LDS at the end; a wave owns all 16 RBW rows of NSW strips, so each
// dequantized B operand feeds RBW MFMAs (8 at 128 rows: about two VALU instructions per MFMA). The activation tile
// (16 RBW x 128 per K tile and K group) goes from memory straight into LDS (buffer_load ... lds, no registers) and
// serves its group's WN waves; its 16-byte chunks are XOR-swizzled by row so that an MFMA operand read touches 16
// distinct bank groups; one barrier per K tile, per two K tiles for the 256-column tiles, or two per K tile where LDS has room
// for two whole tiles only, which then lie in four buffers of half a K tile (64 K) each.
//
// Software pipeline: while the MFMAs of 32-K step mu run, the VALU builds the B operands of step mu + 1 (of the
// next K tile at mu = 3) and the LDS delivers the activation fragments of step mu + 1; sched_group_barrier
// interleaves one MFMA with its share of the VALU instructions. K tile kt + LOOK's weights and activations are
// requested at the start of K tile kt: LOOK = DEPTH - 1 with one barrier per K tile, 2 (four buffers) with one per two. With
// half tiles the weights are requested two K tiles ahead and the activations three half tiles ahead.
//
// Tiles are dealt to XCDs in contiguous runs (workgroup i runs on XCD i % 8 on an MI355X) of an order that walks bands of 4
// row tiles column by column, so the workgroups resident on one XCD share both activation rows and weight
// columns in its L2.
//
// D element i of lane l is row 4 (l / 16) + i, column l % 16. Fused (gate_up, strips alternating gate / up
// per 16 channels): a wave's strips are the gate and up columns of the same channels in the same lanes, so
// the epilogue writes SiLU(gate) * up with fp32 math and one rounding (kernels/gpu/src/gemm_w4a16.cu:229-275
// fuses the same way).
//
// Few rows (17 to about 256) are bound by how long one wave takes over a K tile, not by memory or the MFMAs: with four
// waves on 128 columns a SIMD held one wave, and 37 rows went through 128-row tiles. Eight waves as two K groups of four (or
// four of two, over 64 columns, where the grid is small) put two waves on each SIMD without fp32 partials through memory,
// and tile heights in steps of 16 rows leave little padding. Llama-3-8B layer at M = 37 50.6 -> 37.0 us (gate_up 36 -> 21),
// Qwen2.5-14B at M = 100 88 -> 68, the 4096 + 10240 K-split pair at M = 200 60.5 -> 47.6, Llama-3.2-1B block at M = 300
// 60 -> 51. Without K groups and K splits every output element accumulates in the same order for any M and
// tile shape. A K split (blockIdx.y = split) writes fp32 partials, which sum_splits adds in split order, SwiGLU when
// fused.
#pragma once

#include "hm_device.hpp"
#include "hm_gemm.hpp"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace hm {

namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// Per (strip, group) dequantization constants, made once per K tile from the scale/zero record.
template <class T> struct Deq;
// fp16: d2 = (1024 + z) in both halves, s2 = s in both halves.
// fp16 with the wide nibble positions: pairs 1 and 3 of a dword come out as 1024 + 16 q, so they take
// d2w = 1024 + 16 z and s2w = s / 16 (exact for s >= 2^-10; smaller scales lose their low bits in s / 16).
template <> struct Deq<F16> {
    uint32_t d2, s2, d2w, s2w;
};
// bf16: s, -(1024 + z) s and, for the wide positions, s / 16 and -(1024 + 16 z) s / 16 in fp32 (all exact for scales
// below 2^117).
template <> struct Deq<BF16> {
    float s, d, sw, dw;
};
// bf16 matrices with scales from 2^117 on, where 1024 s leaves fp32: s and z.
struct BF16Large : BF16 {};
template <> struct Deq<BF16Large> {
    float s, z;
};

__device__ __forceinline__ Deq<F16> make_deq(uint32_t rec, F16) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const uint32_t z = (rec >> 16) & 0xFFu;
    const uint32_t d = 0x6400u + z;      // fp16 bits of 1024 + z (z <= 16)
    const uint32_t dw = 0x6400u + 16u * z; // fp16 bits of 1024 + 16 z
    const uint32_t sb = rec & 0xFFFFu;
    const h2 s16 = __builtin_bit_cast(h2, sb | (sb << 16)) * h2{static_cast<_Float16>(0.0625f), static_cast<_Float16>(0.0625f)};
    return Deq<F16>{d | (d << 16), sb | (sb << 16), dw | (dw << 16), __builtin_bit_cast(uint32_t, s16)};
}

__device__ __forceinline__ Deq<BF16> make_deq(uint32_t rec, BF16) {
    const float s = bf16_bits_to_float(rec & 0xFFFFu);
    const float z = static_cast<float>((rec >> 16) & 0xFFu);
    const float sw = 0.0625f * s;
    return Deq<BF16>{s, (-1024.0f - z) * s, sw, __builtin_fmaf(z, -s, -1024.0f * sw)};
}

__device__ __forceinline__ Deq<BF16Large> make_deq(uint32_t rec, BF16Large) {
    return Deq<BF16Large>{bf16_bits_to_float(rec & 0xFFFFu), static_cast<float>((rec >> 16) & 0xFFu)};
}

// B operand of one 32-K step from one strip dword: (q - z) * s in the activation type.
// fp16: (1024 + q) - (1024 + z) is exact, one rounding in the multiply by s.
__device__ __forceinline__ uint4 dequant_operand(uint32_t w, const Deq<F16> &q, const MagicRegs &m) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 d2 = __builtin_bit_cast(h2, q.d2);
    const h2 s2 = __builtin_bit_cast(h2, q.s2);
    const h2 d2w = __builtin_bit_cast(h2, q.d2w);
    const h2 s2w = __builtin_bit_cast(h2, q.s2w);
    const uint32_t u = w >> 8;
    // dword i holds K elements 2i, 2i + 1 (nibbles i and 4 + i); (16 (q - z)) (s / 16) = (q - z) s exactly
    uint4 b;
    b.x = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(h2, (w & m.lo) | m.magic) - d2) * s2);
    b.y = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(h2, (w & m.hi) | m.magic) - d2w) * s2w);
    b.z = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(h2, (u & m.lo) | m.magic) - d2) * s2);
    b.w = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(h2, (u & m.hi) | m.magic) - d2w) * s2w);
    return b;
}

// bf16: exact (q - z) * s in fp32, then one round to nearest even (v_cvt_pk_bf16_f32). The nibbles become fp16 pairs
// 1024 + q and 1024 + 16 q as above, and each half goes through one fp32 FMA that reads it in place
// (v_fma_mix_f32: an fp16 half times fp32 plus fp32): (1024 + q) s - (1024 + z) s = (q - z) s, and
// (1024 + 16 q) (s / 16) - (1024 + 16 z) (s / 16) likewise. Both products' constants are exact in fp32 (11 + 8
// significant bits) and the sum has at most 13, so the FMA is exact. gfx950 has no packed bf16 arithmetic; this takes 17
// VALU instructions per dword against 23 for nibbles spread to bytes, v_cvt_f32_ubyte, FMA and the conversion: Llama-3-8B
// layer at M = 512 190 -> 179 us, Llama-3.2-1B block at M = 300 59.8 -> 57.2, a 4096 + 10240 K-split pair at M = 200
// 59.9 -> 57.7, the same bits.
__device__ __forceinline__ uint4 dequant_operand(uint32_t w, const Deq<BF16> &q, const MagicRegs &m) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const uint32_t u = w >> 8;
    auto pair = [&](uint32_t bits, float s, float d) __attribute__((always_inline)) {
        const h2 v = __builtin_bit_cast(h2, bits);
        const f2 r = {__builtin_fmaf(static_cast<float>(v[0]), s, d), __builtin_fmaf(static_cast<float>(v[1]), s, d)};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(r, b2));
    };
    // dword i holds K elements 2i, 2i + 1 (nibbles i and 4 + i)
    return uint4{pair((w & m.lo) | m.magic, q.s, q.d), pair((w & m.hi) | m.magic, q.sw, q.dw), pair((u & m.lo) | m.magic, q.s, q.d),
                 pair((u & m.hi) | m.magic, q.sw, q.dw)};
}

// bf16 with large scales: (q - z) s by a subtraction and a product in fp32, both exact while the weight is finite, for any
// scale. Such matrices hardly exist, so this one is built for a single tile and not tuned.
__device__ __forceinline__ uint4 dequant_operand(uint32_t w, const Deq<BF16Large> &q, const MagicRegs &) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    // dword i holds K elements 2i, 2i + 1 (nibbles i and 4 + i)
    auto pair = [&](int i) __attribute__((always_inline)) {
        const f2 r = {(static_cast<float>((w >> (4 * i)) & 0xFu) - q.z) * q.s, (static_cast<float>((w >> (4 * i + 16)) & 0xFu) - q.z) * q.s};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(r, b2));
    };
    return uint4{pair(0), pair(1), pair(2), pair(3)};
}

template <class T, int G, int NSW> struct BTile {
    u32x4_t w[NSW];           // strip dwords of one K tile
    uint32_t r[NSW][128 / G]; // scale/zero records of its groups
};

template <class T, int G, bool FUSED, int RBW, int NSW, int WN, int WK, int DEPTH, int KPB>
__global__ void __launch_bounds__(WN * WK * 64) __attribute__((amdgpu_waves_per_eu(2))) gemm_kernel(GemmArgs a) {
    constexpr int BM = RBW * 16;
    constexpr int BN = WN * NSW * 16;
    constexpr int GPT = 128 / G;
    constexpr int SPG = 4 / GPT;                  // 32-K steps per group
    constexpr int TRANSFERS = 4 * RBW;            // 1 KiB activation transfers of one K tile
    constexpr int ADMA = (TRANSFERS + WN - 1) / WN; // per wave (past the last: it is repeated, the same bytes to the same place)
    static_assert(WK == 1 || WK == 2 || WK == 4, "K groups");
    static_assert(WK == 1 || KPB < 2, "K groups whose runs differ by a K tile pass the same barriers");
    // K tiles in flight: LOOK tiles ahead of the one being multiplied, each with its weights in registers and its
    // activations in one of DEPTH LDS buffers. Per K tile a wave issues NB weight/record loads and ADMA activation
    // transfers, in that order; all of them count in vmcnt, in order.
    static_assert(DEPTH == 3 || DEPTH == 4, "pipeline depth");
    // KPB = 2: one barrier per two K tiles. Four LDS buffers, K tiles requested two ahead; the barrier after each odd
    // K tile waits for everything in flight (the next two tiles), and the buffer an iteration fills two tiles ahead was
    // last read before the previous barrier.
    // KPB = 0: half tiles. The four LDS buffers hold activations of 64 K each and are refilled every half tile (two
    // barriers per K tile), so that with the bytes of two whole tiles a transfer has 1.25 K tiles' time instead of one;
    // weights are requested two K tiles ahead.
    static_assert(KPB == 1 || DEPTH == 4, "two K tiles per barrier and half tiles: four buffers");
    constexpr bool kHalf = KPB == 0;
    constexpr int LOOK = KPB == 1 ? DEPTH - 1 : 2; // K tiles requested ahead of the one being multiplied
    constexpr int NB = 2 * NSW;
    constexpr int HDMA = (TRANSFERS / 2 + WN - 1) / WN; // transfers per wave per half tile
    constexpr int BUF = WK * BM * (kHalf ? 128 : 256);  // bytes of an LDS buffer
    constexpr int AHEAD = KPB == 2 ? 0 : (DEPTH - 2) * (NB + ADMA); // loads issued after tile kt + 1's activations at iteration kt
    // Activation tile of one K tile: BM rows of 128 halves (256 B), 16-byte chunks XOR-swizzled by row
    // (chunk c of row r at slot c ^ (r % 16)), so the 16 rows one MFMA operand read touches fall on distinct banks.
    // Separate arrays (not one [DEPTH][...]) so that the compiler can tell the buffers apart and does not
    // make reads of one wait for the transfers into the other.
    __shared__ __align__(1024) uint8_t as0[BUF];
    __shared__ __align__(1024) uint8_t as1[BUF];
    __shared__ __align__(1024) uint8_t as2[BUF];
    __shared__ __align__(1024) uint8_t as3[DEPTH > 3 ? BUF : 16];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = uniform(tid >> 6) % WN; // column position
    const int kg = uniform(tid >> 6) / WN;   // K group
    auto abuf = [&](int buf) __attribute__((always_inline)) { return (buf == 0 ? as0 : buf == 1 ? as1 : buf == 2 ? as2 : as3) + kg * (BUF / WK); };
    const int col = lane & 15;
    const int h = lane >> 4;

    // Workgroup -> tile: XCD x = blockIdx.x % xcds takes a contiguous run of the tile order (row-major, or bands
    // of group_m row tiles walked column by column).
    const int nt = a.tiles_m * a.tiles_n;
    const int qx = nt / a.xcds, rx = nt % a.xcds;
    const int xcd = static_cast<int>(blockIdx.x) % a.xcds;
    const int lin = xcd * qx + min(xcd, rx) + static_cast<int>(blockIdx.x) / a.xcds;
    int tm, tn;
    if (a.group_m > 1) {
        const int band_tiles = a.group_m * a.tiles_n;
        const int band = lin / band_tiles;
        const int idx = lin - band * band_tiles;
        const int rows_in_band = min(a.group_m, a.tiles_m - band * a.group_m);
        tm = band * a.group_m + idx % rows_in_band;
        tn = idx / rows_in_band;
    } else {
        tm = lin / a.tiles_n;
        tn = lin - tm * a.tiles_n;
    }
    const int row0 = tm * BM;
    // K split (small grids only): the call's K tiles in a.splits * WK near equal runs (the first ones a tile longer);
    // this group's is [kt_lo, kt_lo + nkt).
    const int split = static_cast<int>(blockIdx.y);
    const int runs = a.splits * WK;
    const int run = split * WK + kg;
    const int base = a.kt_count / runs, longer = a.kt_count % runs;
    const int kt_lo = run * base + min(run, longer);
    const int nkt = base + (run < longer ? 1 : 0);

    // Buffer resources with per-wave bases; per K tile only the scalar offset moves.
    const int sbase = tn * (BN / 16) + wave * NSW; // first strip of this wave within the call
    const int64_t tile0 = static_cast<int64_t>(a.strip_begin + sbase) * a.kt_pitch + a.kt_begin + kt_lo;
    const uint32_t qstrip = static_cast<uint32_t>(a.kt_pitch) * 1024u;
    const uint32_t mstrip = static_cast<uint32_t>(a.kt_pitch) * 64u * GPT;
    const __amdgpu_buffer_rsrc_t qr = buffer_rsrc(reinterpret_cast<const uint8_t *>(a.quant) + tile0 * 1024, NSW * qstrip);
    const __amdgpu_buffer_rsrc_t mr = buffer_rsrc(reinterpret_cast<const uint8_t *>(a.meta) + tile0 * 64 * GPT, NSW * mstrip);
    const uint32_t ldx2 = static_cast<uint32_t>(a.ldx) * 2u;
    const int rows_here = min(BM, a.m - row0);
    if (rows_here <= 0) {
        return; // never for a consistent plan (its last tile row starts below M); a guard against one that is not
    }
    // x column 0 is the call's first K (kt_begin), as for the GEMV.
    const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(reinterpret_cast<const uint8_t *>(a.x) + static_cast<int64_t>(row0) * a.ldx * 2 +
                                                      static_cast<int64_t>(kt_lo) * 256,
                                                  static_cast<uint32_t>(rows_here - 1) * ldx2 + static_cast<uint32_t>(nkt) * 256u);
    // Transfer j of this wave fills LDS bytes [(wave * ADMA + j) KiB, +1 KiB): lane l -> slot p = 64 (wave ADMA + j) + l,
    // row p / 16, swizzled chunk p % 16 (so source chunk (p % 16) ^ (row % 16)). Rows past M read row M - 1.
    // Half tiles: rows of 8 chunks, row p / 8, chunk (p % 8) ^ (row / 2 % 8), so that 16 rows again fall on 16 distinct slots.
    constexpr int XN = kHalf ? HDMA : ADMA;
    constexpr int XT = kHalf ? TRANSFERS / 2 : TRANSFERS;
    uint32_t xoff[XN];
#pragma unroll
    for (int j = 0; j < XN; ++j) {
        const int p = min(wave * XN + j, XT - 1) * 64 + lane;
        const int r = kHalf ? p >> 3 : p >> 4;
        const int c = kHalf ? (p & 7) ^ ((r >> 1) & 7) : (p & 15) ^ (r & 15);
        xoff[j] = static_cast<uint32_t>(min(r, rows_here - 1)) * ldx2 + static_cast<uint32_t>(c) * 16u;
    }
    const uint32_t qoff = static_cast<uint32_t>(lane) * 16u;
    const uint32_t moff = static_cast<uint32_t>(col) * GPT * 4u;

    auto load_b = [&](int kt, BTile<T, G, NSW> &bt) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < NSW; ++s) {
            const uint32_t mo = moff + s * mstrip;
            const uint32_t ms = static_cast<uint32_t>(kt) * (64u * GPT);
            if constexpr (GPT == 1) {
                bt.r[s][0] = __builtin_amdgcn_raw_buffer_load_b32(mr, mo, ms, 0);
            } else if constexpr (GPT == 2) {
                const auto v = __builtin_amdgcn_raw_buffer_load_b64(mr, mo, ms, 0);
                bt.r[s][0] = v[0];
                bt.r[s][1] = v[1];
            } else {
                const auto v = __builtin_amdgcn_raw_buffer_load_b128(mr, mo, ms, 0);
                bt.r[s][0] = v[0];
                bt.r[s][1] = v[1];
                bt.r[s][2] = v[2];
                bt.r[s][3] = v[3];
            }
        }
#pragma unroll
        for (int s = 0; s < NSW; ++s) {
            bt.w[s] = __builtin_amdgcn_raw_buffer_load_b128(qr, qoff + s * qstrip, static_cast<uint32_t>(kt) * 1024u, 0);
        }
    };
    // Activation chunks of K tile (half tiles: of half tile) kt straight into LDS buffer buf (no registers).
    auto load_a = [&](int kt, int buf) __attribute__((always_inline)) {
        const uint32_t so = static_cast<uint32_t>(kt) * (kHalf ? 128u : 256u);
#pragma unroll
        for (int j = 0; j < XN; ++j) {
            lds_dma16(xr, abuf(buf) + min(wave * XN + j, XT - 1) * 1024, xoff[j], so);
        }
    };

    float4_t acc[RBW][NSW];
#pragma unroll
    for (int rb = 0; rb < RBW; ++rb) {
#pragma unroll
        for (int s = 0; s < NSW; ++s) {
            acc[rb][s] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    const MagicRegs magic = magic_regs<F16>();
    constexpr int SHARE = RBW >= 7 ? 2 : (16 + RBW - 1) / RBW; // VALU instructions after each MFMA

    // Software pipeline over the 32-K steps: while the MFMAs of step mu run, the VALU builds the B operands of
    // step mu + 1 (of the next K tile when mu = 3) and the LDS delivers the activation fragments of step mu + 1.
    struct BOps {
        uint4 v[NSW];
    };
    struct AFr {
        uint4 v[RBW];
    };
    // B operands of step mu of tile bt with the constants dqg of its group; the constants are rebuilt when a group starts.
    auto dequant_step = [&](const BTile<T, G, NSW> &bt, Deq<T> (&dqg)[NSW], int mu, BOps &o) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < NSW; ++s) {
            if (mu % SPG == 0) {
                dqg[s] = make_deq(bt.r[s][mu / SPG], T{});
            }
            o.v[s] = dequant_operand(bt.w[s][mu], dqg[s], magic);
        }
    };
    // Fragment of row block rb, step mu: row rb * 16 + col, chunk 4 mu + h at its swizzled slot.
    const uint32_t aread = static_cast<uint32_t>(col) * (kHalf ? 128u : 256u);
    auto read_a = [&](int buf, int mu, AFr &f) __attribute__((always_inline)) {
        const uint8_t *ab = abuf(buf) + aread + (((4 * mu + h) ^ (kHalf ? col >> 1 : col)) << 4);
#pragma unroll
        for (int rb = 0; rb < RBW; ++rb) {
            f.v[rb] = *reinterpret_cast<const uint4 *>(ab + rb * (kHalf ? 2048 : 4096));
        }
    };

    // One K tile in pipeline slot U = kt % DEPTH. On entry `op` holds step 0's B operands of `cur`, `dq` the
    // constants of `cur`, `fa` step 0's activation fragments; on exit the same for K tile kt + 1. The tile LOOK ahead
    // goes into slot (U + LOOK) % DEPTH, whose registers and LDS buffer were last read before the previous barrier.
    // J >= 0: the J-th iteration behind the loop of whole trips. It requests nothing (two tiles ahead with four slots,
    // KPB = 2, the first one there still does), and its waits count what the loop's iterations left in flight: the
    // compiler drops weight loads whose registers nobody reads, and a wait that counted them would let the activation
    // transfers that it is for slip past.
    auto iteration = [&](int kt, const BTile<T, G, NSW> &cur, const BTile<T, G, NSW> &nxt, BTile<T, G, NSW> &ld, Deq<T> (&dq)[NSW], BOps &op,
                         AFr &fa, auto u, auto j) __attribute__((always_inline)) {
        constexpr int U = decltype(u)::value, J = decltype(j)::value;
        constexpr bool kOdd = U % 2 == 1; // KPB = 2: a barrier follows
        constexpr bool kRequest = J < 0 || (KPB == 2 && J == 0);
        constexpr int ISSUED = KPB == 2 ? 0 : J < 0 ? AHEAD : std::max(0, DEPTH - 3 - J) * (NB + ADMA); // after tile kt + 1's activations
        if constexpr (kRequest) {
            const int ktn = min(kt + LOOK, nkt - 1); // the loop's last iterations re-request the last tile; nothing reads it
            load_b(ktn, ld);
            load_a(ktn, (U + LOOK) % DEPTH);
        }
        // The next tile's activations: this wave's transfers done, then everyone's (KPB = 2: after each odd tile, for the
        // next two). Every read of this tile is done too, so the slot that the next iteration fills is free. This stands
        // before the last step's MFMAs, which then cover the LDS latency of the next tile's first fragments.
        auto next_tile = [&]() __attribute__((always_inline)) {
            if constexpr (KPB == 1 || kOdd) {
                wait_vmcnt<ISSUED>();
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            }
        };
#pragma unroll
        for (int mu = 0; mu < 4; ++mu) {
            BOps on;
            AFr fn;
            if (mu < 3) {
                read_a(U, mu + 1, fn);
                dequant_step(cur, dq, mu + 1, on);
            } else {
                // nxt's weights; what was issued after them may still run. KPB = 2: at an odd kt they were requested one
                // iteration ago, before nxt's and this iteration's transfers; at an even kt the barrier before this
                // iteration already waited for them.
                wait_vmcnt<KPB == 1 ? ADMA + ISSUED : !kOdd ? ADMA + NB : kRequest ? 2 * ADMA + NB : ADMA>();
                next_tile();
                read_a((U + 1) % DEPTH, 0, fn);
                dequant_step(nxt, dq, 0, on);
            }
            // strip-major: the operand of the last strip, finished at the end of the previous step, is needed last
#pragma unroll
            for (int s = 0; s < NSW; ++s) {
#pragma unroll
                for (int rb = 0; rb < RBW; ++rb) {
                    acc[rb][s] = T::mfma16(fa.v[rb], op.v[s], acc[rb][s]);
                }
            }
#pragma unroll
            for (int i = 0; i < RBW * NSW; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);     // one MFMA
                __builtin_amdgcn_sched_group_barrier(0x002, SHARE, 0); // then a share of the next step's operand build
            }
            __builtin_amdgcn_sched_barrier(0);
            op = on;
            fa = fn;
        }
    };

    // Half tiles: the same over the half tiles 2 kt and 2 kt + 1 in LDS buffers 2 U % 4 and the next one. Half tile 2 kt + 3
    // goes where 2 kt - 1 was, 2 kt + 4 where 2 kt was, each behind the barrier after that one's last read.
    auto iteration_half = [&](int kt, const BTile<T, G, NSW> &cur, const BTile<T, G, NSW> &nxt, BTile<T, G, NSW> &ld, Deq<T> (&dq)[NSW], BOps &op,
                              AFr &fa, auto u, auto j) __attribute__((always_inline)) {
        constexpr int U = decltype(u)::value, J = decltype(j)::value;
        // Behind the loop: only what a later iteration there reads (J = 0: weights two ahead; J = 0, 1: activations).
        constexpr bool kWeights = J <= 0, kFirst = J <= 1, kSecond = J <= 0;
#pragma unroll
        for (int mu = 0; mu < 4; ++mu) {
            BOps on;
            AFr fn;
            if (mu == 0) {
                if constexpr (kWeights) {
                    load_b(min(kt + LOOK, nkt - 1), ld);
                }
                if constexpr (kFirst) {
                    load_a(min(2 * kt + 3, 2 * nkt - 1), (2 * U + 3) % 4);
                }
            }
            if (mu == 2) {
                if constexpr (kSecond) {
                    load_a(min(2 * kt + 4, 2 * nkt - 1), (2 * U) % 4);
                }
            }
            if (mu == 1) { // half tile 2 kt + 1 landed (issued after it: 2 kt + 2, then this iteration's first requests)
                wait_vmcnt<J <= 0 ? 2 * HDMA + NB : J == 1 ? 2 * HDMA : 0>();
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            }
            if (mu == 3) { // half tile 2 kt + 2 landed (after it: this iteration's requests)
                wait_vmcnt<J <= 0 ? 2 * HDMA + NB : J == 1 ? HDMA : 0>();
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            }
            read_a((2 * U + (mu + 1) / 2) % 4, (mu + 1) % 2, fn);
            if (mu < 3) {
                dequant_step(cur, dq, mu + 1, on);
            } else {
                dequant_step(nxt, dq, 0, on);
            }
#pragma unroll
            for (int s = 0; s < NSW; ++s) {
#pragma unroll
                for (int rb = 0; rb < RBW; ++rb) {
                    acc[rb][s] = T::mfma16(fa.v[rb], op.v[s], acc[rb][s]);
                }
            }
#pragma unroll
            for (int i = 0; i < RBW * NSW; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, SHARE, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            op = on;
            fa = fn;
        }
    };

    BTile<T, G, NSW> b[DEPTH];
    // The waits below count these in this order.
    if constexpr (kHalf) {
        load_b(0, b[0]);
        __builtin_amdgcn_sched_barrier(0);
        load_a(0, 0);
        __builtin_amdgcn_sched_barrier(0);
        load_b(min(1, nkt - 1), b[1]);
        __builtin_amdgcn_sched_barrier(0);
        load_a(1, 1);
        __builtin_amdgcn_sched_barrier(0);
        load_a(min(2, 2 * nkt - 1), 2);
        __builtin_amdgcn_sched_barrier(0);
    } else {
#pragma unroll
        for (int t = 0; t < LOOK; ++t) {
            load_b(min(t, nkt - 1), b[t]);
            load_a(min(t, nkt - 1), t);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    Deq<T> dq[NSW];
    BOps op;
    AFr fa;
    if constexpr (kHalf) {
        wait_vmcnt<3 * HDMA + NB>();
    } else if constexpr (KPB == 2) {
        wait_vmcnt<2 * ADMA + NB>(); // tile 0's weights (tile 0's transfers and tile 1's loads may still run)
    } else {
        wait_vmcnt<ADMA + AHEAD>();
    }
    dequant_step(b[0], dq, 0, op);
    wait_vmcnt<kHalf ? 2 * HDMA + NB : AHEAD>();
    asm volatile("s_barrier" ::: "memory");
    read_a(0, 0, fa);
    // DEPTH K tiles per trip, so the register sets and LDS buffers rotate without copies.
    auto one = [&](int k, auto u, auto j) __attribute__((always_inline)) {
        constexpr int U = decltype(u)::value;
        if constexpr (kHalf) {
            iteration_half(k, b[U], b[(U + 1) % DEPTH], b[(U + LOOK) % DEPTH], dq, op, fa, u, j);
        } else {
            iteration(k, b[U], b[(U + 1) % DEPTH], b[(U + LOOK) % DEPTH], dq, op, fa, u, j);
        }
    };
    using Steady = std::integral_constant<int, -1>;
    int kt = 0;
    for (; kt + DEPTH - 1 < nkt; kt += DEPTH) {
        one(kt, std::integral_constant<int, 0>{}, Steady{});
        one(kt + 1, std::integral_constant<int, 1>{}, Steady{});
        one(kt + 2, std::integral_constant<int, 2>{}, Steady{});
        if constexpr (DEPTH > 3) {
            one(kt + 3, std::integral_constant<int, 3>{}, Steady{});
        }
    }
    if (kt < nkt) {
        one(kt, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
    }
    if (kt + 1 < nkt) {
        one(kt + 1, std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
    }
    if constexpr (DEPTH > 3) {
        if (kt + 2 < nkt) {
            one(kt + 2, std::integral_constant<int, 2>{}, std::integral_constant<int, 2>{});
        }
    }

    // K groups: the sums meet in LDS, in as0 (free once every transfer has landed and every wave has read its last
    // fragments). Of four groups the upper two first give theirs to the lower two; of two, each gives one half of the
    // row blocks and finishes the other. A group with a K tile less waits here for the others' last barrier.
    constexpr int HALF = WK > 1 ? (RBW + 1) / 2 : RBW;
    if constexpr (WK > 1) {
        static_assert(WK / 2 * WN * RBW * NSW * 1024 <= BUF * (kHalf ? 2 : 1), "exchange buffer");
        // column positions per buffer: all in as0, or (half tiles) the upper half in as1
        constexpr int PER = kHalf ? WK / 2 * WN / 2 : WK / 2 * WN;
        auto slot = [&](int pair) __attribute__((always_inline)) {
            const int i = pair * WN + wave;
            return reinterpret_cast<float4_t *>(i < PER ? as0 : as1) + i % PER * (RBW * NSW * 64) + lane;
        };
        const int longest = base + (split * WK < longer ? 1 : 0); // the split's first run
        if (nkt < longest) {
            asm volatile("s_barrier" ::: "memory");
            if constexpr (kHalf) {
                asm volatile("s_barrier" ::: "memory");
            }
        }
        wait_vmcnt<0>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        auto give = [&](int pair, auto lo, auto hi) __attribute__((always_inline)) {
            float4_t *xch = slot(pair);
#pragma unroll
            for (int rb = decltype(lo)::value; rb < decltype(hi)::value; ++rb) {
#pragma unroll
                for (int s = 0; s < NSW; ++s) {
                    xch[(rb * NSW + s) * 64] = acc[rb][s];
                }
            }
        };
        auto take = [&](int pair, auto lo, auto hi) __attribute__((always_inline)) {
            const float4_t *xch = slot(pair);
#pragma unroll
            for (int rb = decltype(lo)::value; rb < decltype(hi)::value; ++rb) {
#pragma unroll
                for (int s = 0; s < NSW; ++s) {
                    acc[rb][s] += xch[(rb * NSW + s) * 64];
                }
            }
        };
        using Zero = std::integral_constant<int, 0>;
        using Half = std::integral_constant<int, HALF>;
        using All = std::integral_constant<int, RBW>;
        if constexpr (WK == 4) {
            if (kg >= 2) {
                give(kg - 2, Zero{}, All{});
            }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (kg < 2) {
                take(kg, Zero{}, All{});
            }
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        if (kg == 0) {
            give(0, Half{}, All{});
        } else if (WK == 2 || kg == 1) {
            give(0, Zero{}, Half{});
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (kg >= 2) {
            return;
        }
        if (kg == 0) {
            take(0, Zero{}, Half{});
        } else {
            take(0, Half{}, All{});
        }
    }
    // Row blocks this wave writes.
    auto mine = [&](int rb) __attribute__((always_inline)) { return WK == 1 || (rb < HALF) == (kg == 0); };

    if (a.partial != nullptr) {
        // K split: fp32 partials [split][m][ncols] (strip order, so a fused call's gate and up columns alternate
        // per 16), added by sum_splits. Rows past M fall outside the buffer and are dropped: the row offset is
        // part of the vector offset, which the buffer range check covers (the scalar offset is not checked).
        const uint32_t ldp4 = static_cast<uint32_t>(a.ncols) * 4u;
        const __amdgpu_buffer_rsrc_t pr =
            buffer_rsrc(a.partial + (static_cast<int64_t>(split) * a.m + row0) * a.ncols, static_cast<uint32_t>(rows_here) * ldp4);
        const uint32_t pcol = static_cast<uint32_t>(4 * h) * ldp4 + static_cast<uint32_t>(sbase * 16 + col) * 4u;
#pragma unroll
        for (int rb = 0; rb < RBW; ++rb) {
            if (!mine(rb)) {
                continue;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t ro = static_cast<uint32_t>(rb * 16 + i) * ldp4;
#pragma unroll
                for (int s = 0; s < NSW; ++s) {
                    // Element first: a bit cast of a vector element expression reads element 0.
                    const float v = acc[rb][s][i];
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), pr, pcol + ro + s * 64u, 0, 0);
                }
            }
        }
        return;
    }
    // Epilogue through a buffer covering this tile's valid rows: stores of rows past M fall outside it and are
    // dropped by the buffer range check, so no per-row branch. The row offset goes into the vector offset: the
    // range check covers the vector and instruction offsets, not the scalar offset.
    const uint32_t ldy2 = static_cast<uint32_t>(a.ldy) * 2u;
    const __amdgpu_buffer_rsrc_t yr = buffer_rsrc(a.y + static_cast<int64_t>(row0) * a.ldy, static_cast<uint32_t>(rows_here) * ldy2);
    const uint32_t ycol = static_cast<uint32_t>(4 * h) * ldy2 + static_cast<uint32_t>(FUSED ? sbase / 2 * 16 + col : sbase * 16 + col) * 2u;
#pragma unroll
    for (int rb = 0; rb < RBW; ++rb) {
        if (!mine(rb)) {
            continue;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t ro = static_cast<uint32_t>(rb * 16 + i) * ldy2;
            if constexpr (FUSED) {
#pragma unroll
                for (int s = 0; s < NSW; s += 2) {
                    const uint16_t v = T::from_float(silu(acc[rb][s][i]) * acc[rb][s + 1][i]);
                    __builtin_amdgcn_raw_buffer_store_b16(v, yr, ycol + ro + (s / 2) * 32u, 0, 0);
                }
            } else {
#pragma unroll
                for (int s = 0; s < NSW; ++s) {
                    uint16_t v = T::from_float(acc[rb][s][i]);
                    if (a.accumulate) {
                        v = T::from_float(T::to_float(__builtin_amdgcn_raw_buffer_load_b16(yr, ycol + ro + s * 32u, 0, 0)) + T::to_float(v));
                    }
                    __builtin_amdgcn_raw_buffer_store_b16(v, yr, ycol + ro + s * 32u, 0, 0);
                }
            }
        }
    }
}

template <class T, int G, bool FUSED, int I> hipError_t launch_tile(const GemmArgs &a, dim3 grid, hipStream_t s) {
    constexpr GemmTile t = kGemmTiles[I];
    hipLaunchKernelGGL((gemm_kernel<T, G, FUSED, t.rbw, 2, t.wn, t.wk, t.depth, t.kpb>), grid, dim3(t.wn * t.wk * 64), 0, s, a);
    return hipGetLastError();
}

template <class T, int G, int... I>
hipError_t launch_g(const GemmArgs &a, bool fused, int cfg, dim3 grid, hipStream_t s, std::integer_sequence<int, I...>) {
    hipError_t e = hipErrorInvalidValue;
    (void)((cfg == I && ((e = fused ? launch_tile<T, G, true, I>(a, grid, s) : launch_tile<T, G, false, I>(a, grid, s)), true)) || ...);
    return e;
}

// The tiles I... are built; cfg is one of them.
template <class T, int... I>
hipError_t launch_t(const GemmArgs &a, int group, bool fused, int cfg, dim3 grid, hipStream_t s, std::integer_sequence<int, I...> tiles) {
    switch (group) {
    case 32:
        return launch_g<T, 32>(a, fused, cfg, grid, s, tiles);
    case 64:
        return launch_g<T, 64>(a, fused, cfg, grid, s, tiles);
    default:
        return launch_g<T, 128>(a, fused, cfg, grid, s, tiles);
    }
}
using AllTiles = std::make_integer_sequence<int, kGemmTileCount>;

} // namespace

} // namespace hm

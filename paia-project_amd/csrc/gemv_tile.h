// Small-batch GEMV for gfx950, streaming form: M = 2..16 activation rows against one weight matrix, the kernel behind
// the small-batch entry points when the caller leaves the choice to the library.
//
//   y[m, n] = bf16_rn( sum_k deq(W[n,k]) * x[m,k]  (+ bias[n]) ),   x bf16 [M][K], y bf16 [M][N]
//
// Same formats, contraction (v_mfma_f32_16x16x32_bf16, A = x, B = dequantised weights, fp32 accumulation) and tile (16
// weight rows) as gemv_batch_kernel; what differs is how the operands reach the matrix cores and how K is split.
//
// What bounded gemv_batch_kernel: it loads each operand straight into its MFMA lane (lane l = row l%16), so the four
// lanes a load instruction takes per cycle lie in four rows and the texture path spends a cycle on each 16 bytes instead
// of one per 64. At M = 16 that, the restaging of x per block and load waits that drained at every loop head held FP8
// gate_up 28672x4096 at 29.4 us where the bytes take 17.2 at the rate of a streaming read.
//   * Every load here is row-contiguous: 8 consecutive lanes read 128 bytes of one weight row (INT4: 4 lanes, 64 bytes), and
//     x the same way. A wave passes its own data through a private piece of LDS (ds_write_b128, ds_read_b128, XOR swizzle
//     against bank conflicts) to bring it into the MFMA layout: no block barrier, and LDS operations of a wave complete in
//     order, so a slot can be rewritten behind the reads of its last contents. Weights are then worth the streaming (nt)
//     policy: 25.1 -> 21.9 us on that shape, where it cost gemv_batch_kernel 10%.
//   * K is split over S waves of the block. A wave takes its stages (BF16 64 columns, the others 128) for P tiles at a
//     time, so each x fragment it brings in is used P times, with D stages of loads in flight; the S partial tiles are
//     added in a fixed order after the one block barrier at the end. The operands of that epilogue (row scale, bias) are
//     loaded before the first weight load: loaded at the end they cost 1.2 us per launch (FP8 4096x4096 M = 4 6.98 -> 5.68).
//   * INT4 scales and zero points: per-group loads in the loop would touch 16 rows each, as many lines as the weights
//     themselves. The block loads its rows' once, four groups per lane and ahead of its weight loads, and keeps them in LDS
//     as [group][row] words (scale in the upper half, zero point in the low byte): one conflict-free read per tile and
//     stage, one VALU operation each to unpack.
//   * INT4 nibbles are decoded exactly: the byte value q in 0..15 read as e4m3 is q 2^-9 (0..7 subnormal, 8..15 in the
//     first binade), so v_cvt_scalef32_pk_bf16_fp8 gives q times any power of two. No 128 offset to cancel, the same 7 VALU
//     per 8 weights as placing them under a 0x43 byte.
// Rows of D are independent and the split order is fixed, so results are bitwise reproducible and a row's result does not
// depend on the other rows of the call.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <type_traits>

#include "gemv_batch.h"
#include "gemv_device.h"
#include "gemv_kernel.h"

namespace paia {

struct TileParams {
    const uint8_t* W;       // weight rows, row_bytes each
    const uint8_t* meta;    // FP8: fp32 scale [N]; INT4: fp16 scale [N][G]; INT4ZP: bf16 scale [N][G]
    const uint8_t* zeros;   // INT4ZP: [N][zbytes] packed 4-bit zero points
    const uint16_t* x;      // bf16 [M][K]
    const uint16_t* bias;   // bf16 [N] or null
    uint16_t* y;            // bf16 [M][N]
    int M, N, K;
    uint32_t row_bytes, meta_bytes, zbytes;
    int stages;             // ceil(K / columns per stage)
    int tq, tr;             // unit u (a group of S waves) takes tiles tq*u + min(u, tr) .. of its next unit: tq or tq + 1
    int chunks;             // INT4: ceil(G / 4), four-group chunks per row
    uint32_t chunk_mul;     // ceil(2^32 / chunks): i / chunks as the high word of i * chunk_mul (i * chunks < 2^32)
    int mstride;            // INT4: words per group in LDS (the most rows a block takes, plus one against bank conflicts)
    int wide;               // INT4: every chunk's loads are aligned (G % 4 == 0 and aligned bases)
    uint32_t wave_off;      // LDS: first wave's private region
};

template <int F>
struct TileFmt {
    static constexpr bool kI4F = F == kI4 || F == kI4ZP;
    static constexpr int kCols = F == kBF16 ? 64 : 128;             // columns per stage
    static constexpr int kRowBytes = F == kBF16 || F == kFP8 ? 128 : 64;   // weight bytes per row and stage
    static constexpr int kLoads = kRowBytes * kTileRows / kChunkBytes;    // 16-byte weight loads per lane, tile and stage
    static constexpr int kSteps = kCols / 32;                       // MFMA steps per stage
    static constexpr int kXRows = kChunkBytes / (2 * kCols);        // activation rows one load of a wave brings
};

// A wave's private LDS: one stage of x (MT rows), then the stage's weights of two tiles (in order within the wave: the
// third tile's weights overwrite the first's behind their reads), reused for the wave's P partial tiles at the end.
constexpr int kTileSlots = 2;
// RING: the last two 128-byte lines of each of the P tiles' rows instead.
template <int F, int P, int MT, bool RING>
__host__ __device__ constexpr uint32_t tile_wave_bytes()
{
    const uint32_t x = (uint32_t)MT * 2u * TileFmt<F>::kCols;
    const uint32_t w = (uint32_t)(RING ? 2 * P : (P < kTileSlots ? P : kTileSlots)) * kTileRows * TileFmt<F>::kRowBytes;
    return x + w > (uint32_t)P * 1024u ? x + w : (uint32_t)P * 1024u;
}

// LDS order between a lane's writes and other lanes' reads of one wave: the hardware keeps a wave's LDS operations in
// order, the compiler has to (no instruction comes of it).
__device__ __forceinline__ void wave_lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// INT4: the 128 terms of a group, up to 15 |x| each, could leave fp32's range where |x| reaches 2^116 although the output
// (scales are small) does not. So nibbles and sums of x carry a factor 2^-11: no finite x overflows, and at the other end
// nothing is lost (a bf16 x is a multiple of 2^-133, its products of 2^-144, and the matrix cores keep subnormals down to
// 2^-149). The scales carry 2^4 of it back, and the finished sums the rest: sums over the groups have 2^7 of room beyond
// fp32's range, and steps of 2^-142 where the smallest outputs are 2^-133 apart (with all 2^11 left to the end the steps
// were 2^-138, and outputs below 2^-126 had 5% more error). An asymmetric scale that does not take the 2^4 (2^124 or more)
// is kept as it is, with the 2^4 on its nibbles and zero point instead.
constexpr uint32_t kI4Exp = 125, kI4ExpBig = 129;      // factor on q 2^-9 as e4m3, as a float's exponent: 2^-2, 2^2
constexpr uint32_t kI4Ones = 0x3A003A00u;              // a bf16 pair of 2^-11
constexpr float kI4Up = 16.0f, kI4Back = 128.0f, kF32Max = 3.4028234e38f;

// Metadata word of an asymmetric group (scale bf16 in the upper half of `s`): scale, exponent of the nibbles' factor, zero
// point. The scale's 2^4 is exact in bf16, also for a subnormal one.
__device__ __forceinline__ uint32_t i4zp_word(float up, uint32_t z) { return __float_as_uint(up) | kI4Exp << 8 | z; }
__device__ __forceinline__ uint32_t i4zp_word_big(uint32_t s, uint32_t z) { return s | kI4ExpBig << 8 | z << 4; }

// e4m3 byte pair HI of w (0..15 each) -> the two integers times 2^-9 and the scale's power of two (the conversion takes the
// exponent field of `scale` only), as bf16
template <bool HI>
__device__ __forceinline__ uint32_t i4x2_to_bf16x2(uint32_t w, float scale)
{
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, scale, HI));
}

// P tiles per unit, S waves sharing them along K (W / S units per block; every launch has one, S = W, but the schedule the
// compiler finds with the single unit written in was 0.5 to 3% slower: INT4ZP 14336x4096 M = 8 10.04 -> 10.09 us,
// 58559x4608 36.0 -> 37.2), D stages in flight per wave, MT activation
// rows staged (4, 8 or 16 >= M), AUX cache policy of the weight loads, IL: a unit's waves take the stages in turn
// (neighbouring waves read neighbouring bytes of a row) rather than a contiguous range each.
// RING (BF16, FP8; not IL): for rows that are no multiple of 128 bytes, where a stage's 128 bytes of a row lie in two lines
// and each line would be read twice (and fetched 1.6 times: with nt it is gone by the second read). A wave reads the lines of
// its range once each, whole, and a stage takes its columns from the row's last two lines in LDS.
template <int F, int P, int W, int S, int D, int MT, int AUX, bool IL, bool RING>
__global__ void __launch_bounds__(W * kWave, W / 4) gemv_tile_kernel(TileParams p)
{
    using T = TileFmt<F>;
    constexpr bool I4 = T::kI4F;
    constexpr int C = T::kCols, RB = T::kRowBytes, L = T::kLoads, X = T::kSteps, XR = T::kXRows;
    constexpr int XL = (MT + XR - 1) / XR;            // x loads per stage
    constexpr int WP = RB / 16, WR = kWave / WP;      // 16-byte pieces per weight row and stage, rows per load
    constexpr int XP = 2 * C / 16;                    // 16-byte pieces per x row and stage
    constexpr int kUnits = W / S;
    constexpr int kSlots = RING || P < kTileSlots ? P : kTileSlots;
    constexpr uint32_t kXBytes = (uint32_t)MT * 2u * C, kSlotBytes = (uint32_t)kTileRows * RB * (RING ? 2u : 1u);
    constexpr uint32_t kWaveBytes = tile_wave_bytes<F, P, MT, RING>();
    constexpr int kOuts = (kUnits * P + W - 1) / W;   // tiles a wave reduces and stores
    static_assert(W % S == 0 && (MT == 4 || MT == 8 || MT == 16), "launch shape");
    static_assert(!RING || (!I4 && !IL), "lines of contiguous ranges");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int lane = lane_id(), wave = wave_id();
    const int ln = lane & 15, lh = lane >> 4;
    const int split = wave % S, unit = wave / S;
    // logical block: each of the 8 XCDs (workgroups are dealt to them in turn) takes a contiguous range of tiles, so the
    // lines of y, scales and bias that tiles share are touched by one L2
    int lb = (int)blockIdx.x;
    {
        const int g = (int)gridDim.x, xcd = lb % 8, per = g / 8, rem = g % 8;
        lb = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + lb / 8;
    }
    auto tile_at = [&](int u) { return u * p.tq + min(u, p.tr); };
    const int u0 = lb * kUnits;
    const int t0 = tile_at(u0 + unit), nt = tile_at(u0 + unit + 1) - t0;   // this unit's tiles, nt <= P
    const int k0 = IL ? split : split * p.stages / S;
    const int n = IL ? (p.stages - split + S - 1) / S : (split + 1) * p.stages / S - k0;   // this wave's stages
    // RING: line t = 0 only fills the ring, line t > 0 completes stage t - 1 of the range
    const int nl = RING ? (n > 0 ? n + 1 : 0) : n;
    auto stage_at = [&](int t) { return IL ? k0 + t * S : (RING ? k0 + t - 1 : k0 + t); };

    // INT4 metadata of the block's rows: item i is four groups of one row
    const int bt0 = tile_at(u0), brows = I4 ? max(0, min((tile_at(u0 + kUnits) - bt0) * kTileRows, p.N - bt0 * kTileRows)) : 0;
    const size_t brow0 = brows > 0 ? (size_t)(bt0 * kTileRows) : 0;
    const __amdgpu_buffer_rsrc_t rsm = make_rsrc(p.meta + (I4 ? brow0 * p.meta_bytes : 0),
                                                 I4 ? (uint32_t)brows * p.meta_bytes : 0u);
    const __amdgpu_buffer_rsrc_t rsz = make_rsrc(F == kI4ZP ? p.zeros + brow0 * p.zbytes : p.W,
                                                 F == kI4ZP ? (uint32_t)brows * p.zbytes : 0u);
    const int nmeta = I4 ? brows * p.chunks : 0;
    struct Meta {
        uint32_t s[2], z;   // four 16-bit scales, four 4-bit zero points
    };
    auto meta_load = [&](int i) -> Meta {
        Meta m = {{0u, 0u}, 0x8888u};
        const uint32_t r = __umulhi((uint32_t)i, p.chunk_mul), c = (uint32_t)i - r * (uint32_t)p.chunks;
        const uint32_t so = i < nmeta ? r * p.meta_bytes + c * 8u : kOOB, zo = i < nmeta ? r * p.zbytes + c * 2u : kOOB;
        if (p.wide) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(rsm, so, 0u, 0);
            m.s[0] = v[0];
            m.s[1] = v[1];
            if constexpr (F == kI4ZP) m.z = ld_u16(rsz, zo, 0u);
        } else {   // scales and zero points wherever they lie; past the row's last group: another row's, never read
            m.s[0] = ld_u16(rsm, so, 0u) | ld_u16(rsm, so + 2u, 0u) << 16;
            m.s[1] = ld_u16(rsm, so + 4u, 0u) | ld_u16(rsm, so + 6u, 0u) << 16;
            if constexpr (F == kI4ZP) m.z = ld_u8(rsz, zo, 0u) | ld_u8(rsz, zo + 1u, 0u) << 8;
        }
        return m;
    };
    uint32_t* md = reinterpret_cast<uint32_t*>(smem);
    auto meta_put = [&](int i, const Meta& m) {
        const uint32_t r = __umulhi((uint32_t)i, p.chunk_mul), c = (uint32_t)i - r * (uint32_t)p.chunks;
        uint32_t* at = md + 4u * c * (uint32_t)p.mstride + r;
        uint32_t s[4];
        float up[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            s[g] = g & 1 ? m.s[g >> 1] & 0xFFFF0000u : m.s[g >> 1] << 16;
            up[g] = (F == kI4 ? f16_to_f32(s[g] >> 16) : __uint_as_float(s[g])) * kI4Up;
            at[(uint32_t)g * (uint32_t)p.mstride] =
                F == kI4 ? __float_as_uint(up[g]) : i4zp_word(up[g], (m.z >> (4 * g)) & 15u);
        }
        if constexpr (F == kI4ZP) {   // a branch hardly ever taken: chosen word by word it cost 0.07 us a launch more
            const float top = fmaxf(fmaxf(fabsf(up[0]), fabsf(up[1])), fmaxf(fabsf(up[2]), fabsf(up[3])));
            if (__builtin_expect(top > kF32Max, 0)) {
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    if (fabsf(up[g]) > kF32Max)
                        at[(uint32_t)g * (uint32_t)p.mstride] = i4zp_word_big(s[g], (m.z >> (4 * g)) & 15u);
            }
        }
    };
    Meta m0;
    if constexpr (I4) m0 = meta_load((int)threadIdx.x);

    // Epilogue operands of the tiles this wave stores: (unit, tile) number q = wave, wave + W, ...
    uint32_t ep_scale[kOuts], ep_bias[kOuts];
    int ep_row[kOuts];
#pragma unroll
    for (int e = 0; e < kOuts; ++e) {
        const int q = wave + e * W, qu = q / P, qt = q - qu * P;
        const int a0 = tile_at(u0 + qu), a1 = tile_at(u0 + qu + 1);
        const int row = q < kUnits * P && a0 + qt < a1 ? (a0 + qt) * kTileRows + ln : p.N;
        const uint32_t off = row < p.N ? (uint32_t)row : (kOOB >> 2);
        ep_row[e] = row;
        ep_scale[e] = 0u;
        if constexpr (F == kFP8)
            ep_scale[e] = __builtin_amdgcn_raw_buffer_load_b32(make_rsrc(p.meta, (uint32_t)p.N * 4u), off * 4u, 0u, 0);
        ep_bias[e] = ld_u16(make_rsrc(p.bias ? p.bias : p.x, p.bias ? (uint32_t)p.N * 2u : 0u), off * 2u, 0u);
    }
    __builtin_amdgcn_sched_barrier(0);

    // One descriptor per tile, bounded to its rows (the count through readfirstlane: in a VGPR it would wrap every load in
    // a waterfall loop). Columns past K (BF16 and FP8 rows need not fill a stage) are turned into out-of-range offsets,
    // x's too: both operands read zero there.
    __amdgpu_buffer_rsrc_t rw[P];
#pragma unroll
    for (int t = 0; t < P; ++t) {
        const int row0 = (t0 + t) * kTileRows;
        const uint32_t rows = (uint32_t)__builtin_amdgcn_readfirstlane(t < nt ? max(0, min(kTileRows, p.N - row0)) : 0);
        rw[t] = make_rsrc(p.W + (rows ? (size_t)row0 : 0) * p.row_bytes, rows * p.row_bytes);
    }
    const __amdgpu_buffer_rsrc_t xrs = make_rsrc(p.x, (uint32_t)p.M * (uint32_t)p.K * 2u);
    // RING: the row's first byte in its first line (lines counted from the tile's first byte, so that none starts before it;
    // 8 rows are a multiple of 128 bytes, so a row's is that of its lane group)
    const uint32_t ws = RING ? ((uint32_t)(lane / WP) * p.row_bytes) & 127u : 0u;
    const uint32_t lw = (uint32_t)(lane / WP) * p.row_bytes - ws + (uint32_t)(lane % WP) * 16u;
    const uint32_t lx = (uint32_t)(lane / XP) * (uint32_t)p.K * 2u + (uint32_t)(lane % XP) * 16u;
    const int cw = (lane % WP) * (C / WP), cx = (lane % XP) * 8;     // first column of the lane's 16 bytes
    const uint32_t wstep = (uint32_t)WR * p.row_bytes, xstep = (uint32_t)XR * (uint32_t)p.K * 2u;

    struct Stage {
        u32x4 w[P][L];
        u32x4 x[XL];
    };
    // Unconditional loads (a load under a branch makes the compiler wait for every outstanding one); t >= n: none in range.
    auto issue = [&](Stage& B, int t) {
        const int kb = stage_at(t);
        const int left = t < nl ? p.K - kb * C : 0;    // columns from the stage's first one on
        uint32_t wo;
        if constexpr (RING) {   // line kb + 1 of the rows; bytes past a row's end read zero
            const int wl = t < nl ? (int)p.row_bytes - (kb + 1) * RB : -RB;
            wo = (lane % WP) * 16 - (int)ws < wl ? lw + (uint32_t)(kb + 1) * (uint32_t)RB : kOOB;
        } else {
            wo = cw < left ? lw + (uint32_t)kb * (uint32_t)RB : kOOB;
        }
        const uint32_t xo = cx < left && (!RING || t > 0) ? lx + (uint32_t)kb * (uint32_t)(2 * C) : kOOB;
#pragma unroll
        for (int j = 0; j < XL; ++j) B.x[j] = ld16<0>(xrs, xo + xstep * (uint32_t)j, 0u);
#pragma unroll
        for (int t2 = 0; t2 < P; ++t2)
#pragma unroll
            for (int i = 0; i < L; ++i) B.w[t2][i] = ld16<AUX>(rw[t2], wo + wstep * (uint32_t)i, 0u);
    };
    Stage buf[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
        issue(buf[d], d);
        __builtin_amdgcn_sched_barrier(0);   // in stage order: the loop's waits count the loads behind a stage's
    }

    if constexpr (I4) {
        if ((int)threadIdx.x < nmeta) meta_put((int)threadIdx.x, m0);
        for (int i = (int)threadIdx.x + W * kWave; i < nmeta; i += W * kWave) meta_put(i, meta_load(i));
        __syncthreads();
    }

    unsigned char* lds = smem + p.wave_off + (uint32_t)wave * kWaveBytes;
    // 16-byte piece of a staged row: XORed with the row so that 8 rows' same piece lie in 8 different bank groups
    auto w_at = [](int row, int piece) -> uint32_t {
        return RB == 128 ? (uint32_t)(row * 128 + ((piece ^ (row & 7)) << 4))
                         : (uint32_t)(row * 64 + ((piece ^ ((row >> 1) & 3)) << 4));
    };
    auto x_at = [](int row, int piece) -> uint32_t { return (uint32_t)(row * 2 * C + ((piece ^ (row & 7)) << 4)); };
    // RING: 16 pieces a row, a line's in one half, turned back by the line's part before the row and on by the row: a stage's
    // piece then lies at a place that does not depend on the alignment, the 16 rows' in 16 different bank groups
    const uint32_t ring_put = (uint32_t)(lane % WP) + (uint32_t)(lane / WP) - (ws >> 4);
    auto put_w = [&](const Stage& B, int t2, int t) {
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const uint32_t at = RING ? (uint32_t)(i * WR + lane / WP) * 256u +
                                           (((ring_put + (uint32_t)(i * WR) + 8u * (uint32_t)(t & 1)) & 15u) << 4)
                                     : w_at(i * WR + lane / WP, lane % WP);
            *reinterpret_cast<u32x4*>(lds + kXBytes + (uint32_t)(t2 % kSlots) * kSlotBytes + at) = B.w[t2][i];
        }
    };
    auto get_w = [&](int t2, int i, int t) {
        const uint32_t at = RING ? (uint32_t)ln * 256u + (((uint32_t)(4 * i + lh + ln) + 8u * (uint32_t)((t + 1) & 1)) & 15u) * 16u
                                 : w_at(ln, 4 * i + lh);
        return *reinterpret_cast<const u32x4*>(lds + kXBytes + (uint32_t)(t2 % kSlots) * kSlotBytes + at);
    };
    const uint32_t one2 = (uint32_t)__builtin_amdgcn_readfirstlane((int)kI4Ones);
    const u32x4 ones = {one2, one2, one2, one2};
    auto mfma = [](const u32x4 a, const u32x4 b, const f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                       0, 0);
    };
    // INT4: this lane's metadata words. Rows past N and tiles past the unit's read words that nothing wrote; their sums are
    // meaningless, stay in their own D columns and are not stored.
    const uint32_t* mw = md + (I4 ? (t0 - bt0) * kTileRows + ln : 0);

    f32x4 acc[P];
#pragma unroll
    for (int t = 0; t < P; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    auto consume = [&](const Stage& B, int t) {
#pragma unroll
        for (int j = 0; j < XL; ++j) {
            u32x4 v = B.x[j];
            if constexpr (I4) v = i4_pair_x(v);   // to the nibbles' order
            if (XR <= MT || lane < MT * XP) *reinterpret_cast<u32x4*>(lds + x_at(j * XR + lane / XP, lane % XP)) = v;
        }
#pragma unroll
        for (int t2 = 0; t2 < kSlots; ++t2) put_w(B, t2, t);
        wave_lds_order();
        u32x4 a[X];
#pragma unroll
        for (int j = 0; j < X; ++j) {
            // the 8 columns of step j from lane group lh (step_col), as a piece of the staged row; lanes past MT repeat
            const int piece = F == kBF16 ? 4 * j + lh : (F == kFP8 ? 8 * (j >> 1) + 2 * lh + (j & 1) : 4 * lh + j);
            a[j] = *reinterpret_cast<const u32x4*>(lds + x_at(ln & (MT - 1), piece));
        }
        f32x4 xs = {0.0f, 0.0f, 0.0f, 0.0f};   // INT4: group sums of x for the D rows this lane holds
        if constexpr (I4) {
#pragma unroll
            for (int j = 0; j < X; ++j) xs = mfma(a[j], ones, xs);
        }
        const int kb = stage_at(t);
#pragma unroll
        for (int t2 = 0; t2 < P; ++t2) {
            u32x4 w[L];
            uint32_t m = 0u;   // INT4: read ahead of the weights, whose decode needs it
            if constexpr (I4) m = mw[(uint32_t)kb * (uint32_t)p.mstride + (uint32_t)(t2 * kTileRows)];
            if (t2 >= kSlots) wave_lds_order();
#pragma unroll
            for (int i = 0; i < L; ++i) w[i] = get_w(t2, i, t);
            if (t2 + kSlots < P) {
                wave_lds_order();
                put_w(B, t2 + kSlots, t);
            }
            if constexpr (F == kBF16) {
#pragma unroll
                for (int j = 0; j < X; ++j) acc[t2] = mfma(a[j], w[j], acc[t2]);
            } else if constexpr (F == kFP8) {
#pragma unroll
                for (int j = 0; j < X; ++j) {
                    const uint32_t d0 = (j & 1) ? w[j >> 1].z : w[j >> 1].x, d1 = (j & 1) ? w[j >> 1].w : w[j >> 1].y;
                    acc[t2] = mfma(a[j], u32x4{fp8x2_to_bf16x2<false>(d0), fp8x2_to_bf16x2<true>(d0),
                                               fp8x2_to_bf16x2<false>(d1), fp8x2_to_bf16x2<true>(d1)}, acc[t2]);
                }
            } else {
                const float f = __uint_as_float(F == kI4 ? kI4Exp << 23 : m << 15);   // bits 8..15 to the exponent
                f32x4 g = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < X; ++j) {
                    const uint32_t v = j == 0 ? w[0].x : (j == 1 ? w[0].y : (j == 2 ? w[0].z : w[0].w));
                    const uint32_t lo = v & 0x0F0F0F0Fu, hi = (v >> 4) & 0x0F0F0F0Fu;
                    g = mfma(a[j], u32x4{i4x2_to_bf16x2<false>(lo, f), i4x2_to_bf16x2<true>(lo, f),
                                         i4x2_to_bf16x2<false>(hi, f), i4x2_to_bf16x2<true>(hi, f)}, g);
                }
                const float s = __uint_as_float(F == kI4 ? m : m & 0xFFFF0000u);
                const float z = F == kI4 ? 8.0f : (float)(m & 0xFFu);
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[t2][v] = __builtin_fmaf(s, __builtin_fmaf(-z, xs[v], g[v]), acc[t2][v]);
            }
        }
        wave_lds_order();
    };

    // D stages are in flight throughout; a stage's buffer is refilled as soon as it is consumed. The last D stages are
    // consumed without a refill (a round of empty loads would queue behind the CU's outstanding ones).
    constexpr int kFirst = RING ? 1 : 0;   // the first line's buffer moves on at once
    if constexpr (RING) {
#pragma unroll
        for (int t2 = 0; t2 < P; ++t2) put_w(buf[0], t2, 0);
        wave_lds_order();
        issue(buf[0], D);
        __builtin_amdgcn_sched_barrier(0);
    }
    int t = kFirst;
    for (; t + D < nl; t += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            consume(buf[(d + kFirst) % D], t + d);   // t + d < nl: the loop's condition
            issue(buf[(d + kFirst) % D], t + d + D);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (t + d < nl) consume(buf[(d + kFirst) % D], t + d);

    // Partial tiles to the wave's own region, one barrier, then (unit, tile) q is added up in split order and stored.
#pragma unroll
    for (int t2 = 0; t2 < P; ++t2) *reinterpret_cast<f32x4*>(lds + t2 * 1024 + lane * 16) = acc[t2];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kOuts; ++e) {
        const int q = wave + e * W, qu = q / P, qt = q - qu * P;
        if (q >= kUnits * P || ep_row[e] >= p.N) continue;
        const unsigned char* part = smem + p.wave_off + (uint32_t)(qu * S) * kWaveBytes + qt * 1024 + lane * 16;
        f32x4 v = *reinterpret_cast<const f32x4*>(part);
#pragma unroll
        for (int s = 1; s < S; ++s) v += *reinterpret_cast<const f32x4*>(part + (uint32_t)s * kWaveBytes);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int m = 4 * lh + c;
            if (m >= p.M) continue;
            float o = v[c];
            if constexpr (I4) o = o * kI4Back;
            if constexpr (F == kFP8) o = o * __uint_as_float(ep_scale[e]);
            if (p.bias) o = o + bf16_to_f32(ep_bias[e]);
            p.y[(size_t)m * (size_t)p.N + (size_t)ep_row[e]] = (uint16_t)f32_to_bf16_out(o);
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------------------------

// A call the tile kernel does not take (shape, alignment, LDS, or a rule of the choice): nothing was launched.
constexpr int kTileRefused = -100;

// The launch on `st` with `blocks` blocks (raised to one per kUnits * P tiles). Returns 0, kTileRefused when the block's
// metadata does not fit the LDS, or a hipError_t.
template <int F, int P, int W, int S, int D, int MT, int AUX, bool IL, bool RING>
int launch_tile(const BatchParams& b, int blocks, hipStream_t st)
{
    constexpr int kUnits = W / S;
    TileParams p{};
    p.W = b.W;
    p.meta = static_cast<const uint8_t*>(b.meta);
    p.zeros = b.zeros;
    p.x = b.x;
    p.bias = b.bias;
    p.y = b.y;
    p.M = b.M;
    p.N = b.N;
    p.K = b.K;
    p.row_bytes = b.row_bytes;
    p.meta_bytes = b.meta_bytes;
    p.zbytes = b.zbytes;
    p.stages = (b.K + TileFmt<F>::kCols - 1) / TileFmt<F>::kCols;
    const int ntiles = (b.N + kTileRows - 1) / kTileRows;
    const int fewest = (ntiles + kUnits * P - 1) / (kUnits * P);
    if (blocks < fewest) blocks = fewest;
    p.tq = ntiles / (blocks * kUnits);
    p.tr = ntiles % (blocks * kUnits);
    uint64_t lds = 0;
    if (TileFmt<F>::kI4F) {
        const int G = b.K / kBlockCols;
        p.chunks = G > 8 ? (G + 3) / 4 : 2;   // at least two: chunk_mul is 32 bits
        p.chunk_mul = (uint32_t)(((1ull << 32) + p.chunks - 1) / p.chunks);
        // the last unit's first tile, and the P tiles a wave's reads span from there
        p.mstride = kTileRows * ((kUnits - 1) * (p.tq + (p.tr ? 1 : 0)) + P) + 1;
        p.wide = G % 4 == 0 && aligned(b.meta, 8) && (F != kI4ZP || aligned(b.zeros, 2));
        lds = ((uint64_t)p.chunks * 4u * (uint64_t)p.mstride * 4u + 127u) & ~127ull;
        if (lds > rows_max_lds()) return kTileRefused;
    }
    p.wave_off = (uint32_t)lds;
    lds += (uint64_t)W * tile_wave_bytes<F, P, MT, RING>();
    if (lds > rows_max_lds()) return kTileRefused;
    auto kernel = &gemv_tile_kernel<F, P, W, S, D, MT, AUX, IL, RING>;
    if (lds > kMaxLds) {   // beyond the default dynamic-LDS limit: raise it once per device for this kernel
        static std::atomic<uint64_t> raised{0};
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return (int)e;
        const uint64_t bit = 1ull << (dev & 63);
        if (!(raised.load(std::memory_order_relaxed) & bit)) {
            e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)rows_max_lds());
            if (e != hipSuccess) return (int)e;
            raised.fetch_or(bit, std::memory_order_relaxed);
        }
    }
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(W * kWave), (uint32_t)lds, st, p);
    return (int)hipGetLastError();
}

// The tile kernel's launch for a call whose variant is the library's choice, or kTileRefused (gemv_tile.hip). kind: 0
// BF16, 1 FP8, 2 INT4 reference format, 3 INT4 asymmetric; b as the small-batch entry point fills it.
int launch_tile_picked(int kind, const BatchParams& b, hipStream_t st);

}  // namespace paia

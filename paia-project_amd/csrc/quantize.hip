// On-device weight quantizers: the formats of src/paia_gemv/quant.py:8-31 and quant_host.h:74-106, produced on the
// GPU in one pass over W (fp32 [N][K], row-major). No reference C symbol: the reference quantizes with torch on the
// GPU; these are the same values from hand-written gfx950 kernels.
//
//   FP8 rowwise  scale[n] = amax_n / 448 (1 if the row is all zero); q = e4m3_rn(clamp(w / scale, +-448)), the gfx950 OCP
//                e4m3 convert (round to nearest even).
//   INT4 g128    s16 = f16_rn(amax_g / 7) (1 if the group is all zero); sf = float(s16) (1 if it underflowed to 0);
//                n = clamp(rint(w / sf), -7, 7) + 8, packed two per byte (weight 2j low nibble).
//   INT4 g128 asymmetric (no reference counterpart; the format of the BASELINE INT4 configs, dequant (q - z) * s):
//                lo = min(0, min w), hi = max(0, max w) over the group; s = bf16_rn((hi - lo) / 15) (1 if that is 0);
//                z = clamp(rint(-lo / s), 0, 15); q = clamp(rint(w / s) + z, 0, 15). Zero points are packed two
//                groups per byte along G.
// Quotients are correctly rounded, rint rounds half to even, as torch.round and std::nearbyint do.
//
// All three read 4 bytes and write 0.5 to 1 per weight: bound by HBM when W is read once, in 16-byte pieces, and the
// division does not fill the VALU.
//   FP8: the threads of a row keep it in registers between the maximum and the encoding (a wave for K <= 1024, up to 1024
//   threads for K <= 32768; beyond, the row is read twice). With rows read twice, the second time from L2, 4096x14336 took
//   88 us (512 KiB of rows per CU in flight is more than its share of L2) and 28672x4096 121; now 47 and 89 (6.6 TB/s).
//   The loads are non-temporal: a row's bytes are used once (plain: 56 and 105 us).
//   INT4: a group is 16 lanes of 8 weights, so its maximum takes four DPP steps, its scale one conversion per lane and
//   its codes leave as 4 bytes a lane; a wave holds 8 groups. With a group per wave (2 weights and 1 byte a lane)
//   28672x4096 took 147 us, asymmetric 195; now 96 both (5.5 TB/s; in turn with other kernels 149 and 200, now 102 and
//   96). Plain loads: a lane's two 16-byte loads share lines (non-temporal 99).
//   Calls of few weights take fewer of them a lane (kFewWeights).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemv_kernel.h"
#include "paia_gemv.h"

namespace paia {

__device__ __forceinline__ float wave_max(float v)
{
    v = fmaxf(v, dpp_f32<0xB1>(v));
    v = fmaxf(v, dpp_f32<0x4E>(v));
    v = fmaxf(v, dpp_f32<0x124>(v));
    v = fmaxf(v, dpp_f32<0x128>(v));
    const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
    const float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
    const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
    const float d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
    return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

// four fp32 -> four e4m3 codes (byte i = value i), round to nearest even; |v| <= 448 on entry
__device__ __forceinline__ uint32_t e4m3x4(float a, float b, float c, float d)
{
    int w = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false);
    w = __builtin_amdgcn_cvt_pk_fp8_f32(c, d, w, true);
    return (uint32_t)w;
}

// Correctly rounded v / s from y = 1/s (correctly rounded), five multiply-adds and a sign instead of the division's
// sequence with its own reciprocal: two residual corrections, the second of a quotient already within an ulp, which
// Markstein's theorem makes the correctly rounded one. Needs |s| within 2^-60..2^60, so that neither y nor a residual that
// matters leaves the normal range; quotients so small that a residual underflows round to zero in every format here.
__device__ __forceinline__ float div_by(float v, float s, float y)
{
    float q = v * y;
    q = __builtin_fmaf(__builtin_fmaf(-s, q, v), y, q);
    q = __builtin_fmaf(__builtin_fmaf(-s, q, v), y, q);
    return __builtin_copysignf(q, v);   // -0 / s
}
__device__ __forceinline__ bool div_by_ok(float s) { return s >= 0x1p-60f && s <= 0x1p60f; }

typedef float f32x4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4v ld4(const float* p) { return *reinterpret_cast<const f32x4v*>(p); }
__device__ __forceinline__ f32x4v ld4_nt(const float* p)
{
    return __builtin_nontemporal_load(reinterpret_cast<const f32x4v*>(p));
}

// ---- FP8: T threads per row, V float4 of the row per thread in registers (KEEP) or the row read again ----------------
template <int T, int V, bool KEEP>
__global__ void __launch_bounds__(T < 256 ? 256 : T) quantize_fp8_kernel(const float* __restrict__ W,
                                                                        uint8_t* __restrict__ q,
                                                                        float* __restrict__ scale, int N, int K)
{
    constexpr int kRows = T < 256 ? 256 / T : 1;   // rows per block
    __shared__ float red[T / kWave];
    const int tid = (int)threadIdx.x % T;
    const int n = (int)blockIdx.x * kRows + (int)threadIdx.x / T;
    if (kRows > 1 && n >= N) return;               // T = a wave: no barrier follows
    const float* row = W + (size_t)n * K;
    const int K4 = K / 4;
    f32x4v v[KEEP ? V : 1];
    float amax = 0.0f;
    auto take = [&](const f32x4v a) {
        amax = fmaxf(amax, fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))));
    };
    if constexpr (KEEP) {
#pragma unroll
        for (int e = 0; e < V; ++e) {
            v[e] = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};
            if (tid + e * T < K4) v[e] = ld4_nt(row + 4 * (tid + e * T));
        }
#pragma unroll
        for (int e = 0; e < V; ++e) take(v[e]);
    } else {
        for (int i = tid; i < K4; i += T) take(ld4(row + 4 * i));
    }
    amax = wave_max(amax);
    if constexpr (T > kWave) {
        if (lane_id() == 0) red[wave_id()] = amax;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < T / kWave; ++w) amax = fmaxf(amax, red[w]);
    }
    const float s = amax > 0.0f ? amax / 448.0f : 1.0f;
    if (tid == 0) scale[n] = s;
    uint32_t* qrow = reinterpret_cast<uint32_t*>(q + (size_t)n * K);
    constexpr bool kFew = KEEP && V == 1;          // four quotients: the reciprocal would only lengthen the chain
    const bool fast = !kFew && div_by_ok(s);
    const float y = kFew ? 0.0f : 1.0f / s;
    auto code = [&](const f32x4v a) -> uint32_t {
        auto c = [&](float w) {
            const float t = fast ? div_by(w, s, y) : w / s;
            return fminf(fmaxf(t, -448.0f), 448.0f);
        };
        return e4m3x4(c(a.x), c(a.y), c(a.z), c(a.w));
    };
    if constexpr (KEEP) {
#pragma unroll
        for (int e = 0; e < V; ++e)
            if (tid + e * T < K4) qrow[tid + e * T] = code(v[e]);
    } else {
        for (int i = tid; i < K4; i += T) qrow[i] = code(ld4(row + 4 * i));
    }
}

// ---- INT4: L lanes per group, `Steps` steps of 64 / L groups per wave -------------------------------------------------
// Many groups: 16 lanes of 8 weights, two steps. Few: the lanes' chain of quotients is the call's time, so 64 lanes of two
// weights (asymmetric 32 of four, a pair of groups per wave).
constexpr int kQBlock = 256;

__device__ __forceinline__ float row16_max(float v)   // over the 16 lanes of a DPP row, in every lane of it
{
    v = fmaxf(v, dpp_f32<0xB1>(v));
    v = fmaxf(v, dpp_f32<0x4E>(v));
    v = fmaxf(v, dpp_f32<0x124>(v));
    return fmaxf(v, dpp_f32<0x128>(v));
}
template <int L>
__device__ __forceinline__ float group_max(float v)
{
    if constexpr (L == 64) return wave_max(v);
    v = row16_max(v);
    if constexpr (L == 32) {
        const int b = __float_as_int(v);
        const float lo = fmaxf(v, __int_as_float(__builtin_amdgcn_readlane(b, 16)));   // rows 0, 1 (valid in row 0)
        const float hi = fmaxf(v, __int_as_float(__builtin_amdgcn_readlane(b, 48)));   // rows 2, 3 (valid in row 2)
        const int l = __builtin_amdgcn_readlane(__float_as_int(lo), 0), h = __builtin_amdgcn_readlane(__float_as_int(hi), 32);
        v = __int_as_float(lane_id() < 32 ? l : h);
    }
    return v;
}
template <int L>
struct GroupPart {
    float w[128 / L];
};
template <int L>
__device__ __forceinline__ GroupPart<L> group_load(const float* W, size_t gi, int l, bool ok)
{
    constexpr int n = 128 / L;
    GroupPart<L> g;
#pragma unroll
    for (int j = 0; j < n; ++j) g.w[j] = 0.0f;
    if (ok) {
        const float* p = W + gi * 128 + (size_t)(l * n);
        if constexpr (n == 2) {
            const float2 a = *reinterpret_cast<const float2*>(p);
            g.w[0] = a.x;
            g.w[1] = a.y;
        } else {
#pragma unroll
            for (int j = 0; j < n; j += 4) {
                const f32x4v a = ld4(p + j);
                g.w[j] = a.x;
                g.w[j + 1] = a.y;
                g.w[j + 2] = a.z;
                g.w[j + 3] = a.w;
            }
        }
    }
    return g;
}
// The codes of a lane as one word (weight j in nibble j).
template <bool ZP, int L>
__device__ __forceinline__ uint32_t group_codes(const GroupPart<L>& g, float s, float z)
{
    constexpr bool kFew = L > 16;   // few quotients: the reciprocal would only lengthen the chain
    const bool fast = !kFew && div_by_ok(s);
    const float y = kFew ? 0.0f : 1.0f / s;
    uint32_t word = 0;
#pragma unroll
    for (int j = 0; j < 128 / L; ++j) {
        const float t = __builtin_rintf(fast ? div_by(g.w[j], s, y) : g.w[j] / s);
        const int c = ZP ? (int)fminf(fmaxf(t + z, 0.0f), 15.0f) : (int)fminf(fmaxf(t, -7.0f), 7.0f) + 8;
        word |= (uint32_t)c << (4 * j);
    }
    return word;
}
template <int L>
__device__ __forceinline__ void group_store(uint8_t* packed, size_t gi, int l, uint32_t word)
{
    uint8_t* p = packed + gi * 64 + (size_t)(l * (64 / L));
    if constexpr (L == 16) *reinterpret_cast<uint32_t*>(p) = word;
    else if constexpr (L == 32) *reinterpret_cast<uint16_t*>(p) = (uint16_t)word;
    else *p = (uint8_t)word;
}

template <int L, int Steps>
__global__ void __launch_bounds__(kQBlock) quantize_int4_kernel(const float* __restrict__ W,
                                                                uint8_t* __restrict__ packed,
                                                                uint16_t* __restrict__ scales, size_t ngroups)
{
    constexpr int kPer = 64 / L;   // groups per wave and step
    const int lane = lane_id(), l = lane % L;
    const size_t g0 = ((size_t)blockIdx.x * (kQBlock / kWave) + (size_t)wave_id()) * (kPer * Steps) + (size_t)(lane / L);
    GroupPart<L> g[Steps];
#pragma unroll
    for (int e = 0; e < Steps; ++e) g[e] = group_load<L>(W, g0 + kPer * e, l, g0 + kPer * e < ngroups);
#pragma unroll
    for (int e = 0; e < Steps; ++e) {
        const size_t gi = g0 + kPer * e;
        float amax = 0.0f;
#pragma unroll
        for (int j = 0; j < 128 / L; ++j) amax = fmaxf(amax, fabsf(g[e].w[j]));
        amax = group_max<L>(amax);
        const _Float16 s16 = (_Float16)(amax > 0.0f ? amax / 7.0f : 1.0f);   // v_cvt_f16_f32: round to nearest even
        float sf = (float)s16;
        if (!(sf > 0.0f)) sf = 1.0f;
        const uint32_t word = group_codes<false, L>(g[e], sf, 0.0f);
        if (gi < ngroups) {
            group_store<L>(packed, gi, l, word);
            if (l == 0) scales[gi] = __builtin_bit_cast(uint16_t, s16);
        }
    }
}

// A pair of groups (2j, 2j+1 of a row) is 2 L lanes of a wave, so the packed zero-point byte has one writer: the second
// group's first lane, or the first's where G is odd (ODD) and the pair is the row's last.
template <bool ODD, int L, int Steps>
__global__ void __launch_bounds__(kQBlock) quantize_int4_zp_kernel(const float* __restrict__ W,
                                                                   uint8_t* __restrict__ packed,
                                                                   uint16_t* __restrict__ scales,
                                                                   uint8_t* __restrict__ zeros, uint32_t npairs, int G)
{
    static_assert(L == 16 || L == 32, "a pair within a wave");
    constexpr int kPer = 32 / L;   // pairs per wave and step
    const int lane = lane_id(), l = lane % L, h = (lane / L) & 1;
    const uint32_t p0 = (blockIdx.x * (kQBlock / kWave) + (uint32_t)wave_id()) * (kPer * Steps) + (uint32_t)(lane / (2 * L));
    const uint32_t ZB = (uint32_t)(G + 1) / 2;
    GroupPart<L> g[Steps];
    size_t gis[Steps];
    bool ok[Steps], alone[Steps];
#pragma unroll
    for (int e = 0; e < Steps; ++e) {
        const uint32_t pi = p0 + kPer * e;
        alone[e] = false;
        ok[e] = pi < npairs;
        if constexpr (ODD) {
            const uint32_t n = pi / ZB, j = pi - n * ZB;
            alone[e] = 2 * j + 1 >= (uint32_t)G;
            ok[e] = ok[e] && !(alone[e] && h);
            gis[e] = (size_t)n * (size_t)G + 2 * j + (uint32_t)h;
        } else {
            gis[e] = 2 * (size_t)pi + (size_t)h;
        }
        g[e] = group_load<L>(W, gis[e], l, ok[e]);
    }
#pragma unroll
    for (int e = 0; e < Steps; ++e) {
        float lo = g[e].w[0], hi = g[e].w[0];
#pragma unroll
        for (int j = 1; j < 128 / L; ++j) {
            lo = fminf(lo, g[e].w[j]);
            hi = fmaxf(hi, g[e].w[j]);
        }
        lo = fminf(-group_max<L>(-lo), 0.0f);
        hi = fmaxf(group_max<L>(hi), 0.0f);
        const float r = (hi - lo) / 15.0f;
        uint32_t sb = f32_to_bf16_rne(r);
        float s = bf16_to_f32(sb);
        if (!(s > 0.0f)) {
            sb = 0x3F80u;                              // bf16 1.0
            s = 1.0f;
        }
        const float zf = fminf(fmaxf(__builtin_rintf(-lo / s), 0.0f), 15.0f);
        const uint32_t word = group_codes<true, L>(g[e], s, zf);
        // the first group's zero point to the second's lanes (L = 16: row_bcast:15 into rows 1 and 3)
        const uint32_t z = (uint32_t)zf;
        const uint32_t zfirst = L == 16 ? (uint32_t)__builtin_amdgcn_update_dpp(0, (int)z, 0x142, 0xA, 0xF, false)
                                        : (uint32_t)__builtin_amdgcn_readlane((int)z, 0);
        if (ok[e]) {
            group_store<L>(packed, gis[e], l, word);
            if (l == 0) {
                scales[gis[e]] = (uint16_t)sb;
                if (h) zeros[p0 + kPer * e] = (uint8_t)(zfirst | (z << 4));
                else if (alone[e]) zeros[p0 + kPer * e] = (uint8_t)z;
            }
        }
    }
}

}  // namespace paia

namespace {
using namespace paia;

// A launch has less than 2^32 threads: rows beyond kMaxBlocks blocks of 256 go into a further launch (no call on weights
// below 4 GB needs a second).
constexpr size_t kMaxBlocks = (size_t)1 << 23;

unsigned blocks_for(size_t units, size_t per_block) { return (unsigned)((units + per_block - 1) / per_block); }
size_t slice_rows(size_t units_per_row, size_t units_per_block)
{
    const size_t r = kMaxBlocks * units_per_block / units_per_row;
    return r > 0 ? r : 1;
}

template <int T, int V, bool KEEP>
int launch_fp8(const void* W, void* q, void* scale, int N, int K, hipStream_t st)
{
    constexpr int kRows = T < 256 ? 256 / T : 1;
    const size_t step = slice_rows(T < 256 ? 1 : T / 256, kRows);
    for (size_t n = 0; n < (size_t)N; n += step) {
        const size_t rows = (size_t)N - n < step ? (size_t)N - n : step;
        hipLaunchKernelGGL((quantize_fp8_kernel<T, V, KEEP>), dim3(blocks_for(rows, kRows)), dim3(T < 256 ? 256 : T), 0, st,
                           static_cast<const float*>(W) + n * (size_t)K, static_cast<uint8_t*>(q) + n * (size_t)K,
                           static_cast<float*>(scale) + n, (int)rows, K);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return (int)e;
    }
    return 0;
}

template <int L, int Steps>
int launch_int4(const void* W, void* packed, void* scales, int N, int K, hipStream_t st)
{
    const size_t G = (size_t)K / 128;
    constexpr size_t kPerBlock = kQBlock / kWave * (64 / L) * Steps;
    const size_t step = slice_rows(G, kPerBlock);
    for (size_t n = 0; n < (size_t)N; n += step) {
        const size_t ngroups = ((size_t)N - n < step ? (size_t)N - n : step) * G;
        hipLaunchKernelGGL((quantize_int4_kernel<L, Steps>), dim3(blocks_for(ngroups, kPerBlock)), dim3(kQBlock), 0, st,
                           static_cast<const float*>(W) + n * (size_t)K, static_cast<uint8_t*>(packed) + n * (size_t)(K / 2),
                           static_cast<uint16_t*>(scales) + n * G, ngroups);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return (int)e;
    }
    return 0;
}

template <int L, int Steps>
int launch_int4_zp(const void* W, void* packed, void* scales, void* zeros, int N, int K, hipStream_t st)
{
    const size_t G = (size_t)K / 128, ZB = (G + 1) / 2;
    constexpr size_t kPerBlock = kQBlock / kWave * (32 / L) * Steps;
    const size_t step = slice_rows(ZB, kPerBlock);
    for (size_t n = 0; n < (size_t)N; n += step) {
        const size_t pairs = ((size_t)N - n < step ? (size_t)N - n : step) * ZB;
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(blocks_for(pairs, kPerBlock)), dim3(kQBlock), 0, st,
                               static_cast<const float*>(W) + n * (size_t)K, static_cast<uint8_t*>(packed) + n * (size_t)(K / 2),
                               static_cast<uint16_t*>(scales) + n * G, static_cast<uint8_t*>(zeros) + n * ZB, (uint32_t)pairs,
                               (int)G);
        };
        if (G & 1) launch(quantize_int4_zp_kernel<true, L, Steps>);
        else launch(quantize_int4_zp_kernel<false, L, Steps>);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return (int)e;
    }
    return 0;
}

// Up to this many weights the forms with fewer weights a lane are ahead (us, few / many): FP8 rows of at most 1024, a block
// against a wave each, 36x800 2.0 / 2.9, 653x976 3.0 / 3.2, 1057x672 even, 2765x1024 6.3 / 5.1; INT4 163x768 1.9 / 2.9,
// 0.9 to 1.2 million weights 3.25 / 3.42, 1.75 to 2.2 million 5.5 / 4.7; asymmetric 67x1408 2.1 / 3.1, 0.55 to 0.93 million
// 3.2 / 3.5, 1.1 to 1.8 million even.
constexpr int64_t kFewWeights = 1 << 20;
bool few(int N, int K) { return (int64_t)N * K <= kFewWeights; }

}  // namespace

extern "C" {

int paia_quantize_fp8_rowwise(const void* W, void* q, void* scale, int N, int K, void* stream)
{
    if (N <= 0 || K <= 0 || (K & 15) || !aligned(W, 16) || !aligned(q, 16) || !aligned(scale, 4)) return -2;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    // The fewest threads that hold the row with up to 8 float4 (32 registers) each, so that rows in flight fill the chip
    // between a row's two halves; a block for 1024 < K <= 2048, where a wave with 8 left few-row calls longer in flight
    // (513x1040 3.5 us against 3.1).
    if (K <= 256 * 4 && few(N, K)) return launch_fp8<256, 1, true>(W, q, scale, N, K, st);
    if (K <= 64 * 4 * 4) return launch_fp8<64, 4, true>(W, q, scale, N, K, st);
    if (K <= 256 * 4 * 2) return launch_fp8<256, 2, true>(W, q, scale, N, K, st);
    if (K <= 256 * 4 * 4) return launch_fp8<256, 4, true>(W, q, scale, N, K, st);
    if (K <= 256 * 4 * 8) return launch_fp8<256, 8, true>(W, q, scale, N, K, st);
    if (K <= 512 * 4 * 8) return launch_fp8<512, 8, true>(W, q, scale, N, K, st);
    if (K <= 1024 * 4 * 8) return launch_fp8<1024, 8, true>(W, q, scale, N, K, st);
    return launch_fp8<1024, 1, false>(W, q, scale, N, K, st);
}

int paia_quantize_int4_g128(const void* W, void* packed, void* scales, int N, int K, void* stream)
{
    if (N <= 0 || K <= 0 || (K & 127) || !aligned(W, 16) || !aligned(packed, 16) || !aligned(scales, 2)) return -2;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    return few(N, K) ? launch_int4<64, 1>(W, packed, scales, N, K, st) : launch_int4<16, 2>(W, packed, scales, N, K, st);
}

int paia_quantize_int4_zp_g128(const void* W, void* packed, void* scales, void* zeros, int N, int K, void* stream)
{
    if (N <= 0 || K <= 0 || (K & 127) || !aligned(W, 16) || !aligned(packed, 16) || !aligned(scales, 2) ||
        zeros == nullptr)
        return -2;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    return few(N, K) ? launch_int4_zp<32, 1>(W, packed, scales, zeros, N, K, st)
                     : launch_int4_zp<16, 2>(W, packed, scales, zeros, N, K, st);
}

}  // extern "C"

// Dequantisation to fp32 [N][K] -- the bit-exact definitions the fused kernels compute in registers.
// No reference C symbol: the reference dequantises with torch (src/paia_gemv/quant.py:16-17,34-38) and on the host
// (quant_host.h:82-85,106-111). These kernels give the same values on the GPU:
//   FP8      out = float(e4m3(q)) * scale[n]            one fp32 product (round to nearest even)
//   INT4     out = (n - 8) * float(s_fp16)              exact in fp32
//   INT4ZP   out = (q - z) * float(s_bf16)              exact in fp32
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemv_kernel.h"
#include "paia_gemv.h"

namespace paia {

// Bound by the fp32 stores (4 bytes a weight against 0.5 to 1 read): a lane takes 4 neighbouring weights, so a wave's
// store is 1 KiB in a row and every line leaves whole. With 16 or 32 weights a lane, four or eight stores each touched a
// quarter or an eighth of 64 lines. 28672x4096 launched again and again (the codes then come from the Infinity Cache):
// FP8 169 us, INT4 168, INT4ZP 156; now 83, 74 and 72. In turn with other kernels, codes from HBM: 160, 163 and 159; now
// 96, 114 and 116. The stores are non-temporal (each byte is written once and nothing here reads it back). A block takes
// 4096 columns of a row (1024 in calls of few weights, where four steps a lane and a quarter of the blocks cost 0.3 to
// 1.3 us), or for short rows as many whole rows as fit; `mul` = ceil(2^32 / K) then divides a weight's index in the
// block by K (index * K < 2^32).
constexpr int kDqThreads = 256;
constexpr int dq_block(int steps) { return kDqThreads * 4 * steps; }   // weights per block

// Row and column of the lane's 4 weights in step e of kDqSteps; false past the end of the row (long rows, mul = 0: `rows` is
// the blocks per row) or of the rows (short ones).
template <int kDqSteps>
__device__ __forceinline__ bool dq_at(int e, int N, int K, int rows, uint32_t mul, size_t& row, int& col)
{
    const uint32_t u = (uint32_t)(e * kDqThreads + (int)threadIdx.x) * 4u;
    if (mul == 0) {
        const uint32_t r = blockIdx.x / (uint32_t)rows;
        row = r;
        col = (int)((blockIdx.x - r * (uint32_t)rows) * (uint32_t)dq_block(kDqSteps) + u);
        return col < K;
    }
    const uint32_t r = __umulhi(u, mul);
    row = (size_t)blockIdx.x * (size_t)rows + r;
    col = (int)(u - r * (uint32_t)K);
    return (int)r < rows && row < (size_t)N;
}

typedef float f32x4o __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void st_nt(float* p, f32x4o v)
{
    __builtin_nontemporal_store(v, reinterpret_cast<f32x4o*>(p));
}

template <int kDqSteps>
__global__ void __launch_bounds__(kDqThreads) dequant_fp8_kernel(const uint8_t* __restrict__ Wq,
                                                                 const float* __restrict__ scale,
                                                                 float* __restrict__ out, int N, int K, int rows,
                                                                 uint32_t mul)
{
    uint32_t w[kDqSteps];
    float s[kDqSteps];
    size_t at[kDqSteps];
    bool ok[kDqSteps];
#pragma unroll
    for (int e = 0; e < kDqSteps; ++e) {
        size_t row;
        int col;
        ok[e] = dq_at<kDqSteps>(e, N, K, rows, mul, row, col);
        at[e] = row * (size_t)K + (size_t)col;
        w[e] = ok[e] ? *reinterpret_cast<const uint32_t*>(Wq + at[e]) : 0u;
        s[e] = ok[e] ? scale[row] : 0.0f;
    }
#pragma unroll
    for (int e = 0; e < kDqSteps; ++e) {
        const auto lo = __builtin_amdgcn_cvt_pk_f32_fp8(w[e], false);
        const auto hi = __builtin_amdgcn_cvt_pk_f32_fp8(w[e], true);
        if (ok[e]) st_nt(out + at[e], f32x4o{lo[0] * s[e], lo[1] * s[e], hi[0] * s[e], hi[1] * s[e]});
    }
}

// ZP: asymmetric format (bf16 scale, 4-bit zero), else the reference format (fp16 scale, zero 8).
template <bool ZP, int kDqSteps>
__global__ void __launch_bounds__(kDqThreads) dequant_int4_kernel(const uint8_t* __restrict__ Wq,
                                                                  const uint16_t* __restrict__ scales,
                                                                  const uint8_t* __restrict__ zeros,
                                                                  float* __restrict__ out, int N, int K, int rows,
                                                                  uint32_t mul)
{
    const int G = K / 128, ZB = (G + 1) / 2;
    uint32_t w[kDqSteps], sb[kDqSteps], zb[kDqSteps];
    size_t at[kDqSteps];
    int grp[kDqSteps];
    bool ok[kDqSteps];
#pragma unroll
    for (int e = 0; e < kDqSteps; ++e) {
        size_t row;
        int col;
        ok[e] = dq_at<kDqSteps>(e, N, K, rows, mul, row, col);
        at[e] = row * (size_t)K + (size_t)col;
        grp[e] = col >> 7;
        w[e] = ok[e] ? *reinterpret_cast<const uint16_t*>(Wq + at[e] / 2) : 0u;
        sb[e] = ok[e] ? scales[row * (size_t)G + (size_t)grp[e]] : 0u;
        zb[e] = ZP && ok[e] ? zeros[row * (size_t)ZB + (size_t)(grp[e] >> 1)] : 0u;
    }
#pragma unroll
    for (int e = 0; e < kDqSteps; ++e) {
        const float s = ZP ? bf16_to_f32(sb[e]) : f16_to_f32(sb[e]);
        const float z = ZP ? (float)((zb[e] >> ((grp[e] & 1) * 4)) & 0xFu) : 8.0f;
        f32x4o v;
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = ((float)((w[e] >> (4 * t)) & 0xFu) - z) * s;
        if (ok[e]) st_nt(out + at[e], v);
    }
}

}  // namespace paia

namespace {
using namespace paia;

// A launch has less than 2^32 threads: rows beyond kMaxBlocks blocks go into a further launch (outputs above 64 GB).
constexpr size_t kMaxBlocks = (size_t)1 << 23;

// Up to these many weights a lane's one step in four times the blocks is ahead (us, one step / four): FP8 54x4688 1.9 / 2.8,
// 0.66 to 0.97 million weights 2.4 / 2.9, 1.4 to 2.1 million 3.2 / 3.3 (0.85 to 1.21), beyond behind; INT4 44x3328 1.85 /
// 3.2, 1.2 to 1.7 million 3.3 / 4.1, above 1.75 million 0.93 to 1.37.
constexpr int64_t kDqFewFp8 = 1 << 20, kDqFewInt4 = 3 << 19;

struct DqPlan {
    size_t step;       // rows per launch
    int rows;          // rows per block (mul != 0) or blocks per row
    uint32_t mul;
    unsigned blocks(size_t n) const { return (unsigned)(mul ? (n + (size_t)rows - 1) / (size_t)rows : n * (size_t)rows); }
};
DqPlan dq_plan(int K, int steps)
{
    const int block = dq_block(steps);
    if (K <= block / 2) {
        const int rows = block / K;
        return {kMaxBlocks * (size_t)rows, rows, (uint32_t)(((1ull << 32) + (unsigned)K - 1) / (unsigned)K)};
    }
    const int per_row = (int)(((size_t)K + block - 1) / block);   // at most 2^21
    return {kMaxBlocks / (size_t)per_row, per_row, 0u};
}

template <int Steps>
int dequant_fp8(const void* Wq, const void* scale, void* out, int N, int K, hipStream_t st)
{
    const DqPlan p = dq_plan(K, Steps);
    for (size_t n = 0; n < (size_t)N; n += p.step) {
        const size_t m = (size_t)N - n < p.step ? (size_t)N - n : p.step;
        hipLaunchKernelGGL(dequant_fp8_kernel<Steps>, dim3(p.blocks(m)), dim3(kDqThreads), 0, st,
                           static_cast<const uint8_t*>(Wq) + n * (size_t)K, static_cast<const float*>(scale) + n,
                           static_cast<float*>(out) + n * (size_t)K, (int)m, K, p.rows, p.mul);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return (int)e;
    }
    return 0;
}

template <bool ZP, int Steps>
int dequant_int4(const void* Wq, const void* scales, const void* zeros, void* out, int N, int K, hipStream_t st)
{
    const DqPlan p = dq_plan(K, Steps);
    const size_t G = (size_t)K / 128, ZB = (G + 1) / 2;
    for (size_t n = 0; n < (size_t)N; n += p.step) {
        const size_t m = (size_t)N - n < p.step ? (size_t)N - n : p.step;
        hipLaunchKernelGGL((dequant_int4_kernel<ZP, Steps>), dim3(p.blocks(m)), dim3(kDqThreads), 0, st,
                           static_cast<const uint8_t*>(Wq) + n * (size_t)(K / 2),
                           static_cast<const uint16_t*>(scales) + n * G,
                           ZP ? static_cast<const uint8_t*>(zeros) + n * ZB : nullptr,
                           static_cast<float*>(out) + n * (size_t)K, (int)m, K, p.rows, p.mul);
        if (const hipError_t e = hipGetLastError(); e != hipSuccess) return (int)e;
    }
    return 0;
}

}  // namespace

extern "C" {

// Wq [N][K] e4m3 bytes, scale [N] fp32 -> out [N][K] fp32. K % 16 == 0; Wq, out 16 B aligned; scale 4 B aligned.
int paia_dequant_fp8(const void* Wq, const void* scale, void* out, int N, int K, void* stream)
{
    if (N <= 0 || K <= 0 || (K & 15) || !aligned(Wq, 16) || !aligned(out, 16) || !aligned(scale, 4)) return -2;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    return (int64_t)N * K <= kDqFewFp8 ? dequant_fp8<1>(Wq, scale, out, N, K, st)
                                       : dequant_fp8<4>(Wq, scale, out, N, K, st);
}

// Reference INT4: Wq [N][K/2], scales fp16 [N][K/128] -> out [N][K] fp32. K % 128 == 0.
int paia_dequant_int4(const void* Wq, const void* scales, void* out, int N, int K, void* stream)
{
    if (N <= 0 || K <= 0 || (K & 127) || !aligned(Wq, 16) || !aligned(out, 16) || !aligned(scales, 2)) return -2;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    return (int64_t)N * K <= kDqFewInt4 ? dequant_int4<false, 1>(Wq, scales, nullptr, out, N, K, st)
                                       : dequant_int4<false, 4>(Wq, scales, nullptr, out, N, K, st);
}

// Asymmetric INT4: Wq [N][K/2], scales bf16 [N][G], zeros [N][ceil(G/2)] -> out [N][K] fp32. K % 128 == 0.
int paia_dequant_int4_zp(const void* Wq, const void* scales, const void* zeros, void* out, int N, int K, void* stream)
{
    if (N <= 0 || K <= 0 || (K & 127) || !aligned(Wq, 16) || !aligned(out, 16) || !aligned(scales, 2) ||
        zeros == nullptr)
        return -2;
    const hipStream_t st = static_cast<hipStream_t>(stream);
    return (int64_t)N * K <= kDqFewInt4 ? dequant_int4<true, 1>(Wq, scales, zeros, out, N, K, st)
                                       : dequant_int4<true, 4>(Wq, scales, zeros, out, N, K, st);
}

}  // extern "C"

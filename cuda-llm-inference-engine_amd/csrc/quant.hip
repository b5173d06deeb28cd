// quant.hip — per-row symmetric FP32 -> INT8 quantizer for gfx950.
//
// Semantics follow kernels/quantization/14_int8_gemm.cu:10-60 of the
// reference bit for bit: row_max = max|x|, scale = row_max/127 (1 for an
// all-zero row), q = clamp(rint(x * (1/scale)), -128, 127), four q packed
// little-endian per int32 word.  Division is IEEE (correctly rounded) and
// rint is round-half-to-even, as on the reference's device.
//
// Layout on MI355X: the row is read once and kept in registers.
//   * cols <= 1024: one wave per row (four rows per 256-thread workgroup);
//     lane l holds the row's float4s l, l + 64, ... and the row max is a
//     wave reduction (no LDS, no barrier);
//   * cols <= 4096: one 256-thread workgroup per row, up to four float4s per
//     lane, the four wave maxima combined through LDS;
//   * cols <= 16384: 512 threads per row, four or eight float4s per lane
//     (two passes by 256 threads before: 1 / 16 x 8192 4.39 / 4.70 -> 2.63 /
//     2.91 us, 8192 x 8192 91.0 -> 52.9 us, 335 MB at 6.3 TB/s; 256 threads
//     with eight 2.80 / 3.08 / 61.3, 1024 with two 2.70 / 2.95 / 57.9);
//   * wider rows: a 256-thread workgroup walks the row twice (max, then
//     quantize; the second pass hits L2).
// Inputs past half of the 256 MiB MALL are read non-temporally (8192 x 8192:
// 61.1 -> 52.9 us; level or slower below: 2048 x 3072 6.95 against 7.26).
// Every form issues its loads unconditionally with the index clamped into the
// row, so they all go out before the first wait; a clamped duplicate cannot
// change the max, and only in-row words are stored.  The max is exact in any
// order, so all forms give the same bits.
#include "device_util.h"
#include "ie_internal.h"

namespace ie {
namespace {

__device__ __forceinline__ float abs_max4(float4 v) {
    return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
}

// cols <= 64 NV * 4: one wave per row, NV float4s per lane.
template <int NV>
__global__ __launch_bounds__(256) void quantize_rows_wave_kernel(int rows, int cols, const float* __restrict__ in,
                                                                 int32_t* __restrict__ out,
                                                                 float* __restrict__ scales) {
    const int lane = threadIdx.x & 63;
    const int row = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (row >= rows) return;
    const int n4 = cols >> 2;
    const float4* x = reinterpret_cast<const float4*>(in + (size_t)row * cols);
    float4 v[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = x[min(lane + 64 * j, n4 - 1)];
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j) m = fmaxf(m, abs_max4(v[j]));
    m = wave_max(m);
    const float scale = quant_scale(m);
    const float inv = 1.0f / scale;
    if (lane == 0) scales[row] = scale;
    int32_t* o = out + (size_t)row * n4;
#pragma unroll
    for (int j = 0; j < NV; ++j)
        if (lane + 64 * j < n4) o[lane + 64 * j] = quant_word(v[j], inv);
}

// Maximum of the T / 64 waves' m through LDS (every thread gets it).
template <int T>
__device__ __forceinline__ float block_max(float m) {
    __shared__ float wmax[T / 64];
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
    __syncthreads();
    m = wmax[0];
#pragma unroll
    for (int w = 1; w < T / 64; ++w) m = fmaxf(m, wmax[w]);
    return m;
}

template <bool NT>
__device__ __forceinline__ float4 load4(const float4* p) {
    if constexpr (NT) {
        typedef float f32x4 __attribute__((ext_vector_type(4)));
        const f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
        return make_float4(v.x, v.y, v.z, v.w);
    } else {
        return *p;
    }
}

// cols <= T NV * 4: one T-thread workgroup per row, NV float4s per thread.
template <int T, int NV, bool NT = false>
__global__ __launch_bounds__(T) void quantize_rows_reg_kernel(int cols, const float* __restrict__ in,
                                                                int32_t* __restrict__ out,
                                                                float* __restrict__ scales) {
    const int row = blockIdx.x;
    const int n4 = cols >> 2;
    const float4* x = reinterpret_cast<const float4*>(in + (size_t)row * cols);
    float4 v[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = load4<NT>(x + min((int)threadIdx.x + T * j, n4 - 1));
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j) m = fmaxf(m, abs_max4(v[j]));
    m = block_max<T>(m);
    const float scale = quant_scale(m);
    const float inv = 1.0f / scale;
    if (threadIdx.x == 0) scales[row] = scale;
    int32_t* o = out + (size_t)row * n4;
#pragma unroll
    for (int j = 0; j < NV; ++j)
        if ((int)threadIdx.x + T * j < n4) o[threadIdx.x + T * j] = quant_word(v[j], inv);
}

// Any cols: one workgroup per row, two passes.
__global__ __launch_bounds__(256) void quantize_rows_kernel(
    int cols, const float* __restrict__ in, int32_t* __restrict__ out,
    float* __restrict__ scales) {
    const int row = blockIdx.x;
    const int n4 = cols >> 2;
    const float4* x = reinterpret_cast<const float4*>(in + (size_t)row * cols);

    float m = 0.0f;
    for (int i = threadIdx.x; i < n4; i += 256) m = fmaxf(m, abs_max4(x[i]));
    m = block_max<256>(m);

    const float scale = quant_scale(m);
    const float inv = 1.0f / scale;
    if (threadIdx.x == 0) scales[row] = scale;

    int32_t* o = out + (size_t)row * n4;
    for (int i = threadIdx.x; i < n4; i += 256) {
        o[i] = quant_word(x[i], inv);
    }
}

constexpr size_t kStreamInputBytes = 128ull << 20;

}  // namespace

void launch_quantize(int rows, int cols, const float* in, int32_t* packed,
                     float* scales, hipStream_t s) {
    if (rows == 0) return;
    if (cols == 0) {
        // every row is all-zero: scale 1, nothing packed
        quantize_rows_kernel<<<rows, 256, 0, s>>>(cols, in, packed, scales);
        return;
    }
    const int n4 = cols >> 2;
    const unsigned wblocks = (unsigned)((rows + 3) / 4);
    if (n4 <= 64)
        quantize_rows_wave_kernel<1><<<wblocks, 256, 0, s>>>(rows, cols, in, packed, scales);
    else if (n4 <= 128)
        quantize_rows_wave_kernel<2><<<wblocks, 256, 0, s>>>(rows, cols, in, packed, scales);
    else if (n4 <= 192)
        quantize_rows_wave_kernel<3><<<wblocks, 256, 0, s>>>(rows, cols, in, packed, scales);
    else if (n4 <= 256)
        quantize_rows_wave_kernel<4><<<wblocks, 256, 0, s>>>(rows, cols, in, packed, scales);
    else if (n4 <= 512)
        quantize_rows_reg_kernel<256, 2><<<rows, 256, 0, s>>>(cols, in, packed, scales);
    else if (n4 <= 768)
        quantize_rows_reg_kernel<256, 3><<<rows, 256, 0, s>>>(cols, in, packed, scales);
    else if (n4 <= 1024)
        quantize_rows_reg_kernel<256, 4><<<rows, 256, 0, s>>>(cols, in, packed, scales);
    else if (n4 <= 4096) {
        const bool nt = (size_t)rows * cols * sizeof(float) >= kStreamInputBytes;
        auto* k = n4 <= 2048 ? (nt ? quantize_rows_reg_kernel<512, 4, true> : quantize_rows_reg_kernel<512, 4>)
                             : (nt ? quantize_rows_reg_kernel<512, 8, true> : quantize_rows_reg_kernel<512, 8>);
        k<<<rows, 512, 0, s>>>(cols, in, packed, scales);
    } else
        quantize_rows_kernel<<<rows, 256, 0, s>>>(cols, in, packed, scales);
}

}  // namespace ie

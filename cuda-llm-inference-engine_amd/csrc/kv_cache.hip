// kv_cache.hip — paged KV-cache writes.
//
// Layout (src/gpt2_engine.cu:321-346 of the reference): cache
// [num_phys_blocks][block_size][n_heads][d_head]; logical position pos of a
// sequence lives in physical block block_table[pos / block_size] at slot
// pos % block_size.  bf16 caches store round-to-nearest-even bfloat16.
#include <algorithm>
#include <type_traits>

#include "device_util.h"
#include "ie_internal.h"

namespace ie {
namespace {

template <typename KV>
__device__ __forceinline__ KV cvt(float x);
template <>
__device__ __forceinline__ float cvt<float>(float x) { return x; }
template <>
__device__ __forceinline__ uint16_t cvt<uint16_t>(float x) { return f32_to_bf16_rne(x); }

template <typename KV>
__global__ __launch_bounds__(256) void kv_write_kernel(const float* __restrict__ K,
                                                       const float* __restrict__ V,
                                                       KV* __restrict__ kc, KV* __restrict__ vc,
                                                       const int* __restrict__ bt, int seq_len,
                                                       int start_pos, int H, int dh, int bs) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t row = (size_t)H * dh;
    if (idx >= (size_t)seq_len * row) return;
    const int t = (int)(idx / row);
    const size_t rem = idx - (size_t)t * row;
    const int pos = start_pos + t;
    const int blk = pos / bs;
    const size_t dst = ((size_t)bt[blk] * bs + (pos - blk * bs)) * row + rem;
    kc[dst] = cvt<KV>(K[idx]);
    vc[dst] = cvt<KV>(V[idx]);
}

// Rows of n4 float4s: one workgroup per token (x) and 256 float4s (y), so the
// page is looked up once per workgroup and a thread moves 16 bytes of K and of
// V.  Against one element per thread (two integer divisions each): 512 x 768
// 3.16 -> 2.81 us (bf16 cache 3.15 -> 2.73), 1024 x 2048 bf16 7.27 -> 4.50 us.
// NARROW: rows of at most 64, 256 / blockDim.x tokens to a workgroup (with one
// each most threads idled: 10660 tokens of 64 4.82 -> 3.48 us, 7070 of 4 4.04 -> 2.37).
template <typename KV, bool NARROW>
__global__ __launch_bounds__(256) void kv_write_vec_kernel(const float4* __restrict__ K, const float4* __restrict__ V,
                                                           KV* __restrict__ kc, KV* __restrict__ vc,
                                                           const int* __restrict__ bt, int seq_len, int start_pos,
                                                           int n4, int bs) {
    const int j = NARROW ? threadIdx.x : blockIdx.y * 256 + threadIdx.x;
    const unsigned t = NARROW ? blockIdx.x * blockDim.y + threadIdx.y : blockIdx.x;
    if (j >= n4 || (NARROW && t >= (unsigned)seq_len)) return;
    const size_t src = (size_t)t * n4 + j;
    const float4 k = K[src], v = V[src];
    const int pos = start_pos + (int)t, blk = pos / bs;
    const size_t dst = ((size_t)bt[blk] * bs + (pos - blk * bs)) * n4 + j;
    if constexpr (sizeof(KV) == 4) {
        reinterpret_cast<float4*>(kc)[dst] = k;
        reinterpret_cast<float4*>(vc)[dst] = v;
    } else {
        reinterpret_cast<ushort4*>(kc)[dst] = make_ushort4(cvt<KV>(k.x), cvt<KV>(k.y), cvt<KV>(k.z), cvt<KV>(k.w));
        reinterpret_cast<ushort4*>(vc)[dst] = make_ushort4(cvt<KV>(v.x), cvt<KV>(v.y), cvt<KV>(v.z), cvt<KV>(v.w));
    }
}

template <typename KV>
__global__ __launch_bounds__(256) void kv_append_batch_kernel(
    int B, const float* __restrict__ K, const float* __restrict__ V, KV* __restrict__ kc,
    KV* __restrict__ vc, const int* __restrict__ bt, int nbps, const int* __restrict__ positions,
    int H, int dh, int bs) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t row = (size_t)H * dh;
    if (idx >= (size_t)B * row) return;
    const int b = (int)(idx / row);
    const size_t rem = idx - (size_t)b * row;
    const int pos = positions[b];
    const int blk = pos / bs;
    const size_t dst = ((size_t)bt[(size_t)b * nbps + blk] * bs + (pos - blk * bs)) * row + rem;
    kc[dst] = cvt<KV>(K[idx]);
    vc[dst] = cvt<KV>(V[idx]);
}

}  // namespace

void launch_kv_write(const float* K, const float* V, void* kc, void* vc, int kv_dtype,
                     const int* bt, int seq_len, int start_pos, int H, int dh, int bs,
                     hipStream_t s) {
    const size_t total = (size_t)seq_len * H * dh;
    if (total == 0) return;
    const long long row = (long long)H * dh;
    // whole float4s in every row and buffer; otherwise one element per thread
    const uintptr_t esz = kv_dtype == IE_KV_BF16 ? 8 : 16;  // bytes of four cache elements
    if (row % 4 == 0 && row / 4 <= 256LL * 65535 && (((uintptr_t)K | (uintptr_t)V) % 16) == 0 &&
        (((uintptr_t)kc | (uintptr_t)vc) % esz) == 0) {
        const int n4 = (int)(row / 4);
        const float4 *k4 = reinterpret_cast<const float4*>(K), *v4 = reinterpret_cast<const float4*>(V);
        const bool narrow = n4 <= 64;
        dim3 threads((unsigned)std::min(256, (n4 + 63) / 64 * 64)), grid((unsigned)seq_len, (unsigned)((n4 + 255) / 256));
        if (narrow) {
            unsigned tx = 1;
            while ((int)tx < n4) tx *= 2;
            threads = dim3(tx, 256 / tx);
            grid = dim3((unsigned)(((long long)seq_len + threads.y - 1) / threads.y));
        }
        auto go = [&](auto* kcache, auto* vcache) {
            using KV = std::remove_reference_t<decltype(*kcache)>;
            auto* k = narrow ? kv_write_vec_kernel<KV, true> : kv_write_vec_kernel<KV, false>;
            k<<<grid, threads, 0, s>>>(k4, v4, kcache, vcache, bt, seq_len, start_pos, n4, bs);
        };
        if (kv_dtype == IE_KV_BF16)
            go(static_cast<uint16_t*>(kc), static_cast<uint16_t*>(vc));
        else
            go(static_cast<float*>(kc), static_cast<float*>(vc));
        return;
    }
    const unsigned blocks = (unsigned)((total + 255) / 256);
    if (kv_dtype == IE_KV_BF16)
        kv_write_kernel<uint16_t><<<blocks, 256, 0, s>>>(
            K, V, static_cast<uint16_t*>(kc), static_cast<uint16_t*>(vc), bt, seq_len,
            start_pos, H, dh, bs);
    else
        kv_write_kernel<float><<<blocks, 256, 0, s>>>(K, V, static_cast<float*>(kc),
                                                      static_cast<float*>(vc), bt, seq_len,
                                                      start_pos, H, dh, bs);
}

void launch_kv_append_batch(int B, const float* K, const float* V, void* kc, void* vc,
                            int kv_dtype, const int* bt, int nbps, const int* positions,
                            int H, int dh, int bs, hipStream_t s) {
    const size_t total = (size_t)B * H * dh;
    if (total == 0) return;
    const unsigned blocks = (unsigned)((total + 255) / 256);
    if (kv_dtype == IE_KV_BF16)
        kv_append_batch_kernel<uint16_t><<<blocks, 256, 0, s>>>(
            B, K, V, static_cast<uint16_t*>(kc), static_cast<uint16_t*>(vc), bt, nbps,
            positions, H, dh, bs);
    else
        kv_append_batch_kernel<float><<<blocks, 256, 0, s>>>(
            B, K, V, static_cast<float*>(kc), static_cast<float*>(vc), bt, nbps, positions, H,
            dh, bs);
}

}  // namespace ie

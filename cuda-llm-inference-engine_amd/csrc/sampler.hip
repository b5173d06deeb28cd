// Device half of the top-k sampler (src/sampler.cu:16-45): the k largest
// logits of each row with their indices, sorted by value descending and, for
// equal values, by index ascending (std::partial_sort leaves the order of
// equal values unspecified; this is the order a stable sort gives).  Only
// these k pairs cross PCIe; the reference copies the whole row (201 KB for
// GPT-2) and partial-sorts it on the host.  The draw itself (temperature
// softmax over the k values and the rand() threshold) stays on the host,
// where it is the same float arithmetic as the reference's.
//
// One 1024-thread workgroup per row.  Rows of up to 65533 logits (GPT-2's
// 50257 among them) are read once, as 16-byte chunks, into registers (64 keys
// per thread):
//   1. a lower bound M of the k-th largest key.  For k up to 64 (of 16 full
//      waves): each wave finds, by a bit search with one ballot per bit, the
//      first 20 bits of the r-th largest of its 64 per-thread maxima, r =
//      ceil(k / waves), and M is the least of those, so at least k keys reach
//      it; one barrier.  For larger k the least of the waves' bounds lets ever
//      more keys through (8 rows at k = 400 83.8 against 24.2 us): M is the
//      k-th largest of the 1024 maxima (a radix select over one key per
//      thread, sixteen barriers).  Rows of fewer than 260 logits, and k past
//      the number of maxima, have no bound: every key is a candidate (8 rows of
//      6 at k = 3 13.0 -> 9.9 us), or the row is streamed at once if it has
//      more than are ranked (1 of 3063 at k = 1024 39.6 -> 32.5);
//   2. the keys >= M (typically k to a few times k) gathered into LDS;
//   3. each gathered key ranked by counting those before it (larger key, or
//      equal key and lower index), several threads per key while there are
//      fewer keys than threads, and the first k written.
// Bound by its chain of barriers and by one CU's intake of the row.  Against
// keys in place of floats, the radix select for every k and one thread per
// ranked key: 8 rows of 50257 at k = 40 17.0 -> 9.4 us, 16 at 100 22.7 ->
// 12.2, 4 at 600 83.6 -> 36.7, 1 at 1 12.2 -> 7.8; 3 rows of 1000 at 10 11.5 ->
// 8.5.
// Longer rows, rows that hold a NaN (whose order is its key's: the floats
// above would drop it), and rows where more than 2048 keys reach M (many
// equal values, or k near 1024), are streamed from memory (L2 after the first
// pass) through an exact radix select of the k-th largest key, 8 bits per
// pass (the histogram in LDS; each wave instruction adds its leading lane's
// bin with one atomic, the other lanes' bins lane by lane), a gather of the
// keys above it plus the lowest-index keys equal to it (ranked in index order
// only when some equal keys are left out), and a bitonic sort of those k.
#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>

#include "ie_internal.h"

namespace ie {
namespace {

constexpr int kTopkThreads = 1024;
constexpr int kTopkWaves = kTopkThreads / 64;
constexpr int kTopkUnroll = 8;
constexpr int kTopkRegPer = 64;  // keys per thread in the register-resident kernel
constexpr int kTopkCand = 2048;  // candidates (keys >= the lower bound) sorted directly

// Unsigned key with the order of the floats; -0.0 is keyed as +0.0 so that
// values the reference compares equal are equal here.
__device__ __forceinline__ uint32_t order_key(float x) {
    uint32_t b = __float_as_uint(x);
    if (b == 0x80000000u) b = 0;
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

__device__ __forceinline__ float key_value(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

struct TopkShared {
    uint32_t hist[256];
    uint32_t prefix, remaining, eqcount, gt, eq;
    uint32_t wave_tot[kTopkWaves];
    uint32_t ckey[kTopkCand];
    int cidx[kTopkCand];
};

// Adds one key per lane (where `match`) to bin `digit`: the leading lane's
// bin in one atomic for every lane that shares it.
__device__ __forceinline__ void hist_add(uint32_t* hist, bool match, uint32_t digit, int lane) {
    const uint64_t mm = __ballot(match);
    if (!mm) return;
    const int lead = __ffsll((unsigned long long)mm) - 1;
    const uint32_t d0 = __shfl(digit, lead, 64);
    const uint64_t same = __ballot(match && digit == d0);
    if (match && digit != d0) atomicAdd(&hist[digit], 1u);
    if (lane == lead) atomicAdd(&hist[d0], (uint32_t)__popcll(same));
}

// Wave 0 finds the bin holding the remaining-th largest key among those with
// the current prefix and publishes the longer prefix, the keys still needed
// within it and its count.  Called by every thread between two barriers.
__device__ __forceinline__ void select_digit(TopkShared& sh, uint32_t prefix, uint32_t remaining, int shift,
                                             int lane, int wid) {
    if (wid != 0) return;
    uint32_t c[4], s = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // lane l holds bins 255-4l .. 252-4l: lanes run from the top
        c[j] = sh.hist[255 - 4 * lane - j];
        s += c[j];
    }
    uint32_t incl = s;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t t = __shfl_up(incl, off, 64);
        if (lane >= off) incl += t;
    }
    uint32_t acc = incl - s;
    if (acc < remaining && remaining <= incl) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (acc < remaining && remaining <= acc + c[j]) {
                sh.prefix = prefix | ((uint32_t)(255 - 4 * lane - j) << shift);
                sh.remaining = remaining - acc;
                sh.eqcount = c[j];
            }
            acc += c[j];
        }
    }
}

__device__ __forceinline__ void put(TopkShared& sh, uint32_t slot, uint32_t key, int i) {
    sh.ckey[slot] = key;
    sh.cidx[slot] = i;
}

// Radix select of the k-th largest key, 8 bits per pass from the top:
// add(hmask, prefix, shift) puts every candidate key whose bits under hmask
// equal prefix into bin (key >> shift) & 255.  Returns the key; `remaining`
// = how many keys equal to it belong to the top k, `eqcount` = how many
// candidates equal it.  Called by every thread.
template <typename Add>
__device__ __forceinline__ uint32_t radix_kth(TopkShared& sh, uint32_t k, Add&& add, int lane, int wid,
                                              uint32_t& remaining, uint32_t& eqcount) {
    uint32_t prefix = 0;
    remaining = k;
    for (int pass = 0; pass < 4; ++pass) {
        const int shift = 24 - 8 * pass;
        const uint32_t hmask = pass == 0 ? 0u : (0xffffffffu << (shift + 8));
        if (threadIdx.x < 256) sh.hist[threadIdx.x] = 0;
        __syncthreads();
        add(hmask, prefix, shift);
        __syncthreads();
        select_digit(sh, prefix, remaining, shift, lane, wid);
        __syncthreads();
        prefix = sh.prefix;
        remaining = sh.remaining;
        eqcount = sh.eqcount;
        __syncthreads();  // all have read before the next pass publishes
    }
    return prefix;
}

// Bitonic sort of the `count` gathered entries (larger key first, then
// lower index); the first k are the output row.
__device__ __forceinline__ void sort_and_write(TopkShared& sh, int count, int k, float* out_vals, int* out_idx) {
    int KP = 1;
    while (KP < count) KP <<= 1;
    for (int t = count + threadIdx.x; t < KP; t += kTopkThreads) put(sh, t, 0u, INT_MAX);
    __syncthreads();
    for (int size = 2; size <= KP; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int t = threadIdx.x; t < KP / 2; t += kTopkThreads) {
                const int i = 2 * stride * (t / stride) + (t % stride), j = i + stride;
                const bool desc = (i & size) == 0;
                const uint32_t ka = sh.ckey[i], kb = sh.ckey[j];
                const int ia = sh.cidx[i], ib = sh.cidx[j];
                const bool a_first = ka > kb || (ka == kb && ia < ib);
                if (a_first != desc) {
                    put(sh, i, kb, ib);
                    put(sh, j, ka, ia);
                }
            }
            __syncthreads();
        }
    }
    for (int t = threadIdx.x; t < k; t += kTopkThreads) {
        out_vals[(size_t)blockIdx.x * k + t] = key_value(sh.ckey[t]);
        out_idx[(size_t)blockIdx.x * k + t] = sh.cidx[t];
    }
}

// Streams one row (every pass re-reads it: L2 after the first).
__device__ __forceinline__ void topk_stream_row(TopkShared& sh, const float* __restrict__ x, int n, int k,
                                                float* __restrict__ out_vals, int* __restrict__ out_idx, int lane,
                                                int wid) {
    // visits every index in rounds of kTopkUnroll coalesced loads per thread
    auto for_each = [&](auto&& f) {
        for (int base = threadIdx.x; base < n; base += kTopkThreads * kTopkUnroll) {
            float v[kTopkUnroll];
#pragma unroll
            for (int u = 0; u < kTopkUnroll; ++u) {
                const int i = base + u * kTopkThreads;
                v[u] = x[min(i, n - 1)];
            }
#pragma unroll
            for (int u = 0; u < kTopkUnroll; ++u) f(base + u * kTopkThreads, order_key(v[u]));
        }
    };

    uint32_t remaining, eqcount;
    const uint32_t prefix = radix_kth(
        sh, (uint32_t)k,
        [&](uint32_t hmask, uint32_t prefix, int shift) {
            for_each([&](int i, uint32_t key) {
                hist_add(sh.hist, i < n && (key & hmask) == prefix, (key >> shift) & 255u, lane);
            });
        },
        lane, wid, remaining, eqcount);
    const uint32_t T = prefix, kgt = (uint32_t)k - remaining;

    if (threadIdx.x == 0) sh.gt = sh.eq = 0;
    if (eqcount == remaining) {
        __syncthreads();
        for_each([&](int i, uint32_t key) {
            if (i < n && key >= T) put(sh, key > T ? atomicAdd(&sh.gt, 1u) : kgt + atomicAdd(&sh.eq, 1u), key, i);
        });
    } else {
        // Wave w walks indices [w S, (w+1) S) in order; a first walk counts
        // its equal keys so that every equal key gets its global rank.
        const int S = ((n + kTopkWaves - 1) / kTopkWaves + 63) & ~63;
        const int lo = wid * S, hi = min(n, lo + S);
        uint32_t cnt = 0;
        for (int i0 = lo; i0 < hi; i0 += 64) {
            const int i = i0 + lane;
            cnt += (uint32_t)__popcll(__ballot(i < hi && order_key(x[i]) == T));
        }
        if (lane == 0) sh.wave_tot[wid] = cnt;
        __syncthreads();
        uint32_t rank = 0;
        for (int w = 0; w < wid; ++w) rank += sh.wave_tot[w];
        const uint64_t below = (1ull << lane) - 1;
        for (int i0 = lo; i0 < hi; i0 += 64) {
            const int i = i0 + lane;
            const uint32_t key = i < hi ? order_key(x[i]) : 0u;
            const uint64_t eq = __ballot(i < hi && key == T);
            if (i < hi && key > T) put(sh, atomicAdd(&sh.gt, 1u), key, i);
            const uint32_t r = rank + (uint32_t)__popcll(eq & below);
            if (i < hi && key == T && r < remaining) put(sh, kgt + r, key, i);
            rank += (uint32_t)__popcll(eq);
        }
    }
    __syncthreads();
    sort_and_write(sh, k, k, out_vals, out_idx);
}

// Rows whose 16-byte chunks number at most 16 x 1024 (n + 3 <= 65536): the
// row is read once as 16-byte chunks from its 16-byte-aligned base, thread t
// holding chunks t + 1024 q (q < 16), i.e. indices 4 (t + 1024 q) + c - s
// where s = the row start's float offset within its chunk; slots outside the
// row hold -inf.
__global__ __launch_bounds__(kTopkThreads) void topk_reg_kernel(const float* __restrict__ logits, int n, int k,
                                                                float* __restrict__ out_vals,
                                                                int* __restrict__ out_idx) {
    __shared__ TopkShared sh;
    const float* x = logits + (size_t)blockIdx.x * n;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int s = (int)(((uintptr_t)x & 15u) >> 2);
    const float4* x4 = reinterpret_cast<const float4*>(x - s);
    // chunks wholly inside the row: [cf, cl]; the (at most two) others that
    // touch it are read element by element by the one lane that holds each
    const int cf = s == 0 ? 0 : 1, cl = (n + s) / 4 - 1;
    // The row's values stay floats (compared as such: -0 equals +0, and the
    // slots past its ends hold -inf); only maxima and candidates become keys.
    constexpr int NC = kTopkRegPer / 4;
    float4 val[NC];
#pragma unroll
    for (int q = 0; q < NC; ++q) {
        const int c = (int)threadIdx.x + q * kTopkThreads;
        // branch-free for whole chunks, so all 16 loads are in flight together
        val[q] = cf <= cl ? x4[min(max(c, cf), cl)] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float fmx = -INFINITY;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
        const int c = (int)threadIdx.x + q * kTopkThreads, e0 = 4 * c - s;
        if (c < cf || c > cl) {
            auto at = [&](int e) { return e >= 0 && e < n ? x[e] : -INFINITY; };
            val[q] = make_float4(at(e0), at(e0 + 1), at(e0 + 2), at(e0 + 3));
        }
        // (a NaN stays in this maximum)
        fmx = __builtin_elementwise_maximum(fmx, __builtin_elementwise_maximum(val[q].x, val[q].y));
        fmx = __builtin_elementwise_maximum(fmx, __builtin_elementwise_maximum(val[q].z, val[q].w));
    }
    const bool nan = __ballot(fmx != fmx) != 0;  // in this wave's part
    // index of a chunk's first element: one base per thread plus a constant
    const int ibase = 4 * (int)threadIdx.x - s;

    // Lower bound M of the k-th largest (see the top).  (Every loop over val[]
    // is fully unrolled: an early exit would leave the array indexed at run
    // time, i.e. in scratch memory.)
    const uint32_t tmax = order_key(fmx);
    // Full waves: every lane holds at least one whole chunk of the row.
    const int full = min(kTopkWaves, (n - 4) / 256);
    const int held = (n + s + 3) / 4;  // threads that hold any of it, if below 1024
    if (k > held && n > kTopkCand) {   // uniform: no bound below the whole row, which is too much
        topk_stream_row(sh, x, n, k, out_vals, out_idx, lane, wid);
        return;
    }
    uint32_t M;
    if (k > held || full == 0) {  // uniform: every key is a candidate
        if (lane == 0) sh.wave_tot[wid] = nan ? 0u : order_key(-INFINITY);
        if (threadIdx.x == 0) sh.gt = 0;
        __syncthreads();
        M = sh.wave_tot[0];
#pragma unroll
        for (int w = 1; w < kTopkWaves; ++w) M = min(M, sh.wave_tot[w]);
    } else if (k <= 4 * full) {  // uniform
        const int r = (k + full - 1) / full;
        uint32_t m = 0;
#pragma unroll
        for (int bit = 31; bit >= 12; --bit) {
            const uint32_t c = m | (1u << bit);
            if (__popcll(__ballot(tmax >= c)) >= r) m = c;
        }
        if (lane == 0) sh.wave_tot[wid] = nan ? 0u : wid < full ? m : 0xffffffffu;  // (no real m is 0)
        if (threadIdx.x == 0) sh.gt = 0;
        __syncthreads();
        M = sh.wave_tot[0];
#pragma unroll
        for (int w = 1; w < kTopkWaves; ++w) M = min(M, sh.wave_tot[w]);
    } else {
        uint32_t remaining, eqcount;
        M = radix_kth(
            sh, (uint32_t)k,
            [&](uint32_t hmask, uint32_t prefix, int shift) {
                hist_add(sh.hist, (tmax & hmask) == prefix, (tmax >> shift) & 255u, lane);
            },
            lane, wid, remaining, eqcount);
        if (lane == 0) sh.wave_tot[wid] = nan ? 0u : M;
        if (threadIdx.x == 0) sh.gt = 0;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kTopkWaves; ++w) M = min(M, sh.wave_tot[w]);
    }
    if (M == 0) {  // uniform: a NaN in the row
        __syncthreads();
        topk_stream_row(sh, x, n, k, out_vals, out_idx, lane, wid);
        return;
    }
    const float Mf = M <= order_key(-INFINITY) ? -INFINITY : key_value(M);
#pragma unroll
    for (int q = 0; q < NC; ++q) {
        const float e[4] = {val[q].x, val[q].y, val[q].z, val[q].w};
        if (__ballot(fmaxf(fmaxf(e[0], e[1]), fmaxf(e[2], e[3])) >= Mf)) {  // (uniform: few chunks have any)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = ibase + q * (4 * kTopkThreads) + u;
                if (e[u] >= Mf && i >= 0 && i < n) {
                    const uint32_t slot = atomicAdd(&sh.gt, 1u);
                    if (slot < (uint32_t)kTopkCand) put(sh, slot, order_key(e[u]), i);
                }
            }
        }
    }
    __syncthreads();
    const uint32_t cnt = sh.gt;
    if (cnt > (uint32_t)kTopkCand) {  // uniform
        __syncthreads();  // all have read the count before the stream resets it
        topk_stream_row(sh, x, n, k, out_vals, out_idx, lane, wid);
        return;
    }
    // rank sort: a candidate's place is the number of candidates before it
    // (larger key, or equal key and lower index: the larger of the words
    // packed here); places are distinct.  2^per threads share a candidate,
    // reading two others at a time.
    __shared__ __attribute__((aligned(16))) uint64_t pk[kTopkCand + 2];
    for (int t = threadIdx.x; t < (int)cnt + 2; t += kTopkThreads)
        pk[t] = t < (int)cnt ? ((uint64_t)sh.ckey[t] << 32) | (0xffffffffu - (uint32_t)sh.cidx[t]) : 0;
    __syncthreads();
    int per = 0;
    while (per < 5 && ((int)cnt << (per + 1)) <= kTopkThreads) ++per;
    const int sub = threadIdx.x & ((1 << per) - 1);
    for (int t = threadIdx.x >> per; t < (int)cnt; t += kTopkThreads >> per) {
        const uint64_t mine = pk[t];
        int rank = 0;
#pragma unroll 4
        for (int u = 2 * sub; u < (int)cnt; u += 2 << per) {
            const ulonglong2 o = *reinterpret_cast<const ulonglong2*>(pk + u);
            rank += (int)(o.x > mine) + (int)(o.y > mine);
        }
        for (int o = 1; o < 1 << per; o <<= 1) rank += __shfl_xor(rank, o, 64);
        if (sub == 0 && rank < k) {
            out_vals[(size_t)blockIdx.x * k + rank] = key_value(sh.ckey[t]);
            out_idx[(size_t)blockIdx.x * k + rank] = sh.cidx[t];
        }
    }
}

// Longer rows.
__global__ __launch_bounds__(kTopkThreads) void topk_stream_kernel(const float* __restrict__ logits, int n, int k,
                                                                   float* __restrict__ out_vals,
                                                                   int* __restrict__ out_idx) {
    __shared__ TopkShared sh;
    topk_stream_row(sh, logits + (size_t)blockIdx.x * n, n, k, out_vals, out_idx, threadIdx.x & 63,
                    threadIdx.x >> 6);
}

}  // namespace

void launch_topk(int rows, const float* logits, int n, int k, float* out_vals, int* out_idx, hipStream_t s) {
    if (rows == 0) return;
    if (n + 3 <= kTopkRegPer * kTopkThreads)
        topk_reg_kernel<<<rows, kTopkThreads, 0, s>>>(logits, n, k, out_vals, out_idx);
    else
        topk_stream_kernel<<<rows, kTopkThreads, 0, s>>>(logits, n, k, out_vals, out_idx);
}

}  // namespace ie

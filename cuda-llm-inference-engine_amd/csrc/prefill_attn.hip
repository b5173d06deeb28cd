// prefill_attn.hip — causal attention over a prompt chunk, for gfx950.
//
// Computes what the reference's K10 FlashAttention-2 forward computes
// (kernels/flash_attention/10_flash_attn_v2.cu:27-236; called for a fresh
// prompt at src/gpt2_engine.cu:484-493): for every sequence b, head h and query
// t, O = softmax(q . K^T / sqrt(d)) V over the keys at positions <= the
// query's position (all keys when not causal).  Two operand layouts:
//   * paged (the engine's prefill): Q and O token-major [B, P, H_q, d] (the
//     QKV projection's own layout, so no transposes), K/V read back from the
//     paged cache [phys][block_size][H_kv][d] (fp32 or bf16) through the block
//     table after the chunk's K/V were appended; query t of a sequence sits at
//     position start + t, so a chunk continuing an existing context sees the
//     earlier tokens too;
//   * contiguous [B, H, N, d] fp32 for Q, K, V, O (the reference's K10
//     signature, run_flash_attn_v2).
//
// Two families of kernels.
//
// prefill_fp32_kernel (fp32 operands): S^T = K Q^T and O^T += V^T P^T on
// v_mfma_f32_16x16x4_f32, one workgroup per 16 queries, its four waves taking
// the 16-token chunks round-robin, merged in LDS.  Lane l (i = l % 16, g =
// l / 16) holds, for query i of the tile, q elements d/4 g .. + d/4 - 1 (MFMA
// step s takes element d/4 g + s of K and q alike), the scores of keys 4g .. 4g+3
// of a chunk (the MFMA result layout, which is the B operand P^T of the second
// product), and output elements d/16 (4g + v) + t.
//
// prefill_split_kernel and prefill_tile_kernel: the fp32 matrix rate is a
// sixteenth of the bf16 one, so here the two products run on
// v_mfma_f32_16x16x32_bf16 with every fp32 operand written as the sum of three
// bf16 (each rounded to nearest even, 8 bits apiece, so the sum is the fp32
// value; V and the weights are scaled for it, keys below 2^-110 lose less
// than 2^-133, see split_query): six of the nine partial products (those down to 2^-16 of the
// largest; the rest are below 2^-24 of it) accumulate in fp32.  A bf16 cache is
// exact in one part and takes three.  Error against 64 bits: about half the
// fp32 kernel's over d, keys and caches (flash 2048 x 128 1.9e-7 against
// 3.7e-7, paged bf16 300 x 64 1.1e-7 against 2.2e-7).  Every query sees the same
// operations in the same order whatever the tile or kernel of the two:
//   * keys in blocks of 32 from position 0 on, block c in group c % 4; each
//     group keeps its own running maximum m, sum l and output o (an online
//     softmax step per block), and the four groups are merged in order at the
//     end (merge_weights).  Keys past a query's limit have weight exactly 0, so
//     a block or group without keys changes nothing;
//   * scores are pre-multiplied by log2(e)/sqrt(d) (folded into q, as in the
//     fp32 kernel), so the softmax uses the hardware exp2.
// An operand that is infinite, NaN or too large for its (scaled) parts makes
// NaN, and a query may be too small or too large for its own (split_query): the
// queries of a tile whose outputs are not all finite, and such queries, are
// computed again with fp32 MFMAs (exact_tile), which gives what the operands'
// own arithmetic gives; the tile's others keep their bits.
//
// Which family: a paged launch by the cache type alone (bf16: the three-part
// kernels), so over finite operands a query's bits never depend on the batch or on
// how a prompt is chunked; a contiguous one by its shape (prefill_form).  (An
// infinite or NaN value of V at a key that a query does not see can still reach it,
// 0 times it being a NaN: from a later key of its block, and in the fp32 MFMAs from
// the keys of its own 16 queries.  Such a query is computed again, or is itself a
// NaN, as its tile lies.)
//
// In the three-part kernels a wave owns 16 queries of one (b, h).  Operands
// (lane l: i = l % 16, g = l / 16): S^T = K Q^T, 16 keys x 16 queries per MFMA, leaves lane l with query i and
// key 4g + v of the tile in result v, so the eight weights of a 32-key block
// that a lane ends with (keys 4g + v and 16 + 4g + v: octet g) are already the
// B operand P^T of O^T += V^T P^T, whose A operand V^T takes the same octet.
//   * prefill_tile_kernel: 64 queries on GW x 4 waves, waves w, w + 4, ...
//     sharing 16 queries, each four walking 4 / GW of the groups.  They load
//     their next step's K and V into registers, split them once for the four
//     and write them to LDS (K rows as they are, V transposed with a row's
//     keys in octet order, 16-byte chunks XOR-swizzled); two barriers a step.
//     GW = 1 leaves LDS for several workgroups per CU, which fill each other's
//     gaps; GW = 2 halves a tile's chain of dependent steps.
//   * prefill_split_kernel (few or short queries): one workgroup per 16
//     queries, its four waves the four groups, each loading its blocks
//     straight into the operand layout (O^T row (t, i) then is element
//     d/16 i + t, so V loads are 16 bytes per key); the merge goes through LDS.
// The grid is one-dimensional, tile rank major: workgroup u takes pair p =
// u % (H_q B) and tile rank r = u / (H_q B) (rank 0 = the last, longest tile),
// so the longest tiles (causal triangles) are dispatched first and, as
// workgroups go to the XCDs round-robin, with H_q B a multiple of 8 all tiles
// of one (b, h) run on one XCD (its K/V fetched into one L2) and every XCD
// gets the same mix of tile lengths.
#include <cmath>

#include "device_util.h"
#include "ie_internal.h"

namespace ie {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kQW = 16;     // queries per wave
constexpr int kKB = 32;     // keys per block
constexpr int kGroups = 4;  // block c belongs to group c % 4
constexpr int kWaves = 4;

template <int W>
__device__ __forceinline__ void load_words(const void* p, uint32_t (&w)[W]) {
    if constexpr (W % 4 == 0) {
#pragma unroll
        for (int i = 0; i < W / 4; ++i) {
            const uint4 v = reinterpret_cast<const uint4*>(p)[i];
            w[4 * i] = v.x;
            w[4 * i + 1] = v.y;
            w[4 * i + 2] = v.z;
            w[4 * i + 3] = v.w;
        }
    } else if constexpr (W == 2) {
        const uint2 v = *reinterpret_cast<const uint2*>(p);
        w[0] = v.x;
        w[1] = v.y;
    } else {
        static_assert(W == 1, "slice width");
        w[0] = *reinterpret_cast<const uint32_t*>(p);
    }
}

// Element j of a lane's raw K or V slice.
template <typename KV, int W>
__device__ __forceinline__ float elem(const uint32_t (&w)[W], int j) {
    if constexpr (sizeof(KV) == 4) {
        return __builtin_bit_cast(float, w[j]);
    } else {
        const uint32_t x = w[j >> 1];
        return __builtin_bit_cast(float, (j & 1) ? (x & 0xffff0000u) : (x << 16));
    }
}

// ---- fp32 MFMA form: 16 queries, 16-token chunks.
// A lane's share of one 16-token chunk: d/4 elements of key i's K, and
// d/16 elements (from d/16 * i) of each of the keys 4g .. 4g+3's V.
template <int D, typename KV>
struct Chunk {
    static constexpr int KW = D / 4 * (int)sizeof(KV) / 4;
    static constexpr int VW = D / 16 * (int)sizeof(KV) / 4;
    uint32_t k[KW];
    uint32_t v[4][VW];
};

// Where token `pos` of the current (b, kv head) lives, in elements from the
// head's base pointer.
//   LAYOUT 0, PAGE 1: paged, blocks of 16 tokens; `phys` is the chunk's block.
//   LAYOUT 0, PAGE 2: blocks of 2^run_log runs of 16 tokens; `phys` is the
//                     chunk's run in the cache.
//   LAYOUT 0, PAGE 0: any block size (per-lane table lookup).
//   LAYOUT 1:         contiguous rows.
template <int LAYOUT, int PAGE>
struct TokenMap {
    const int* bt;
    int block_size, run_log;
    size_t stride;  // elements between consecutive token rows of one head
    __device__ __forceinline__ size_t off(int pos, int phys) const {
        if constexpr (LAYOUT == 1) {
            return (size_t)pos * stride;
        } else if constexpr (PAGE) {
            return ((size_t)phys * 16 + (pos & 15)) * stride;
        } else {
            const int blk = pos / block_size;
            return ((size_t)bt[blk] * block_size + (pos - blk * block_size)) * stride;
        }
    }
    // the run that holds token pos (PAGE 1 and 2; wave-uniform).  A form of its own
    // for blocks of 16: shifts cost a long prompt 1-2% here, a branch 5% (each
    // lookup then waits for the one before).
    __device__ __forceinline__ int run_of(int pos) const {
        const int r = pos >> 4;
        if constexpr (PAGE == 1) return bt[r];
        return (bt[r >> run_log] << run_log) + (r & ((1 << run_log) - 1));
    }
};

template <int D, typename KV, int LAYOUT, int PAGE>
__device__ __forceinline__ void load_chunk(Chunk<D, KV>& c, int c0, int kend, int i, int g, int phys,
                                           const TokenMap<LAYOUT, PAGE>& map, const KV* kbase,
                                           const KV* vbase) {
    const int kp = min(c0 + i, kend - 1);
    load_words(kbase + map.off(kp, phys) + (D / 4) * g, c.k);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int vp = min(c0 + 4 * g + s, kend - 1);
        load_words(vbase + map.off(vp, phys) + (D / 16) * i, c.v[s]);
    }
}

// One chunk: scores, masked online softmax, P.V.  qpos = this lane's query
// position (keys > qpos are masked when causal), kend = keys in range.
template <int D, typename KV>
__device__ __forceinline__ void consume(const Chunk<D, KV>& c, int c0, int g, const float (&q)[D / 4],
                                        int klim, float& m, float& l, f32x4 (&o)[D / 16]) {
    f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int e = 0; e < D / 4; ++e)
        s = __builtin_amdgcn_mfma_f32_16x16x4f32(elem<KV>(c.k, e), q[e], s, 0, 0, 0);
    float cm = -INFINITY;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        if (c0 + 4 * g + v >= klim) s[v] = -INFINITY;
        cm = fmaxf(cm, s[v]);
    }
    cm = max_xor32(max_xor16(cm));
    const float mn = fmaxf(m, cm);
    const float mu = mn == -INFINITY ? 0.0f : mn;  // no key yet: keep o, l at 0
    const float alpha = exp2_sm(m - mu);
    float p[4], ls = 0.0f;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        p[v] = exp2_sm(s[v] - mu);
        ls += p[v];
    }
    ls = sum_xor32(sum_xor16(ls));
    l = fmaf(l, alpha, ls);
    m = mn;
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
        o[t] *= alpha;
#pragma unroll
        for (int sv = 0; sv < 4; ++sv)
            o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(elem<KV>(c.v[sv], t), p[sv], o[t], 0, 0, 0);
    }
}

// ---- fp32 MFMA kernel: 16 queries per workgroup, its four waves taking the
// 16-token chunks round-robin, merged in LDS.
// LAYOUT 0: Q/O [B, P, H_q, D], keys = start + P cached tokens.
// LAYOUT 1: Q/K/V/O [B, H, P, D], keys = P, start = 0.
template <int D, typename KV, int LAYOUT, int PAGE>
__global__ __launch_bounds__(256) void prefill_fp32_kernel(
    const float* __restrict__ Q, const KV* __restrict__ kcache, const KV* __restrict__ vcache,
    const int* __restrict__ block_table, int nbps, int block_size, int P, int H_q, int H_kv,
    int start, int causal, float qscale, float* __restrict__ O) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int ntiles = (P + kQW - 1) / kQW;
    const int pairs = (int)(gridDim.x / (unsigned)ntiles);  // H_q B
    const int r = (int)blockIdx.x / pairs, pr = (int)blockIdx.x - r * pairs;
    const int qt = ntiles - 1 - r;  // longest (last) tiles first
    const int h = pr % H_q, b = pr / H_q;
    const int kvh = h / (H_q / H_kv);
    const int q0 = qt * kQW;
    const int qlast = min(q0 + kQW - 1, P - 1);
    const int nkeys = start + P;
    // Keys this tile needs, and this lane's own limit.
    const int kend = causal ? min(start + qlast + 1, nkeys) : nkeys;
    const int klim = causal ? min(start + q0 + i + 1, kend) : kend;
    const int qi = min(q0 + i, P - 1);

    size_t qrow;
    TokenMap<LAYOUT, PAGE> map{};
    const KV* kbase;
    const KV* vbase;
    if constexpr (LAYOUT == 0) {
        qrow = (((size_t)b * P + qi) * H_q + h) * D;
        map.bt = block_table + (size_t)b * nbps;
        map.block_size = block_size;
        map.stride = (size_t)H_kv * D;
        kbase = kcache + (size_t)kvh * D;
        vbase = vcache + (size_t)kvh * D;
    } else {
        qrow = (((size_t)b * H_q + h) * P + qi) * D;
        map.stride = D;
        kbase = kcache + ((size_t)b * H_kv + kvh) * P * D;
        vbase = vcache + ((size_t)b * H_kv + kvh) * P * D;
    }

    float q[D / 4];
#pragma unroll
    for (int e = 0; e < D / 4; e += 4) {
        const float4 v = *reinterpret_cast<const float4*>(Q + qrow + (D / 4) * g + e);
        q[e] = v.x * qscale;
        q[e + 1] = v.y * qscale;
        q[e + 2] = v.z * qscale;
        q[e + 3] = v.w * qscale;
    }

    float m = -INFINITY, l = 0.0f;
    f32x4 o[D / 16];
#pragma unroll
    for (int t = 0; t < D / 16; ++t) o[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    constexpr int STEP = 16 * kWaves;
    auto phys = [&](int cs) {
        if constexpr (LAYOUT == 0 && PAGE) return map.bt[min(cs, kend - 1) >> 4];
        else return 0;
    };
    Chunk<D, KV> ca, cb;
    int c0 = 16 * wave;
    int pn = 0;
    if (c0 < kend) {
        load_chunk(ca, c0, kend, i, g, phys(c0), map, kbase, vbase);
        pn = phys(c0 + STEP);
    }
    auto next = [&](Chunk<D, KV>& c, int cs) {
        load_chunk(c, cs, kend, i, g, pn, map, kbase, vbase);
        pn = phys(cs + STEP);
    };
    // Ping-pong: chunk c0 + STEP (clamped past the end) is always in flight
    // while chunk c0 is computed.
    while (c0 < kend) {
        next(cb, c0 + STEP);
        consume(ca, c0, g, q, klim, m, l, o);
        c0 += STEP;
        if (c0 >= kend) break;
        next(ca, c0 + STEP);
        consume(cb, c0, g, q, klim, m, l, o);
        c0 += STEP;
    }

    // Merge the four waves' partial softmax states in LDS.
    __shared__ float sm_o[kWaves][kQW][D + 4];
    __shared__ float sm_m[kWaves][kQW], sm_l[kWaves][kQW];
#pragma unroll
    for (int t = 0; t < D / 16; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) sm_o[wave][i][(D / 16) * (4 * g + v) + t] = o[t][v];
    if (g == 0) {
        sm_m[wave][i] = m;
        sm_l[wave][i] = l;
    }
    __syncthreads();

    constexpr int PER = kQW * D / 256;  // outputs per thread (4 or 8)
    const int qq = threadIdx.x / 16, col = (threadIdx.x % 16) * PER;
    if (q0 + qq >= P) return;
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, sm_m[w][qq]);
    float f[kWaves], L = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        f[w] = sm_m[w][qq] == -INFINITY ? 0.0f : exp2_sm(sm_m[w][qq] - mx);
        L = fmaf(f[w], sm_l[w][qq], L);
    }
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    float out[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        float acc = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) acc = fmaf(f[w], sm_o[w][qq][col + e], acc);
        out[e] = acc * inv;
    }
    const int qo = q0 + qq;
    float* orow = LAYOUT == 0 ? O + (((size_t)b * P + qo) * H_q + h) * D
                              : O + (((size_t)b * H_q + h) * P + qo) * D;
#pragma unroll
    for (int e = 0; e < PER; e += 4)
        *reinterpret_cast<float4*>(orow + col + e) = make_float4(out[e], out[e + 1], out[e + 2], out[e + 3]);
}

// ---- three-part bf16 form
// bf16 parts of a pair: x0 in the low half of each word.
__device__ __forceinline__ uint32_t round_pair(float x0, float x1) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{x0, x1}), bf16x2));
}
// The parts of x0 s and x1 s, what the first leaves taken from the unrounded
// product.
__device__ __forceinline__ void split_pair(float x0, float x1, float s, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = round_pair(x0 * s, x1 * s);
    const float r0 = fmaf(x0, s, -__builtin_bit_cast(float, h << 16));
    const float r1 = fmaf(x1, s, -__builtin_bit_cast(float, h & 0xffff0000u));
    m = round_pair(r0, r1);
    l = round_pair(r0 - __builtin_bit_cast(float, m << 16), r1 - __builtin_bit_cast(float, m & 0xffff0000u));
}

// Eight elements of an MFMA operand, NP parts: 3 for fp32, 1 for bf16.
template <int NP>
struct Parts {
    uint4 p[NP];
};
template <typename KV>
constexpr int kParts = sizeof(KV) == 4 ? 3 : 1;

// The weights and the fp32 values of V are split times 2^24 (exact), so that no
// part of a normal weight or of any value is below bf16's range; the output
// is divided by both.  (Unscaled, values below 1e-34 lost their third part and
// those below 1e-36 more than 1e-5 of themselves; 1 x 16 x 2048 x 128 125.8 -> 126.8 us
// for the multiplications, ordinary operands' bits unchanged.)
constexpr float kUp = 0x1p24f;
template <typename KV>
constexpr float kDown = sizeof(KV) == 4 ? 0x1p-48f : 0x1p-24f;  // (a bf16 value is one part as it is)

__device__ __forceinline__ Parts<3> split8(const float (&x)[8], float s = 1.0f) {
    Parts<3> r;
    split_pair(x[0], x[1], s, r.p[0].x, r.p[1].x, r.p[2].x);
    split_pair(x[2], x[3], s, r.p[0].y, r.p[1].y, r.p[2].y);
    split_pair(x[4], x[5], s, r.p[0].z, r.p[1].z, r.p[2].z);
    split_pair(x[6], x[7], s, r.p[0].w, r.p[1].w, r.p[2].w);
    return r;
}

// Elements `odd` (0 or 1) of two words, as one word (one v_perm).
__device__ __forceinline__ uint32_t pair_bf16(uint32_t lo, uint32_t hi, int odd) {
    return __builtin_amdgcn_perm(hi, lo, odd ? 0x07060302u : 0x05040100u);
}
// A lane's eight consecutive raw elements as parts.
template <typename KV, int W>
__device__ __forceinline__ Parts<kParts<KV>> parts8(const uint32_t (&w)[W]) {
    if constexpr (sizeof(KV) == 4) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = __builtin_bit_cast(float, w[e]);
        return split8(x);
    } else {
        return Parts<1>{{make_uint4(w[0], w[1], w[2], w[3])}};
    }
}

__device__ __forceinline__ f32x4 mfma(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <int D>
struct Group {
    float m, l;
    f32x4 o[D / 16];  // o[t][v]: row 4g + v of tile t
    __device__ __forceinline__ void clear() {
        m = -INFINITY;
        l = 0.0f;
#pragma unroll
        for (int t = 0; t < D / 16; ++t) o[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
};

// Scores of one block: key(j, s) = the A operand of keys 16 j .. 16 j + 15 at
// k-step s; sc[4 j + v] is key 16 j + 4 g + v.  Keys at or past klim are masked
// when `edge` (uniform) says that the block has some.
template <int D, int NP, typename GetK>
__device__ __forceinline__ void scores(GetK&& key, const Parts<3> (&q)[D / 32], int c0, int klim, bool edge, int g,
                                       float (&sc)[8]) {
    f32x4 big[2], small[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) big[j] = small[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < D / 32; ++s) {
        Parts<NP> k[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) k[j] = key(j, s);
        // small and large products in chains of their own, the two key tiles side by side
        auto all = [&](f32x4(&acc)[2], int kp, int qp) {
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[j] = mfma(k[j].p[kp], q[s].p[qp], acc[j]);
        };
        if constexpr (NP == 3) {
            all(small, 2, 0);
            all(small, 0, 2);
            all(small, 1, 1);
            all(small, 1, 0);
        } else {
            all(small, 0, 2);
        }
        all(small, 0, 1);
        all(big, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 8; ++v) sc[v] = big[v >> 2][v & 3] + small[v >> 2][v & 3];
    if (edge) {
#pragma unroll
        for (int v = 0; v < 8; ++v)
            if (c0 + 16 * (v >> 2) + 4 * g + (v & 3) >= klim) sc[v] = -INFINITY;
    }
}

// Online softmax step and P.V of one block: val(t) = the A operand (16 rows
// of tile t, octet g).
template <int D, int NP, typename GetV>
__device__ __forceinline__ void attend(GetV&& val, const float (&sc)[8], Group<D>& gr) {
    float cm = sc[0];
#pragma unroll
    for (int v = 1; v < 8; ++v) cm = fmaxf(cm, sc[v]);
    cm = max_xor32(max_xor16(cm));
    const float mn = fmaxf(gr.m, cm);
    const float mu = mn == -INFINITY ? 0.0f : mn;  // no key yet: keep o, l at 0
    const float alpha = exp2_sm(gr.m - mu);
    float p[8], ls = 0.0f;
#pragma unroll
    for (int v = 0; v < 8; ++v) {
        p[v] = exp2_sm(sc[v] - mu);
        ls += p[v];
    }
    ls = sum_xor32(sum_xor16(ls));
    gr.l = fmaf(gr.l, alpha, ls);
    gr.m = mn;
    if (__ballot(alpha != 1.0f)) {  // (a factor of 1 changes nothing)
#pragma unroll
        for (int t = 0; t < D / 16; ++t) gr.o[t] *= alpha;
    }
    const Parts<3> pp = split8(p, kUp);
    // four tiles side by side, so that an accumulator's MFMAs are not back to back
#pragma unroll
    for (int t0 = 0; t0 < D / 16; t0 += 4) {
        Parts<NP> x[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) x[k] = val(t0 + k);
        auto all = [&](int vp, int wp) {
#pragma unroll
            for (int k = 0; k < 4; ++k) gr.o[t0 + k] = mfma(x[k].p[vp], pp.p[wp], gr.o[t0 + k]);
        };
        if constexpr (NP == 3) {
            all(2, 0);
            all(0, 2);
            all(1, 1);
            all(1, 0);
        } else {
            all(0, 2);
        }
        all(0, 1);
        all(0, 0);
    }
}

// Weights of the running total (M) and of the next group (m); the total is
// scaled by a and the group added with b.
__device__ __forceinline__ float merge_weights(float M, float m, float& a, float& b) {
    const float mn = fmaxf(M, m);
    a = M == -INFINITY ? 0.0f : exp2_sm(M - mn);
    b = m == -INFINITY ? 0.0f : exp2_sm(m - mn);
    return mn;
}
__device__ __forceinline__ float merge_value(float X, float x, float a, float b) { return fmaf(X, a, x * b); }

// Where a tile's queries, keys and outputs are.
template <int D, typename KV, int LAYOUT, int PAGE>
struct Where {
    TokenMap<LAYOUT, PAGE> map{};
    const KV *kbase, *vbase;
    const float* Q;
    float* O;
    int P, H_q, h, b, start, causal, nkeys;

    __device__ __forceinline__ size_t qrow(int qi) const {
        return LAYOUT == 0 ? (((size_t)b * P + qi) * H_q + h) * D : (((size_t)b * H_q + h) * P + qi) * D;
    }
    // keys that queries up to qi need
    __device__ __forceinline__ int limit(int qi) const { return causal ? min(start + qi + 1, nkeys) : nkeys; }
    __device__ __forceinline__ int phys(int pos, int kend) const {
        if constexpr (LAYOUT == 0 && PAGE) return map.run_of(min(pos, kend - 1));
        else return 0;
    }
};

template <int D, typename KV, int LAYOUT, int PAGE>
__device__ __forceinline__ Where<D, KV, LAYOUT, PAGE> locate(const float* Q, const KV* kcache, const KV* vcache,
                                                             const int* block_table, int nbps, int block_size, int P,
                                                             int H_q, int H_kv, int start, int causal, float* O, int h,
                                                             int b) {
    Where<D, KV, LAYOUT, PAGE> w;
    const int kvh = h / (H_q / H_kv);
    if constexpr (LAYOUT == 0) {
        w.map.bt = block_table + (size_t)b * nbps;
        w.map.block_size = block_size;
        w.map.run_log = 27 - __builtin_clz(block_size);
        w.map.stride = (size_t)H_kv * D;
        w.kbase = kcache + (size_t)kvh * D;
        w.vbase = vcache + (size_t)kvh * D;
    } else {
        w.map.stride = D;
        w.kbase = kcache + ((size_t)b * H_kv + kvh) * P * D;
        w.vbase = vcache + ((size_t)b * H_kv + kvh) * P * D;
    }
    w.Q = Q;
    w.O = O;
    w.P = P;
    w.H_q = H_q;
    w.h = h;
    w.b = b;
    w.start = start;
    w.causal = causal;
    w.nkeys = start + P;
    return w;
}

// 16 queries from q0 on with fp32 MFMAs, one wave over all their keys: the
// form for operands that have no three-part one.  Writes those of `rows` (bit
// i: query q0 + i).
template <int D, typename KV, int LAYOUT, int PAGE>
__device__ __forceinline__ void exact_tile(const Where<D, KV, LAYOUT, PAGE>& w, int q0, float qscale,
                                           uint32_t rows) {
    if (q0 >= w.P) return;
    const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
    const int qi = min(q0 + i, w.P - 1);
    const int kend = w.limit(min(q0 + 15, w.P - 1)), klim = w.limit(qi);
    float q[D / 4];
#pragma unroll
    for (int e = 0; e < D / 4; e += 4) {
        const float4 v = *reinterpret_cast<const float4*>(w.Q + w.qrow(qi) + (D / 4) * g + e);
        q[e] = v.x * qscale;
        q[e + 1] = v.y * qscale;
        q[e + 2] = v.z * qscale;
        q[e + 3] = v.w * qscale;
    }
    float m = -INFINITY, l = 0.0f;
    f32x4 o[D / 16];
#pragma unroll
    for (int t = 0; t < D / 16; ++t) o[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
    for (int c0 = 0; c0 < kend; c0 += 16) {
        Chunk<D, KV> c;
        load_chunk(c, c0, kend, i, g, w.phys(c0, kend), w.map, w.kbase, w.vbase);
        consume(c, c0, g, q, klim, m, l, o);
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    if (q0 + i < w.P && (rows >> i & 1)) {
        float* out = w.O + w.qrow(qi);
#pragma unroll
        for (int t = 0; t < D / 16; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) out[(D / 16) * (4 * g + v) + t] = o[t][v] * inv;
    }
}

// The queries (bit i) that have a lane (i, g) among `lanes`.
__device__ __forceinline__ uint32_t query_rows(uint64_t lanes) {
    const uint32_t x = (uint32_t)lanes | (uint32_t)(lanes >> 32);
    return (x | x >> 16) & 0xffffu;
}

// A lane's share of its query's row: elements 32 s + 8 g on.
template <int D>
__device__ __forceinline__ void load_query(const float* row, int g, float (&x)[D / 32][8]) {
#pragma unroll
    for (int s = 0; s < D / 32; ++s) {
        const float4 a = *reinterpret_cast<const float4*>(row + 32 * s + 8 * g);
        const float4 b = *reinterpret_cast<const float4*>(row + 32 * s + 8 * g + 4);
        const float y[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) x[s][e] = y[e];
    }
}

// The query's operand; whether one of the lane's elements has no three-part
// form that serves: a non-zero one below 2^-98 (2^-102 with qscale, about 1/8),
// whose parts bf16 may not hold (what they lose is below 2^-133 and counts
// beside keys of 2^64 and more), or one from 2^64 on, beside which what tiny
// keys lose counts.
template <int D>
__device__ __forceinline__ bool split_query(const float (&x)[D / 32][8], float qscale, Parts<3> (&q)[D / 32]) {
    float lo = INFINITY, hi = 0.0f;
#pragma unroll
    for (int s = 0; s < D / 32; ++s) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            lo = fminf(lo, fabsf(x[s][e]));
            hi = fmaxf(hi, fabsf(x[s][e]));
        }
        q[s] = split8(x[s], qscale);
    }
    bool bad = false;
    if (__ballot(lo < 0x1p-98f || hi >= 0x1p64f)) {  // (uniform; seldom, zeros among them)
#pragma unroll
        for (int s = 0; s < D / 32; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                bad |= x[s][e] != 0.0f && !(fabsf(x[s][e]) >= 0x1p-98f && fabsf(x[s][e]) < 0x1p64f);
    }
    return bad;
}

// Rows of a block's keys for a lane.  With pages of 2^n 16-token runs and
// contiguous rows key r of half j of a block at c0 lies at a uniform base (of
// the run, or of the half) plus r rows, so an address is a scalar base plus a
// 32-bit lane offset; other block sizes look each key up.  Keys at or past kend read the
// last one.
template <typename KV, int LAYOUT, int PAGE>
struct BlockRows {
    const TokenMap<LAYOUT, PAGE>& map;
    const KV* base;  // the head's rows
    const KV *half0, *half1;
    int c0, kend;
    __device__ __forceinline__ BlockRows(const TokenMap<LAYOUT, PAGE>& m, const KV* b, int c0_, int kend_)
        : map(m), base(b), c0(c0_), kend(kend_) {
        half0 = start_of(c0);
        half1 = start_of(min(c0 + 16, (kend - 1) & ~15));  // (past the end: its keys read the first half's last)
    }
    __device__ __forceinline__ const KV* start_of(int pos) const {
        if constexpr (LAYOUT == 1) return base + (size_t)pos * map.stride;
        else if constexpr (PAGE) return base + (size_t)map.run_of(pos) * 16 * map.stride;
        else return base;
    }
    // elements `elem` on of key 16 j + r (r < 16); j uniform
    __device__ __forceinline__ const KV* at(int j, int r, int elem) const {
        if constexpr (LAYOUT == 0 && !PAGE) {
            return base + map.off(min(c0 + 16 * j + r, kend - 1), 0) + elem;
        } else {
            const int pos = min(c0 + 16 * j, (kend - 1) & ~15);
            // (16 rows are at most 2^32 bytes: launch_d)
            const uint32_t ofs = ((uint32_t)min(r, kend - 1 - pos) * (uint32_t)map.stride + elem) * (uint32_t)sizeof(KV);
            return reinterpret_cast<const KV*>(reinterpret_cast<const char*>(j ? half1 : half0) + ofs);
        }
    }
};

// LAYOUT 0: Q/O [B, P, H_q, D], keys = start + P cached tokens.
// LAYOUT 1: Q/K/V/O [B, H, P, D], keys = P, start = 0.
template <int D, typename KV, int LAYOUT, int PAGE, int GW>
__global__ __launch_bounds__(256 * GW, D != 64 ? 2 : sizeof(KV) == 2 ? 4 : GW == 1 ? 3 : 2) void prefill_tile_kernel(
    const float* __restrict__ Q, const KV* __restrict__ kcache, const KV* __restrict__ vcache,
    const int* __restrict__ block_table, int nbps, int block_size, int P, int H_q, int H_kv,
    int start, int causal, float qscale, float* __restrict__ O) {
    constexpr int NP = kParts<KV>, QT = kWaves * kQW, T = 256;
    constexpr int CK = D / 8;                   // 16-byte chunks of a K row
    constexpr int KBYTES = kKB * D * 2;         // one part of a block's K (or V)
    constexpr int HBYTES = 2 * NP * KBYTES;     // K and V of a block
    constexpr int KT = kKB * CK / T;            // K chunks per thread
    constexpr int VE = 8 * D / T;               // V: elements per thread, of four keys
    constexpr int KW = 4 * (int)sizeof(KV) / 2, VW = VE * (int)sizeof(KV) / 4;  // raw words
    constexpr int TT = D / 16;
    // (the merge passes two states per lane of four waves through it)
    constexpr int MBYTES = GW == 1 ? 0 : 2 * kWaves * 64 * (TT * 16 + 8), PER = kGroups / GW;
    __shared__ __attribute__((aligned(16))) int8_t lds_all[GW * HBYTES > MBYTES ? GW * HBYTES : MBYTES];
    const int lane = threadIdx.x & 63, g = lane >> 4, i = lane & 15;
    const int wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hf = GW == 1 ? 0 : wave8 >> 2, wave = wave8 & 3, tid = threadIdx.x & (T - 1);
    int8_t* lds = lds_all + hf * HBYTES;
    const int ntiles = (P + QT - 1) / QT;
    const int pairs = (int)(gridDim.x / (unsigned)ntiles);  // H_q B
    const int r = (int)blockIdx.x / pairs, pr = (int)blockIdx.x - r * pairs;
    const int q0 = (ntiles - 1 - r) * QT;  // longest (last) tiles first
    const auto w = locate<D, KV, LAYOUT, PAGE>(Q, kcache, vcache, block_table, nbps, block_size, P, H_q, H_kv, start,
                                               causal, O, pr % H_q, pr / H_q);
    const int kend = w.limit(min(q0 + QT - 1, P - 1));
    const int nblk = (kend + kKB - 1) / kKB;
    const int qw = q0 + wave * kQW, qi = min(qw + i, P - 1);
    const int klim = w.limit(qi);
    const int wlo = w.limit(min(qw, P - 1)), whi = qw < P ? w.limit(min(qw + kQW - 1, P - 1)) : 0;  // uniform

    // The thread's raw share of a block, and its way into LDS: K chunks of
    // eight elements; V, VE elements of keys 16 vj + 4 vo .. + 3 (half vj of
    // octet vo).
    uint32_t kr[KT][KW], vr[4][VW];
    const int vj = wave & 1, vo = 2 * (wave >> 1) + (lane >> 5), ve = (lane & 31) * VE;
    auto load = [&](int blk) {
        const int c0 = blk * kKB;
        const BlockRows<KV, LAYOUT, PAGE> kb(w.map, w.kbase, c0, kend), vb(w.map, w.vbase, c0, kend);
#pragma unroll
        for (int j = 0; j < KT; ++j) {
            const int id = tid + T * j, key = id / CK, c = id % CK;
            load_words(kb.at(__builtin_amdgcn_readfirstlane(key >> 4), key & 15, 8 * c), kr[j]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) load_words(vb.at(vj, 4 * vo + e, ve), vr[e]);
    };
    auto k_at = [&](int part, int key, int c) {
        return reinterpret_cast<uint4*>(lds + part * KBYTES + key * (2 * D) +
                                        ((c ^ (D == 128 ? key & 15 : (key >> 1) & 7)) << 4));
    };
    auto v_at = [&](int part, int e, int c) {
        return lds + (NP + part) * KBYTES + e * (2 * kKB) + ((c ^ ((e >> 2) & 3)) << 4);
    };
    auto store = [&] {
#pragma unroll
        for (int j = 0; j < KT; ++j) {
            const int id = tid + T * j, key = id / CK, c = id % CK;
            const Parts<NP> s = parts8<KV>(kr[j]);
#pragma unroll
            for (int p = 0; p < NP; ++p) *k_at(p, key, c) = s.p[p];
        }
#pragma unroll
        for (int d = 0; d < VE; ++d) {
            uint2 s[NP];
            if constexpr (NP == 3) {
                split_pair(elem<KV>(vr[0], d), elem<KV>(vr[1], d), kUp, s[0].x, s[1].x, s[2].x);
                split_pair(elem<KV>(vr[2], d), elem<KV>(vr[3], d), kUp, s[0].y, s[1].y, s[2].y);
            } else {
                s[0] = make_uint2(pair_bf16(vr[0][d / 2], vr[1][d / 2], d & 1), pair_bf16(vr[2][d / 2], vr[3][d / 2], d & 1));
            }
#pragma unroll
            for (int p = 0; p < NP; ++p) *reinterpret_cast<uint2*>(v_at(p, ve + d, vo) + 8 * vj) = s[p];
        }
    };

    // These four waves' steps: groups PER hf .. PER hf + PER - 1, a block at a time.
    int grp = PER * hf, blk = grp;
    bool act = blk < nblk;
    float qx[D / 32][8];
    load_query<D>(Q + w.qrow(qi), g, qx);
    if (act) load(blk);
    auto steps = [&](int k) { return k < nblk ? (nblk - k + kGroups - 1) / kGroups : 0; };
    int iters = 0;  // (the second half has no more than the first)
#pragma unroll
    for (int k = 0; k < PER; ++k) iters += steps(k);
    Parts<3> q[D / 32];
    const bool qbad = split_query<D>(qx, qscale, q);
    Group<D> gr, tot;
    gr.clear();
    tot.clear();
    auto merge = [&](const Group<D>& x) {
        float a, b;
        tot.m = merge_weights(tot.m, x.m, a, b);
        tot.l = merge_value(tot.l, x.l, a, b);
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) tot.o[t][v] = merge_value(tot.o[t][v], x.o[t][v], a, b);
    };
#pragma unroll 1
    for (int it = 0; it < iters; ++it) {
        const int c0 = blk * kKB, cg = grp;
        const bool cact = act, gend = blk + kGroups >= nblk;
        __syncthreads();  // the last block has been read
        if (cact) store();
        __syncthreads();
        blk = gend ? ++grp : blk + kGroups;
        act = act && grp < PER * hf + PER && blk < nblk;
        if (act) load(blk);
        if (!cact) continue;
        if (c0 < whi) {
            float sc[8];
            scores<D, NP>(
                [&](int j, int s) {
                    Parts<NP> x;
#pragma unroll
                    for (int p = 0; p < NP; ++p) x.p[p] = *k_at(p, 16 * j + i, 4 * s + g);
                    return x;
                },
                q, c0, klim, c0 + kKB > wlo, g, sc);
            attend<D, NP>(
                [&](int t) {
                    Parts<NP> x;
#pragma unroll
                    for (int p = 0; p < NP; ++p) x.p[p] = *reinterpret_cast<uint4*>(v_at(p, 16 * t + i, g));
                    return x;
                },
                sc, gr);
        }
        // into the total in order; of GW = 2's second half, group 2 into its
        // own (empty, so it is kept as it is) and 3 stays in gr
        if (gend && (GW == 1 || cg < 3)) {
            merge(gr);
            gr.clear();
        }
    }
    if constexpr (GW == 2) {
    // Groups 2 and 3 from the second half, in order.
    __syncthreads();
    float4* mo = reinterpret_cast<float4*>(lds_all);
    float2* ml = reinterpret_cast<float2*>(lds_all + 2 * kWaves * 64 * TT * 16);
    auto slot = [&](int k) { return (k * kWaves + wave) * 64 + lane; };
    if (hf == 1) {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            mo[t * (2 * kWaves * 64) + slot(0)] = make_float4(tot.o[t][0], tot.o[t][1], tot.o[t][2], tot.o[t][3]);
            mo[t * (2 * kWaves * 64) + slot(1)] = make_float4(gr.o[t][0], gr.o[t][1], gr.o[t][2], gr.o[t][3]);
        }
        ml[slot(0)] = make_float2(tot.m, tot.l);
        ml[slot(1)] = make_float2(gr.m, gr.l);
    }
    __syncthreads();
    if (hf == 1) return;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const float2 x = ml[slot(k)];
        gr.m = x.x;
        gr.l = x.y;
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const float4 y = mo[t * (2 * kWaves * 64) + slot(k)];
            gr.o[t] = f32x4{y.x, y.y, y.z, y.w};
        }
        merge(gr);
    }
    }

    const float inv = tot.l > 0.0f ? 1.0f / tot.l * kDown<KV> : 0.0f;
    float bad = qbad ? 1.0f : 0.0f;
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            tot.o[t][v] *= inv;
            bad = fmaf(tot.o[t][v], 0.0f, bad);
        }
    const uint32_t rows = query_rows(__ballot(!(bad == 0.0f)));  // not all finite, or without parts
    if (qw + i < P && !(rows >> i & 1)) {
        float* out = O + w.qrow(qi) + 4 * g;
#pragma unroll
        for (int t = 0; t < TT; ++t)
            *reinterpret_cast<float4*>(out + 16 * t) = make_float4(tot.o[t][0], tot.o[t][1], tot.o[t][2], tot.o[t][3]);
    }
    if (rows) exact_tile(w, qw, qscale, rows);
}

template <int D, typename KV, int LAYOUT, int PAGE>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void prefill_split_kernel(
    const float* __restrict__ Q, const KV* __restrict__ kcache, const KV* __restrict__ vcache,
    const int* __restrict__ block_table, int nbps, int block_size, int P, int H_q, int H_kv,
    int start, int causal, float qscale, float* __restrict__ O) {
    constexpr int NP = kParts<KV>;
    constexpr int KW = 4 * (int)sizeof(KV) / 2;       // raw words of eight elements
    constexpr int VW = D / 16 * (int)sizeof(KV) / 4;  // of d / 16
    __shared__ float sm_o[kGroups][kQW][D + 4];
    __shared__ float sm_m[kGroups][kQW], sm_l[kGroups][kQW];
    __shared__ uint32_t sm_bad;  // queries without parts
    const int lane = threadIdx.x & 63, g = lane >> 4, i = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // its group
    const int ntiles = (P + kQW - 1) / kQW;
    const int pairs = (int)(gridDim.x / (unsigned)ntiles);  // H_q B
    const int r = (int)blockIdx.x / pairs, pr = (int)blockIdx.x - r * pairs;
    const int q0 = (ntiles - 1 - r) * kQW;  // longest (last) tiles first
    const auto w = locate<D, KV, LAYOUT, PAGE>(Q, kcache, vcache, block_table, nbps, block_size, P, H_q, H_kv, start,
                                               causal, O, pr % H_q, pr / H_q);
    const int kend = w.limit(min(q0 + kQW - 1, P - 1));
    const int qi = min(q0 + i, P - 1);
    const int klim = w.limit(qi), wlo = w.limit(q0);

    // K: elements 32 s + 8 g .. of key 16 j + i; V: elements d/16 i .. of the
    // keys of octet g.
    uint32_t kr[2][D / 32][KW], vr[8][VW];
    auto load_k = [&](int c0) {
        const BlockRows<KV, LAYOUT, PAGE> kb(w.map, w.kbase, c0, kend);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int s = 0; s < D / 32; ++s) load_words(kb.at(j, i, 32 * s + 8 * g), kr[j][s]);
    };
    auto load_v = [&](int c0) {
        const BlockRows<KV, LAYOUT, PAGE> vb(w.map, w.vbase, c0, kend);
#pragma unroll
        for (int e = 0; e < 8; ++e) load_words(vb.at(e >> 2, 4 * g + (e & 3), D / 16 * i), vr[e]);
    };

    // (a wave without blocks has nothing to do here; in one branch, so that no
    // wait is for more than the path has issued)
    if (int c0 = wave * kKB; c0 < kend) {
        // the query first: it waits for no block table, and is split while the keys arrive
        float qx[D / 32][8];
        load_query<D>(Q + w.qrow(qi), g, qx);
        load_k(c0);
        load_v(c0);
        Parts<3> q[D / 32];
        const bool qbad = split_query<D>(qx, qscale, q);
        if (wave == 0) sm_bad = query_rows(__ballot(qbad));  // (wave 0 has a block)
        Group<D> gr;
        gr.clear();
        while (c0 < kend) {
            const int cn = c0 + kGroups * kKB;
            float sc[8];
            scores<D, NP>([&](int j, int s) { return parts8<KV>(kr[j][s]); }, q, c0, klim, c0 + kKB > wlo, g, sc);
            if (cn < kend) load_k(cn);
            attend<D, NP>(
                [&](int t) {
                    if constexpr (NP == 3) {
                        const float x[8] = {elem<KV>(vr[0], t), elem<KV>(vr[1], t), elem<KV>(vr[2], t), elem<KV>(vr[3], t),
                                            elem<KV>(vr[4], t), elem<KV>(vr[5], t), elem<KV>(vr[6], t), elem<KV>(vr[7], t)};
                        return split8(x, kUp);
                    } else {
                        auto pair = [&](int e) { return pair_bf16(vr[e][t / 2], vr[e + 1][t / 2], t & 1); };
                        return Parts<1>{{make_uint4(pair(0), pair(2), pair(4), pair(6))}};
                    }
                },
                sc, gr);
            if (cn < kend) load_v(cn);
            c0 = cn;
        }
#pragma unroll
        for (int t = 0; t < D / 16; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) sm_o[wave][i][(D / 16) * (4 * g + v) + t] = gr.o[t][v];
        if (g == 0) {
            sm_m[wave][i] = gr.m;
            sm_l[wave][i] = gr.l;
        }
    }
    __syncthreads();

    constexpr int PER = kQW * D / 256;  // outputs per thread (4 or 8)
    const int qq = threadIdx.x / 16, col = (threadIdx.x % 16) * PER;
    float M = -INFINITY, L = 0.0f, x[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) x[e] = 0.0f;
#pragma unroll
    for (int k = 0; k < kGroups; ++k) {
        if (k * kKB >= kend) break;  // uniform: a group without blocks changes nothing
        float a, b;
        M = merge_weights(M, sm_m[k][qq], a, b);
        L = merge_value(L, sm_l[k][qq], a, b);
#pragma unroll
        for (int e = 0; e < PER; ++e) x[e] = merge_value(x[e], sm_o[k][qq][col + e], a, b);
    }
    const float inv = L > 0.0f ? 1.0f / L * kDown<KV> : 0.0f;
    float bad = 0.0f;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
        x[e] *= inv;
        bad = fmaf(x[e], 0.0f, bad);
    }
    // of this wave's four queries (16 lanes each): not all finite, or without parts
    const uint64_t lanes = __ballot(!(bad == 0.0f));
    uint32_t rows = __builtin_amdgcn_readfirstlane(sm_bad) & (0xfu << (4 * wave));
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (lanes >> (16 * k) & 0xffff) rows |= 1u << (4 * wave + k);
    if (q0 + qq < P && !(rows >> qq & 1)) {
        float* out = O + w.qrow(q0 + qq) + col;
#pragma unroll
        for (int e = 0; e < PER; e += 4) *reinterpret_cast<float4*>(out + e) = make_float4(x[e], x[e + 1], x[e + 2], x[e + 3]);
    }
    if (rows) exact_tile(w, q0, qscale, rows);
}

enum PrefillForm { kFp32, kSplit, kTile1, kTile2 };

// Measured on one box (us, graph-timed), split / GW = 1 / GW = 2 (/ fp32 MFMAs);
// tiles: of 64 queries.
// Paged bf16.  Few tiles take the split kernel (d 64: 1 x 512 x 8 heads 13.7 /
// 19.7 / 16.4 / 20.3 for 256 of them), and so do up to 16 queries, of which a tile
// would fill one wave in four (d 64, 1 query of 400 pairs after 800 tokens 20.2 /
// 27 / 31 / 28.6), and at d = 64, after more than 256 tokens, all that are one round
// of it (400 tiles of 32 queries after 800 26.7 / 33.2 / 31.4 / 46.0).  From 320 tiles
// on GW = 2 in one round of two per CU at d = 64 (384 of 40 queries after 2400 103 /
// 89.8 / 77.8; 528 of 200 after 300 24.5 / 25.6 / 29.3, and a little past it in long
// prompts, whose first tiles set the time: 528 of 700 25.6 / 27.0 / 22.8), at d = 128
// (one per CU) for those alone (384 of 1024 48.1 / 47.6 / 39.9; 384 of 64 after 300
// 51.0 / 30.2 / 38.8); else GW = 1, whose workgroups share a CU (d 64, 1024 tiles of 512
// 40.3 / 25.8 / 30.3).
// Contiguous fp32.  The tile kernels where they have the tiles (d 128: 4 x 512 x 32
// heads 146 -> 76 on GW = 1; 1 x 2048 x 16 heads 210 -> 127 on GW = 2, 161 on GW = 1).
// GW = 2 takes a CU per workgroup, so its second round must be worth it: causal
// d 128 from 256 tiles on (288 tiles of N = 1000 88.0 / 80.1 / 61.6 / 73.0; 192: 60.9 /
// 78.3 / 59.6 / 48.2), non-causal, twice the work, from 144 (168 of 1500 120 / 115 / 87 /
// 119; 130 of 800 55.0 / 64.2 / 49.8 / 47.5), d 64 from 384 (408 of 1500 62.3 / 76.2 / 53.5 /
// 63.0; 264 of 2100 55.1 / 102.4 / 72.7 / 61.5; non-causal 286 of 800 50.8 / 53.9 / 60.0 / 51.0),
// causal N < 1500 from 300 (403 of 800 44.8 / 42.5 / 33.4 / 41.2).  Below, the split
// kernel for a few long problems (d 128: 96 tiles of 1000 35.4 / 78.0 / 58.9 / 40.1,
// non-causal 59.5 / 80.2 / 60.3 / 54.6; 40 of 600 22.8 / 48.2 / 38.6 / 23.7, 28 of 420 19.4 /
// 37.5 / 31.1 / 17.9) and at d 64 for any number of long ones (188 of 3000
// 60.4 / 142.7 / 100.3 / 69.9), the fp32 kernel for the rest, whose launches are over
// before the splitting pays.
PrefillForm prefill_form(const PrefillArgs& a) {
    const long long tiles = (long long)((a.P + kWaves * kQW - 1) / (kWaves * kQW)) * a.H_q * a.B;
    const int keys = a.start_pos + a.P;
    if (a.paged) {
        if (a.kv_dtype != IE_KV_BF16) return kFp32;
        if (a.P <= kQW || tiles < 320) return kSplit;
        if (a.d == 128) return a.P >= 512 && a.start_pos <= a.P / 3 && tiles <= 512 ? kTile2 : kTile1;
        if (keys <= 256) return kTile1;
        if ((long long)((a.P + kQW - 1) / kQW) * a.H_q * a.B <= 960) return kSplit;
        return tiles <= (a.P >= 512 ? 576 : 512) ? kTile2 : kTile1;
    }
    if (tiles >= (keys <= 768 ? 512 : 1024)) return kTile1;
    if (keys < 768) return a.d == 128 && keys >= 576 && tiles <= 64 ? kSplit : kFp32;
    if (a.d == 64) {
        if (tiles >= (a.causal && keys < 1500 ? 300 : 384)) return kTile2;
        return tiles <= 128 || keys >= 1500 ? kSplit : kFp32;
    }
    if (tiles >= (a.causal ? 256 : 144)) return kTile2;
    return tiles <= (a.causal ? 128 : 64) ? kSplit : kFp32;
}

template <int D, typename KV, int LAYOUT, int PAGE>
void launch_t(const PrefillArgs& a, hipStream_t s) {
    const float qscale = 1.4426950408889634f / sqrtf((float)D);
    const PrefillForm form = prefill_form(a);
    const int per = form == kTile1 || form == kTile2 ? kWaves * kQW : kQW;  // queries per workgroup
    const unsigned grid = (unsigned)((long long)((a.P + per - 1) / per) * a.H_q * a.B);
    auto* k = prefill_split_kernel<D, KV, LAYOUT, PAGE>;
    if (form == kTile1) k = prefill_tile_kernel<D, KV, LAYOUT, PAGE, 1>;
    if (form == kTile2) k = prefill_tile_kernel<D, KV, LAYOUT, PAGE, 2>;
    k<<<grid, form == kTile2 ? 512 : 256, 0, s>>>(a.Q, static_cast<const KV*>(a.k), static_cast<const KV*>(a.v),
                                                 a.block_table, a.num_blocks_per_seq, a.block_size, a.P, a.H_q, a.H_kv,
                                                 a.start_pos, a.causal ? 1 : 0, qscale, a.O);
}

template <int D, int LAYOUT, int PAGE>
void launch_fp32(const PrefillArgs& a, hipStream_t s) {
    const float qscale = 1.4426950408889634f / sqrtf((float)D);
    const unsigned grid = (unsigned)((long long)((a.P + kQW - 1) / kQW) * a.H_q * a.B);
    prefill_fp32_kernel<D, float, LAYOUT, PAGE><<<grid, 256, 0, s>>>(
        a.Q, static_cast<const float*>(a.k), static_cast<const float*>(a.v), a.block_table, a.num_blocks_per_seq,
        a.block_size, a.P, a.H_q, a.H_kv, a.start_pos, a.causal ? 1 : 0, qscale, a.O);
}

template <int D>
void launch_d(const PrefillArgs& a, hipStream_t s) {
    const bool fp32 = prefill_form(a) == kFp32;
    if (!a.paged) return fp32 ? launch_fp32<D, 1, 0>(a, s) : launch_t<D, float, 1, 0>(a, s);
    if (fp32) return a.block_size == 16 ? launch_fp32<D, 0, 1>(a, s) : launch_fp32<D, 0, 0>(a, s);
    // BlockRows: runs of 16 tokens, and 32-bit offsets inside one
    const bool narrow = 16ull * a.H_kv * D * sizeof(uint16_t) <= 1ull << 32;
    if (a.block_size == 16 && narrow)
        launch_t<D, uint16_t, 0, 1>(a, s);
    else if (a.block_size > 16 && (a.block_size & (a.block_size - 1)) == 0 && narrow)
        launch_t<D, uint16_t, 0, 2>(a, s);
    else
        launch_t<D, uint16_t, 0, 0>(a, s);
}

}  // namespace

void launch_prefill_attn(const PrefillArgs& a, hipStream_t s) {
    if (a.B == 0 || a.P == 0) return;
    if (a.d == 64)
        launch_d<64>(a, s);
    else
        launch_d<128>(a, s);
}

}  // namespace ie

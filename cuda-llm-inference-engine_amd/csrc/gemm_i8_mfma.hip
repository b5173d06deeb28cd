// gemm_i8_mfma.hip — INT8 GEMM on the gfx950 i8 matrix cores: the dispatch,
// and the kernel for widths and alignments that the copying kernels cannot
// take.
//
// Same result as the reference's K14 kernel (kernels/quantization/
// 14_int8_gemm.cu:65-170): exact int32 sum over K of int8 products, then the
// dequant epilogue.  The reference uses __dp4a with a 64x64 tile and a 4x4
// register tile; here the sum runs on v_mfma_i32_32x32x32_i8 (32x32 outputs,
// 32 K-bytes per instruction) with LDS-staged int8 tiles.
//
// The kernel here: rows at any 4-byte address (K % 4 == 0, K >= 16).  Direct
// copies into LDS want 16-byte aligned sources, so the operands pass through
// registers: a 256-thread workgroup (4 waves, 2x2, one 32x32 block each) owns
// a 64x64 tile of C; K advances 128 bytes per stage through two LDS buffers,
// and a stage's loads are issued two stages before they are written, so two
// stages are in flight per workgroup, with several workgroups per CU.  LDS
// rows are 128 bytes with chunk c of row r at slot c ^ ((r >> 1) & 7).  A
// chunk past the row's end is read as the row's last 16 bytes on both sides,
// and the A words already counted (all of them past K) are zeroed.
// Bound by its stages' memory latency; one thread per output, which took
// these before, read every row uncoalesced: M = 512, K = 1000, N = 3000 1513 ->
// 9.9 us, M = 100, K = N = 1000 104 -> 5.6.  It also takes K < 128, too short
// for a whole stage (M = N = 2048, K = 80: 13.6 us on 128x128 tiles, 6.9).
//
// MFMA operand convention: lane l supplies row (l % 32) of A and column
// (l % 32) of B, each with 16 K-bytes; A and B take the same K-bytes from the
// same lane, so the product is the full K-sum whatever order the hardware
// adds them in.  Accumulator v of lane l holds C[8*(v/4) + 4*(l/32) + v%4]
// [l % 32] of the 32x32 block.
#include <stdexcept>

#include "device_util.h"
#include "epilogue.h"
#include "ie_internal.h"

namespace ie {
namespace {

constexpr int BM = 64, BN = 64, BK = 128;
constexpr int CHUNKS = BK / 16;       // 16-byte chunks per LDS row
constexpr int OPER = BM * BK;         // bytes of one operand, one stage
constexpr int PER = OPER / 16 / 256;  // chunks of an operand per thread

__device__ __forceinline__ int slot_of(int row, int chunk) {
    return row * BK + ((chunk ^ ((row >> 1) & 7)) << 4);
}

template <int EPI>
__global__ __launch_bounds__(256) void gemm_i8_ragged_kernel(
    int M, int N, int K, const int8_t* __restrict__ A, const int8_t* __restrict__ BT,
    const float* __restrict__ sA, const float* __restrict__ sB, const float* bias,
    const float* residual, void* C) {
    typedef i32x4 i32x4_a4 __attribute__((aligned(4)));
    __shared__ __attribute__((aligned(16))) int8_t lds[2][2][OPER];  // [buffer][A, B]
    const int t = threadIdx.x, lane = t & 63;
    const int wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int nk = (K + BK - 1) / BK;

    // This thread's chunks: rows t / 8 + 32 j, chunk t % 8.
    const int crow = t / CHUNKS, cc = t % CHUNKS;
    const int8_t* pa[PER];
    const int8_t* pb[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        pa[j] = A + (size_t)min(m0 + crow + 32 * j, M - 1) * K;
        pb[j] = BT + (size_t)min(n0 + crow + 32 * j, N - 1) * K;
    }
    struct Regs {
        i32x4 a[PER], b[PER];
    };
    auto load = [&](Regs& r, int kt) {
        const int k = min(kt * BK + cc * 16, K - 16);
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            r.a[j] = *reinterpret_cast<const i32x4_a4*>(pa[j] + k);
            r.b[j] = *reinterpret_cast<const i32x4_a4*>(pb[j] + k);
        }
    };
    auto store = [&](const Regs& r, int kt) {
        const int over = kt * BK + cc * 16 + 16 - K;  // bytes of the chunk past K
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            i32x4 a = r.a[j];
#pragma unroll
            for (int w = 0; w < 4; ++w) a[w] = 4 * w < over ? 0 : a[w];
            *reinterpret_cast<i32x4*>(lds[kt & 1][0] + slot_of(crow + 32 * j, cc)) = a;
            *reinterpret_cast<i32x4*>(lds[kt & 1][1] + slot_of(crow + 32 * j, cc)) = r.b[j];
        }
    };

    i32x16 acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0;
    const int frow = lane & 31, fchunk = lane >> 5;
    // Stage kt from LDS while stages kt + 1 (in r) and kt + 2 are in flight;
    // kt + 1 goes into the other buffer, free since the last barrier.
    auto step = [&](Regs& r, int kt) {
        const int8_t* sa = lds[kt & 1][0];
        const int8_t* sb = lds[kt & 1][1];
#pragma unroll
        for (int ks = 0; ks < BK / 32; ++ks) {
            const i32x4 af = *reinterpret_cast<const i32x4*>(sa + slot_of(wm * 32 + frow, ks * 2 + fchunk));
            const i32x4 bf = *reinterpret_cast<const i32x4*>(sb + slot_of(wn * 32 + frow, ks * 2 + fchunk));
            acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, bf, acc, 0, 0, 0);
        }
        if (kt + 1 < nk) store(r, kt + 1);
        load(r, kt + 3);  // past the last stage: its last chunks again, never stored
        __syncthreads();
    };
    Regs r0, r1;
    load(r0, 0);
    load(r1, 1);
    store(r0, 0);
    load(r0, 2);
    __syncthreads();
    for (int kt = 0; kt < nk; kt += 2) {
        step(r1, kt);
        if (kt + 1 >= nk) break;
        step(r0, kt + 1);
    }

    // Every operand the stores need first (clamped indices), as in
    // gemm_i8_tile.hip.
    const int rbase = m0 + wm * 32 + 4 * (lane >> 5);
    const int n = n0 + wn * 32 + (lane & 31), nc = min(n, N - 1);
    constexpr bool HAS_BIAS = EPI == IE_EPI_BIAS || EPI == IE_EPI_BIAS_GELU || EPI == IE_EPI_BIAS_RESIDUAL;
    constexpr bool HAS_RES = EPI == IE_EPI_BIAS_RESIDUAL;
    float sa[16] = {}, rv[16] = {}, sb = 0.0f, bv = 0.0f;
    auto row = [&](int v) { return rbase + 8 * (v >> 2) + (v & 3); };
    if constexpr (EPI != IE_EPI_I32) {
        sb = sB[nc];
        if constexpr (HAS_BIAS) bv = bias[nc];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int m = min(row(v), M - 1);
            sa[v] = sA[m];
            if constexpr (HAS_RES) rv[v] = residual[(size_t)m * N + nc];
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            asm volatile("" ::"v"(sa[v]));
            if constexpr (HAS_RES) asm volatile("" ::"v"(rv[v]));
        }
        asm volatile("" ::"v"(sb));
        if constexpr (HAS_BIAS) asm volatile("" ::"v"(bv));
    }
    if (n < N) {
#pragma unroll
        for (int v = 0; v < 16; ++v)
            if (row(v) < M) store_epilogue_v<EPI>(C, (size_t)row(v) * N + n, acc[v], sa[v], sb, bv, rv[v]);
    }
}

template <int EPI>
struct RaggedLaunch {
    static void run(const GemmArgs& a, hipStream_t s) {
        const dim3 grid((a.N + BN - 1) / BN, (a.M + BM - 1) / BM);
        gemm_i8_ragged_kernel<EPI><<<grid, 256, 0, s>>>(
            a.M, a.N, a.K, reinterpret_cast<const int8_t*>(a.A),
            reinterpret_cast<const int8_t*>(a.BT), a.sA, a.sB, a.bias, a.residual, a.C);
    }
};

}  // namespace

void launch_gemm_i8_qkv_route(const GemmArgs& a, hipStream_t s) {
    if (a.M == 0 || a.N == 0) return;
    if (gemm_i8_stream_applies(a))
        launch_gemm_i8_stream(a, s);
    else if (gemm_i8_tile_applies(a))
        launch_gemm_i8_tile(a, s);
    else
        throw std::logic_error("launch_gemm_i8_qkv_route: K % 128 != 0 or unaligned operands");
}

void launch_gemm_i8_mfma(const GemmArgs& a, hipStream_t s) {
    if (a.M == 0 || a.N == 0) return;
    const bool vec = (a.K % 16) == 0 && ((uintptr_t)a.A % 16) == 0 && ((uintptr_t)a.BT % 16) == 0;
    if (!vec || a.K < 128) {
        // K < 16, a few short rows, or more 64-row tiles than a grid has in y: one
        // thread per output
        if (a.K >= 16 && (vec || !short_ragged_rows(a)) && (a.M + BM - 1) / BM <= 65535)
            dispatch_epilogue<RaggedLaunch>(a.epi, a, s);
        else
            launch_gemm_i8_generic(a, s);
        return;
    }
    if (gemm_i8_wide_applies(a)) {
        launch_gemm_i8_wide(a, s);
        return;
    }
    if (gemm_i8_big_applies(a)) {
        launch_gemm_i8_big(a, s);
        return;
    }
    // Small grids (one round of 32 x 32 blocks): the K-split kernel that
    // streams each block's K through per-wave LDS rings.
    if (gemm_i8_stream_applies(a)) {
        launch_gemm_i8_stream(a, s);
        return;
    }
    // Prefill-sized problems: the multi-stage LDS tile kernel (M = 2048:
    // 22.1 -> 12.1 us at N = 2304, 37.7 -> 13.0 us at K = 3072, N = 768;
    // at par with or ahead of hipBLASLt on the same shapes).
    if (gemm_i8_tile_applies(a))
        launch_gemm_i8_tile(a, s);
    else
        dispatch_epilogue<RaggedLaunch>(a.epi, a, s);
}

}  // namespace ie

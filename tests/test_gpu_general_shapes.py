"""Widths and alignments that no kernel is specialised for, through the public
entry points: the kernels that take K, N and the operands' alignment at run
time, at the sizes where their tiles, slices and last chunks end."""
import numpy as np
import pytest

from conftest import bf16_bits, pack_i8, rng

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _padded(a, words):
    """The int8 matrix as device words that start `words` words past a 256-byte boundary, 0x7f bytes on both sides (a
    read past a row's end would show in the sums)."""
    import torch

    flat = pack_i8(a).reshape(-1)
    buf = torch.full((words + flat.size + 64,), 0x7F7F7F7F, dtype=torch.int32, device="cuda")
    buf[words:words + flat.size] = torch.from_numpy(flat)
    return buf[words:words + flat.size].view(a.shape[0], -1)


def _gemm_case(ie, orc, M, N, K, epi, words, seed):
    r = rng(seed)
    A = r.integers(-128, 128, (M, K), dtype=np.int64).astype(np.int8)
    B = r.integers(-128, 128, (N, K), dtype=np.int64).astype(np.int8)
    Ap, Bp = _padded(A, words), _padded(B, words)
    if epi == ie.EPI_I32:
        got = ie.int8_gemm(Ap, Bp, epilogue=epi).cpu().numpy()
        assert np.array_equal(got, orc.gemm_i32(pack_i8(A), pack_i8(B)))
        return
    sA, sB = (r.uniform(1e-3, 1e-2, n).astype(np.float32) for n in (M, N))
    bias = r.standard_normal(N).astype(np.float32)
    res = r.standard_normal((M, N)).astype(np.float32)
    out = _dev(res)  # the residual in place
    got = ie.int8_gemm(Ap, Bp, _dev(sA), _dev(sB), epi, _dev(bias) if epi else None, out if epi == 3 else None,
                       out if epi == 3 else None).cpu().numpy()
    want = orc.gemm(pack_i8(A), pack_i8(B), sA, sB, epi, bias if epi else None, res if epi == 3 else None)
    if epi == ie.EPI_BIAS_GELU:  # the oracle's 1 + tanhf cancels where tanhf nears -1: an error of up to 1.2e-7 |v|
        v = orc.gemm(pack_i8(A), pack_i8(B), sA, sB, ie.EPI_BIAS, bias, None)
        assert (np.abs(got - want) <= 2e-6 * np.abs(want) + 1.2e-7 * np.abs(v)).all()
    else:
        assert np.array_equal(got, want)


# Decode rows.  K: one 16-byte chunk, a straddling chunk (K % 16 != 0) in a first, middle and last step, just past a
# 256-byte step, and slices of uneven length; N: one feature, a partial 4-feature item, fewer items than workgroups,
# several items per wave; M: one, two and four blocks of activation rows, each full and partial.
@pytest.mark.parametrize("K,N,words", [(16, 5, 0), (20, 1, 1), (252, 33, 0), (260, 1030, 1), (1000, 515, 3),
                                       (1040, 4099, 0), (2176, 500, 0), (4096, 9, 0), (4100, 4097, 1), (8188, 301, 0),
                                       (1536, 9001, 0), (3072, 4100, 0), (8192, 700, 0), (768, 4099, 2)])
@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 9, 16])
def test_gemv_any_width(ie, orc, M, K, N, words):
    _gemm_case(ie, orc, M, N, K, ie.EPI_I32, words, 3 * M + K + N)


@pytest.mark.parametrize("M,K,N,words", [(1, 1000, 1030, 1), (6, 2176, 501, 0), (16, 4096, 1027, 0), (16, 10176, 37, 0)])
@pytest.mark.parametrize("epi", [0, 1, 2, 3])
def test_gemv_any_width_epilogues(ie, orc, epi, M, K, N, words):
    _gemm_case(ie, orc, M, N, K, epi, words, M + K + N + epi)


# Prompt rows.  K % 16 == 0: the small-grid kernel (one and two 128-byte groups), the 64x64 and 128x64 LDS tiles (two to
# four stages) and the 256x256 tiles (two and an odd number of stages, a second tile per workgroup), each with a last
# stage that repeats 16 to 112 bytes.  K % 16 != 0, K < 128 or 4-byte aligned rows: the register-staged kernel, whose
# last chunk straddles K (K = 20: the only one), with one to eight stages.
@pytest.mark.parametrize("M,K,N,words", [(40, 144, 700, 0), (17, 240, 33, 0), (40, 8176, 200, 0), (1200, 272, 1100, 0),
                                         (700, 1616, 1000, 0), (2100, 400, 2200, 0), (2100, 2064, 2200, 0),
                                         (2900, 272, 3000, 0), (4352, 400, 4352, 0), (17, 16, 5, 0), (17, 20, 9, 1),
                                         (64, 124, 64, 0), (65, 132, 65, 0), (130, 1000, 700, 3), (300, 768, 301, 1),
                                         (257, 80, 129, 0)])
def test_gemm_any_width(ie, orc, M, K, N, words):
    _gemm_case(ie, orc, M, N, K, ie.EPI_I32, words, M + K + N)


@pytest.mark.parametrize("M,K,N,words", [(33, 208, 701, 0), (1200, 272, 1099, 0), (2100, 144, 2200, 0), (2900, 144, 3001, 0),
                                         (130, 140, 131, 1)])
@pytest.mark.parametrize("epi", [0, 1, 2, 3])
def test_gemm_any_width_epilogues(ie, orc, epi, M, K, N, words):
    _gemm_case(ie, orc, M, N, K, epi, words, M + K + N + epi)


# Rows of more than 4096 columns: 512 threads with the row in registers up to 8192 and 16384 columns (a partial and a
# full last chunk on both sides of each limit), two passes beyond, and an input past the size that is read
# non-temporally.
@pytest.mark.parametrize("rows,cols", [(3, 4100), (2, 8188), (5, 8192), (2, 8196), (3, 16384), (2, 16388), (4100, 8192)])
def test_quantize_wide_rows(ie, orc, rows, cols):
    r = rng(rows + cols)
    x = r.standard_normal((rows, cols)).astype(np.float32)
    x[0, -4:] = [127.0, -126.5, 0.5, -1.5]  # the row's maximum in its last chunk; ties
    x[1] = 0.0
    p, s = (t.cpu().numpy() for t in ie.quantize(_dev(x)))
    want_p, want_s = orc.quantize(x)
    assert np.array_equal(s, want_s) and np.array_equal(p, want_p)


# Paged cache writes.  Rows of whole float4s (one, a partial workgroup, exactly one, several), rows that are not
# (H dh % 4 != 0), and buffers that start one element into a 16-byte chunk; the first position inside a page.
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("seq,start,H,dh,bs,skew", [(1, 0, 1, 4, 16, 0), (7, 5, 3, 20, 4, 0), (33, 15, 16, 64, 16, 0),
                                                    (3, 2, 20, 128, 5, 0), (9, 30, 3, 5, 16, 0), (20, 3, 12, 64, 8, 1),
                                                    (2, 1, 24, 96, 16, 2)])
def test_kv_write_rows(ie, seq, start, H, dh, bs, skew, bf16):
    import torch

    r = rng(seq + H + dh)
    P = (start + seq + bs - 1) // bs + 2
    table = r.permutation(P).astype(np.int32)
    K, V = (r.standard_normal((seq, H, dh)).astype(np.float32) for _ in range(2))
    K.reshape(-1)[:4] = [np.inf, -np.inf, -0.0, 1e-40]

    def skewed(a):
        buf = torch.zeros(a.size + skew, dtype=torch.float32, device="cuda")
        buf[skew:] = torch.from_numpy(a.reshape(-1))
        return buf[skew:].view(seq, H, dh)

    def cache():
        n = P * bs * H * dh
        return torch.full((n + skew,), -7, dtype=torch.int16 if bf16 else torch.int32, device="cuda")[skew:].view(
            P, bs, H, dh)

    kc, vc = cache(), cache()
    ie.kv_cache_write(skewed(K), skewed(V), kc, vc, _dev(table), start, bs, kv_dtype=ie.KV_BF16 if bf16 else ie.KV_F32)
    for src, c in ((K, kc), (V, vc)):
        bits = bf16_bits(src).view(np.int16) if bf16 else src.view(np.int32)
        want = np.full((P, bs, H, dh), -7, bits.dtype)
        pos = start + np.arange(seq)
        want[table[pos // bs], pos % bs] = bits
        assert np.array_equal(c.cpu().numpy(), want)


# Rows of at most 64 float4s share a workgroup: a power of two of them, one short of and past one, tokens that fill a
# workgroup and a last one that is partial.
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("seq,start,H,dh,bs", [(255, 3, 1, 4, 16), (257, 0, 1, 12, 16), (70, 15, 1, 64, 8), (33, 1, 2, 66, 16),
                                               (5, 2, 2, 128, 16), (9, 2, 1, 260, 16), (129, 7, 2, 20, 5)])
def test_kv_write_narrow_rows(ie, seq, start, H, dh, bs, bf16):
    test_kv_write_rows(ie, seq, start, H, dh, bs, 0, bf16)


def _key_order(row):
    """Indices by the float's order key (a NaN past the infinity of its sign), descending, lower index first."""
    b = row.view(np.uint32).copy()
    b[b == 0x80000000] = 0
    key = np.where(b & 0x80000000, ~b, b | 0x80000000).astype(np.uint32)
    return np.argsort(-key.astype(np.int64), kind="stable")


# Top-k.  n: fewer than 256 + 4 logits (no wave whose lanes all hold a chunk), one such wave, 15 and 16; k on both sides
# of four per full wave, and where the gathered keys pass the 2048 that are ranked; the maxima in one thread's or one
# wave's chunks (the bound lets every key through); rows mostly -inf; rows that hold NaNs.
@pytest.mark.parametrize("n,k", [(4, 4), (259, 3), (260, 4), (260, 5), (3844, 60), (3844, 61), (4100, 64), (4099, 65),
                                 (4101, 512), (50257, 64), (50257, 65), (50257, 700), (65533, 1024), (8000, 16)])
def test_topk_bounds(ie, n, k):
    import torch

    r = rng(n + k)
    x = r.standard_normal((7, n)).astype(np.float32)
    x[1, :min(n, 64)] += 50  # the first chunks
    x[2, ::max(1, min(4096, n // 2))] += 50  # one thread's
    x[3, r.random(n) < 0.995] = -np.inf
    x[4] = np.round(x[4] * 2)
    x[5, r.integers(0, n, 3)] = np.nan
    x[6] = np.nan
    v, i = ie.topk(torch.from_numpy(x).cuda(), k)
    v, i = v.cpu().numpy(), i.cpu().numpy()
    for b in range(7):
        want = _key_order(x[b])[:k]
        assert np.array_equal(i[b], want), b
        assert np.array_equal(v[b], x[b][want], equal_nan=True), b


# Rows without a bound: fewer than 260 logits, k past the threads that hold any (2048 logits are ranked, more streamed).
@pytest.mark.parametrize("n,k", [(1, 1), (3, 3), (6, 2), (255, 64), (259, 1), (259, 259), (260, 65), (261, 66), (1000, 251),
                                 (2047, 1000), (2048, 512), (2048, 513), (2049, 513), (2050, 514), (3063, 1024), (4090, 1024)])
def test_topk_without_a_bound(ie, n, k):
    test_topk_bounds(ie, n, k)


# The language-model head at widths that are no multiple of 256 (or past 1280).  d: one float4, a partial chunk of 64, a
# whole one, either side of the chunks in flight (8 x 64, 4 x 64); rows at each padded count and either side; V: part of
# a tile, one and two vocabulary rows per wave (16384 on is the rule's line on 256 units), several tiles per wave; the
# last rows x d that is staged whole (16 x 2048) and the first that is not.
@pytest.mark.parametrize("d,V", [(4, 33), (60, 5), (64, 1027), (260, 2050), (516, 17001), (300, 50257), (1328, 999),
                                 (2044, 16383), (2048, 16385), (2052, 300), (4096, 77)])
def test_vocab_proj_any_width(ie, d, V):
    import torch

    r = rng(d + V)
    h = torch.from_numpy(r.standard_normal((16, d)).astype(np.float32)).cuda()
    w = torch.from_numpy((0.02 * r.standard_normal((V, d))).astype(np.float32)).cuda()
    one = torch.cat([ie.vocab_proj(h[i:i + 1].contiguous(), w) for i in range(16)])
    # chains of 4 ceil(d / 64) fused multiply-adds, then four additions: n roundings of at most 2^-24 each
    n = 4 * ((d + 63) // 64) + 4
    bound = n * 2.0 ** -24 * (h.double().abs() @ w.double().abs().t().contiguous())
    assert ((one.double() - h.double() @ w.double().t().contiguous()).abs() <= bound).all()
    for rows in (2, 3, 4, 5, 8, 9, 15, 16):
        out = torch.full((rows * V + 8,), 7.0, device="cuda")
        ie.vocab_proj(h[:rows].contiguous(), w, out[:rows * V].view(rows, V))
        assert torch.equal(out[:rows * V].view(rows, V), one[:rows]), rows
        assert (out[rows * V:] == 7.0).all()


# The GELU epilogue against 64 bits, v given as the bias of a zero product, over every size of v: 0.5 v (1 + tanh u) =
# v s with s = 1 / (1 + exp(-2u)).  Five roundings of the exponent (three operations, two constants) move v s by at most
# 5 |2u| s (1 - s) <= 1.12 units of 2^-24 |v|, the exponential's last place by 2 s (1 - s) <= 0.5, the result's by 1.
@pytest.mark.parametrize("M", [1, 16, 40, 600])
def test_gelu_epilogue_range(ie, M):
    r = rng(M)
    mag = np.concatenate([2.0 ** r.uniform(-140, 127, 2000), r.uniform(0, 12, 4000), [0.0, 1e-45, 5.5, 5.6, 3e38]])
    v = np.concatenate([mag, -mag]).astype(np.float32)
    N = v.size
    A, W = np.zeros((M, 64), np.int8), np.ones((N, 64), np.int8)
    got = ie.int8_gemm(_dev(pack_i8(A)), _dev(pack_i8(W)), _dev(np.ones(M, np.float32)), _dev(np.ones(N, np.float32)),
                       ie.EPI_BIAS_GELU, _dev(v)).cpu().numpy().astype(np.float64)
    d = v.astype(np.float64)
    u = 0.7978845608 * (d + 0.044715 * d ** 3)
    with np.errstate(over="ignore"):
        want = d / (1.0 + np.exp(-2.0 * u))
    assert (np.abs(got - want) <= 2.7 * 2.0 ** -24 * np.abs(d) + 2.0 ** -149).all()


# Decode rows whose cheapest slicing does not fit LDS although another one does (K % 16 == 0 and not).
@pytest.mark.parametrize("M,K,N,words", [(14, 8708, 1024, 0), (16, 8704, 1027, 0), (16, 9700, 500, 1), (4, 36900, 5, 0),
                                         (1, 131068, 9, 0)])
def test_gemv_any_width_second_slicing(ie, orc, M, K, N, words):
    _gemm_case(ie, orc, M, N, K, ie.EPI_I32, words, M + K + N)


# The lines between the kernels of short rows.  Unaligned rows of 16 to 64 bytes: one thread per output or staged, by rows
# and products (decode and prompt rows); aligned decode rows: K and N on both sides of the dot4 kernel's.  K = 128 and 240
# on a small grid: one and two groups without the ring's loop.
@pytest.mark.parametrize("M,K,N,words", [(1, 28, 37, 0), (1, 32, 37, 1), (1, 60, 10001, 0), (7, 40, 33, 0), (7, 44, 33, 0),
                                         (12, 44, 15000, 0), (12, 44, 17500, 0), (16, 60, 4700, 0), (16, 64, 77, 3),
                                         (17, 16, 4000, 1), (300, 20, 1100, 0), (300, 28, 900, 0), (100, 44, 1100, 0),
                                         (100, 44, 1200, 0), (60, 60, 1000, 0), (60, 60, 1200, 0), (9, 256, 70, 0),
                                         (9, 272, 70, 0), (16, 16, 5, 0), (1, 864, 2048, 0), (1, 880, 2047, 0),
                                         (2, 640, 3200, 0), (4, 1040, 12499, 0), (8, 1056, 8192, 0), (2, 1600, 9001, 0),
                                         (3, 752, 16385, 0), (8, 752, 16384, 0), (5, 656, 20481, 0),
                                         (33, 128, 65, 0), (200, 240, 70, 0), (17, 144, 33, 0)])
def test_gemm_short_rows(ie, orc, M, K, N, words):
    _gemm_case(ie, orc, M, N, K, ie.EPI_I32, words, M + K + N)
    _gemm_case(ie, orc, M, N, K, ie.EPI_BIAS_GELU if K % 32 else 3, words, M + K + N)


# Infinities and NaNs through the GELU of every GEMM family (decode, small-grid, LDS tiles, register-staged): from the
# bias, and from a product whose scale overflows.  As the oracle's tanh form: +inf stays, -inf and NaN give NaN.
@pytest.mark.parametrize("M,K", [(1, 768), (3, 256), (16, 768), (16, 4096), (40, 768), (40, 60), (600, 768), (600, 100)])
def test_gelu_epilogue_infinities(ie, orc, M, K):
    N = 900
    A, W = np.ones((M, K), np.int8), np.ones((N, K), np.int8)
    W[5] = -1
    sA, sB, bias = np.ones(M, np.float32), np.full(N, 1e-3, np.float32), np.zeros(N, np.float32)
    bias[[0, 1, 2, 3, 4]] = [np.inf, -np.inf, np.nan, 3.4e38, -3.4e38]
    sB[[5, 6]] = np.inf  # -inf and inf out of the product itself
    got = ie.int8_gemm(_dev(pack_i8(A)), _dev(pack_i8(W)), _dev(sA), _dev(sB), ie.EPI_BIAS_GELU,
                       _dev(bias)).cpu().numpy()
    want = orc.gemm(pack_i8(A), pack_i8(W), sA, sB, ie.EPI_BIAS_GELU, bias, None)
    assert np.isposinf(want[:, [0, 6]]).all() and np.isnan(want[:, [1, 2, 5]]).all()
    assert np.allclose(got, want, rtol=2e-6, atol=1e-7, equal_nan=True)


# The 64 x 64 and 128 x 64 LDS tiles: fewer stages than the ring (one to three of 128), as many, more, and a tail; one
# workgroup per CU, two, up to three, and past each (256 units; partial tiles both ways).
@pytest.mark.parametrize("K", [128, 256, 272, 384, 512, 1296, 2064])
@pytest.mark.parametrize("M,N", [(640, 1600), (641, 1601), (512, 4096), (1150, 1800), (768, 4096), (833, 3840),
                                 (1000, 4160)])
def test_gemm_tile_rounds(ie, orc, M, N, K):
    _gemm_case(ie, orc, M, N, K, ie.EPI_I32, 0, M + N + K)
    if K in (256, 1296):
        for epi in (ie.EPI_BIAS_GELU, 3):
            _gemm_case(ie, orc, M, N, K, epi, 0, M + N + K)

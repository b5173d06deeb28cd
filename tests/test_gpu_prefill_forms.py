"""The prompt attention's kernels for bf16 caches and for long or many contiguous
problems (three-part bf16 products), through the public entry points: every
form the launch rule can take, its ends of tiles, blocks and groups, the
promise that a query's bits do not depend on the form, and operands that have
no three-part form.  Reference and bar as test_gpu_prefill_attn.py's."""
import numpy as np
import pytest

from conftest import rng
from test_gpu_prefill_attn import REL, case, dev, host, oracle_prefill, rel_err

pytestmark = pytest.mark.gpu


# Paged bf16.  Fewer than 320 tiles of 64 queries: the split kernel (one key, one to five 32-key blocks, a context that
# ends in a block's second page, other block sizes); 320 and more: the tile kernel, one set of waves up to 256 keys, from
# 1024 tiles on and at d = 128, two at d = 64 between (a partial last tile, groups of unequal length).
@pytest.mark.parametrize("B,P,start,H_kv,G,d,bs", [
    (1, 1, 0, 1, 1, 64, 16), (2, 33, 0, 2, 1, 64, 16), (1, 17, 126, 2, 4, 128, 16), (2, 50, 300, 2, 2, 64, 16),
    (1, 40, 57, 2, 1, 128, 8), (1, 70, 13, 2, 2, 64, 48),
    (4, 100, 11, 20, 2, 64, 16), (2, 130, 0, 27, 2, 128, 16), (4, 65, 100, 20, 2, 128, 48),
    (2, 129, 190, 27, 2, 64, 16), (2, 150, 200, 27, 2, 128, 16), (2, 150, 140, 27, 2, 64, 8),
    (8, 65, 330, 64, 1, 64, 16)])
def test_paged_bf16_forms(ie, orc, B, P, start, H_kv, G, d, bs):
    Q, kc, vc, table = case(P + start + H_kv + d, B, P, start, H_kv, G, d, bs, 1)
    want = oracle_prefill(orc, Q, kc, vc, table, start, bs, H_kv, 1)
    got = host(ie.prefill_attn(dev(Q), dev(kc), dev(vc), dev(table), start, bs, H_kv, kv_dtype=ie.KV_BF16))
    assert rel_err(got, want) < REL


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("P,B", [(200, 4), (300, 4), (130, 12)])
def test_paged_bf16_bits_do_not_depend_on_the_form(ie, d, P, B):
    """B prompts at once (the tile kernel: 20 heads x 4 x 4 tiles of at most
    256 keys, x 5 of more, or x 3 x 12) against one prompt in chunks of 37 and
    of 1 (the split kernel)."""
    Q, kc, vc, table = case(7 * P + d, B, P, 0, 20, 1, d, 16, 1)
    whole = host(ie.prefill_attn(dev(Q), dev(kc), dev(vc), dev(table), 0, 16, 20, kv_dtype=ie.KV_BF16))
    kd, vd, td = dev(kc), dev(vc), dev(table[1:2])
    for t0, t1 in ((0, 37), (37, 74), (P - 40, P - 3), (P - 1, P)):
        part = host(ie.prefill_attn(dev(Q[1:2, t0:t1]), kd, vd, td, t0, 16, 20, kv_dtype=ie.KV_BF16))
        assert np.array_equal(part[0], whole[1, t0:t1])


# Contiguous fp32: few long problems on the split kernel (385 keys: the fp32 one), the tile kernel with two sets of waves
# (312 causal tiles at d = 64, 260 at d = 128, of 768 keys and more) and with one (512 tiles, 1024 of long ones).
@pytest.mark.parametrize("B,H,N,d,causal", [(1, 2, 769, 64, True), (1, 2, 801, 128, False), (1, 4, 385, 128, True),
                                            (1, 24, 780, 64, True), (2, 10, 800, 128, False), (2, 64, 250, 64, True),
                                            (4, 32, 200, 128, False), (8, 32, 97, 64, False), (2, 40, 801, 64, True)])
def test_flash_forms(ie, orc, B, H, N, d, causal):
    r = rng(N + H + d)
    Q, K, V = (r.standard_normal((B, H, N, d)).astype(np.float32) for _ in range(3))
    kc, vc, Qt = (np.ascontiguousarray(x.transpose(0, 2, 1, 3)) for x in (K, V, Q))
    table = np.arange(B, dtype=np.int32).reshape(B, 1)
    got = host(ie.flash_attn(dev(Q), dev(K), dev(V), causal=causal)).transpose(0, 2, 1, 3)
    # every head of a few query positions (all keys' block and group ends among them)
    for t in sorted({0, 15, 16, 31, 32, 63, 64, 95, N // 2, N - 2, N - 1}):
        n = t + 1 if causal else N
        want = orc.decode_attn(np.ascontiguousarray(Qt[:, t]), kc, vc, table, np.full(B, n, np.int32), n, N, H)
        assert rel_err(got[:, t], want) < REL


# A K entry of -inf gives its key a weight of 0 for the queries whose element there is positive; a V entry of inf makes
# that output element inf for the queries that see its key and leaves the others' finite; values that round to an
# infinite bf16 stay what they are.
@pytest.mark.parametrize("shape", ["split", "tile1", "tile2"])
@pytest.mark.parametrize("d", [64, 128])
def test_flash_operands_without_three_parts(ie, d, shape):
    import torch

    B, H, N = {"split": (1, 1, 800), "tile1": (2, 64, 250), "tile2": (1, 24, 780)}[shape]
    g = torch.Generator().manual_seed(d + N)
    Q, K, V = (torch.randn(B, H, N, d, generator=g) for _ in range(3))
    Q[..., 3] = Q[..., 3].abs() + 0.1
    K[0, 0, 70, 3] = -float("inf")       # never attended to by head 0
    V[0, 0, 150, 5] = float("inf")
    V[0, 0, 40, 7] = 3.4e38              # bf16 rounds it to inf; its weight keeps the output finite
    K[0, 0, 90, 9] = -3.4e38
    Q[0, 0, :, 9] = 1e-37                # a score of -3.4 / sqrt(d) from that element
    got = ie.flash_attn(Q.cuda(), K.cuda(), V.cuda(), causal=True).cpu().double()
    q, k, v = (x[0, 0].double() for x in (Q, K, V))
    s = (q @ k.t()) / d**0.5
    w = torch.softmax(s.masked_fill(~torch.ones(N, N, dtype=torch.bool).tril(), -float("inf")), dim=1)
    # weight 0 times an infinity is no part of the sum
    want = torch.where(w[:, :, None] == 0, torch.zeros(()), w[:, :, None] * v[None]).sum(1)
    # fp32 MFMAs take 16 queries and their keys together: the queries of the infinite value's own tile that
    # do not see its key get 0 x inf
    rows = torch.ones(N, dtype=torch.bool)
    rows[144:150] = False
    o = got[0, 0]
    assert torch.equal(o[rows].isinf(), want[rows].isinf()) and not o[rows].isnan().any()
    finite = rows & ~want.isinf().any(1)
    scale = want[finite].abs().amax(0)
    assert ((o[finite] - want[finite]).abs().amax(0) <= REL * scale).all()
    # untouched heads are as they are
    assert got[0, 1 % H][200:].isfinite().all() or H == 1


def test_paged_bf16_infinite_value(ie):
    """An infinity in a bf16 cache (exact in one part, but the weights' parts
    have signs of their own): inf where its key is seen, finite elsewhere."""
    B, P, H, d = 1, 100, 2, 64
    Q, kc, vc, table = case(5, B, P, 0, H, 1, d, 16, 1)
    page, slot = int(table[0, 3]), 5  # position 53
    vc = vc.copy()
    vc[page, slot, 0, 8] = 0x7F80
    kc = kc.copy()
    kc[page, slot + 2, 1, 4] = 0xFF80  # position 55, head 1: -inf
    Q[:, :, 1, 4] = np.abs(Q[:, :, 1, 4]) + 0.1
    got = host(ie.prefill_attn(dev(Q), dev(kc), dev(vc), dev(table), 0, 16, H, kv_dtype=ie.KV_BF16))[0]
    assert np.isposinf(got[53:, 0, 8]).all()
    assert np.isfinite(got[:48]).all() and np.isfinite(got[64:, 1]).all()
    kept = np.delete(got[53:, 0], 8, axis=1)
    assert np.isfinite(kept).all()


FORM_SHAPES = {"split": (1, 1, 800), "tile1": (2, 64, 250), "tile2": (1, 24, 780)}


def attention64(q, k, v, causal):
    """softmax(q k^T / sqrt(d)) v per (b, h) on the CPU in 64 bits."""
    import torch

    q, k, v = (x.double() for x in (q, k, v))
    s = q @ k.transpose(-1, -2) / q.shape[-1] ** 0.5
    if causal:
        s = s.masked_fill(~torch.ones(s.shape[-2:], dtype=torch.bool).tril(), -float("inf"))
    return torch.softmax(s, dim=-1) @ v


# Operands far from 1, whose bf16 parts could fall below bf16's range (2^-133) or pass it: V at the smallest normal
# numbers and among the subnormals, at both ends of the range, Q and K of sizes that offset each other.  The bar is
# the other tests'; subnormal results have 2^-149 of their own.
@pytest.mark.parametrize("shape", sorted(FORM_SHAPES))
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("qs,ks,vs", [(1, 1, 1e-33), (1, 1, 1e-36), (1, 1, 2.0 ** -126), (1, 1, 2.0 ** -135),
                                      (1, 1, 1e25), (1, 1, 1e37), (1e37, 1e-37, 1), (1e-37, 1e37, 1e-20),
                                      (1e36, 1e-36, 1e-36)])
def test_flash_operand_sizes(ie, d, shape, qs, ks, vs):
    import torch

    B, H, N = FORM_SHAPES[shape]
    g = torch.Generator().manual_seed(d + N)
    Q, K, V = (torch.randn(B, H, N, d, generator=g) * s for s in (qs, ks, vs))
    got = ie.flash_attn(Q.cuda(), K.cuda(), V.cuda(), causal=True).cpu().double()
    for h in {0, H - 1}:
        want = attention64(Q[0, h], K[0, h], V[0, h], True)
        assert ((got[0, h] - want).abs() <= REL * want.abs().max() + 2.0 ** -149).all()


# Weights near the smallest normal number on values as much larger than the others': the small weights' own bits
# count.  The score of about -125 (in powers of two) has three roundings, each moving its weight by up to 125 x 2^-24 ln 2.
@pytest.mark.parametrize("shape", sorted(FORM_SHAPES))
@pytest.mark.parametrize("d", [64, 128])
def test_flash_tiny_weights(ie, d, shape):
    import torch

    B, H, N = FORM_SHAPES[shape]
    g = torch.Generator().manual_seed(d + N)
    Q, K = torch.zeros(B, H, N, d), torch.zeros(B, H, N, d)
    Q[..., 0] = 1.0
    K[..., 3, 0] = -125 * d ** 0.5 * 0.6931471805599453
    V = (1.0 + torch.rand(B, H, N, d, generator=g)) * 2.0 ** -64
    V[:, :, 3] = (1.0 + torch.rand(B, H, d, generator=g)) * 2.0 ** 75
    got = ie.flash_attn(Q.cuda(), K.cuda(), V.cuda(), causal=False).cpu().double()
    want = attention64(Q[0, 0], K[0, 0], V[0, 0], False)
    assert (want > 4 * 2.0 ** -64).all()  # the one key's share is the larger part
    assert ((got[0, 0] - want).abs() <= (3 * 125 * 2.0 ** -24 + REL) * want).all()


@pytest.mark.parametrize("qs,ks,vs", [(1e-37, 1e37, 1), (1e36, 1e-36, 1), (1, 1, 2.0 ** -130), (1, 1, 1e37)])
@pytest.mark.parametrize("P,H", [(70, 2), (100, 170)])  # the split kernel, the tile kernel
def test_paged_bf16_operand_sizes(ie, P, H, qs, ks, vs):
    import torch

    d, bs = 64, 16
    nb = (P + bs - 1) // bs
    g = torch.Generator().manual_seed(P)
    Q = torch.randn(1, P, H, d, generator=g) * qs
    K, V = ((torch.randn(nb, bs, H, d, generator=g) * s).to(torch.bfloat16) for s in (ks, vs))
    table = torch.arange(nb, dtype=torch.int32).view(1, nb)
    got = ie.prefill_attn(Q.cuda(), K.cuda(), V.cuda(), table.cuda(), 0, bs, H, kv_dtype=ie.KV_BF16).cpu().double()
    for h in {0, H - 1}:
        k, v = (x.view(-1, H, d)[:P, h].float() for x in (K, V))
        want = attention64(Q[0, :, h], k, v, True)
        assert ((got[0, :, h] - want).abs() <= REL * want.abs().max() + 2.0 ** -149).all()


# Queries that are computed again (they see an infinite key, or are themselves too small for three parts) and the others
# of their tiles: those keep the bits that they have in any other chunk of the prompt.
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("H", [2, 170])  # the split kernel, the tile kernel for the whole prompt
def test_paged_bf16_queries_beside_one_computed_again(ie, d, H):
    import torch

    P, bs = 100, 16
    Q, kc, vc, table = case(3 * H + d, 1, P, 0, H, 1, d, bs, 1)
    plain = host(ie.prefill_attn(dev(Q), dev(kc), dev(vc), dev(table), 0, bs, H, kv_dtype=ie.KV_BF16))[0]
    kc = kc.copy()
    kc[int(table[0, 40 // bs]), 40 % bs, 0, 4] = 0x7F80  # position 40, head 0: inf
    Q = Q.copy()
    Q[0, 70, 1] *= 1e-33
    Q[0, 5, 1, 3] = 1e-38
    kd, vd, td = dev(kc), dev(vc), dev(table)
    for chunks in ((0, P), (0, 33, P), (0, 41, 71, P), (0, 7, 35, 60, P)):
        got = np.concatenate([host(ie.prefill_attn(dev(Q[:, a:b]), kd, vd, td, a, bs, H, kv_dtype=ie.KV_BF16))[0]
                              for a, b in zip(chunks, chunks[1:])])
        assert np.array_equal(got[:40, 0], plain[:40, 0]), chunks
        assert not np.isfinite(got[40:, 0]).all()
        same = np.delete(np.arange(P), [5, 70])
        assert np.array_equal(got[same, 1], plain[same, 1]), chunks
        # the small queries: (almost) equal weights
        k, v = (torch.from_numpy(x.astype(np.int32) << 16).view(torch.float32)[table[0]].reshape(-1, H, d)[:, 1].double()
                for x in (kc, vc))
        for t in (5, 70):
            w = torch.softmax(k[:t + 1] @ torch.from_numpy(Q[0, t, 1]).double() / d ** 0.5, 0)
            want = (w @ v[:t + 1]).numpy()
            assert np.abs(got[t, 1] - want).max() <= REL * np.abs(want).max()
        assert np.array_equal(got[:, 2:], plain[:, 2:])


# 16 rows of a page past 4 GiB (2.24 million heads): 32-bit row offsets would wrap from the last row on.  A few heads
# hold values, the others zeros; the split kernel (P = 16) and the tile kernel (17, a second page).
@pytest.mark.parametrize("P", [16, 17])
def test_paged_bf16_rows_past_4_gib(ie, P):
    import torch

    H, d, bs = 2_240_000, 64, 16
    nb = (P + bs - 1) // bs
    heads = torch.tensor([0, 1, H // 2 + 1, H - 1])
    g = torch.Generator().manual_seed(P)
    q = torch.randn(P, 4, d, generator=g)
    k, v = (torch.randn(nb, bs, 4, d, generator=g).to(torch.bfloat16) for _ in range(2))
    Q = torch.zeros(1, P, H, d, device="cuda")
    K, V = (torch.zeros(nb, bs, H, d, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    Q[0][:, heads.cuda()] = q.cuda()
    for big, small in ((K, k), (V, v)):
        big[:, :, heads.cuda()] = small.cuda()
    table = torch.arange(nb, dtype=torch.int32, device="cuda").view(1, nb)
    got = ie.prefill_attn(Q, K, V, table, 0, bs, H, kv_dtype=ie.KV_BF16)[0][:, heads.cuda()].cpu().double()
    del Q, K, V
    torch.cuda.empty_cache()
    for i in range(4):
        want = attention64(q[:, i], *(x.reshape(-1, 4, d)[:P, i].float() for x in (k, v)), True)
        assert (got[:, i] - want).abs().max() <= REL * want.abs().max()


# The launch rule's other lines for bf16 pages: at most 16 queries of many pairs (the split kernel), a long prompt from
# the start at d = 128 (two sets of waves), one round of the split kernel and of two sets of waves at d = 64, blocks of
# two and three 16-token runs and of none.  Each against the prompt in one-query chunks of one sequence at the same positions.
@pytest.mark.parametrize("B,P,start,H,d,bs", [(8, 16, 100, 48, 128, 16), (8, 17, 100, 48, 64, 16), (1, 520, 0, 36, 128, 16),
                                              (2, 520, 130, 18, 128, 32), (6, 32, 300, 56, 64, 16), (2, 210, 60, 45, 64, 48), (6, 70, 90, 30, 64, 32),
                                              (6, 70, 90, 30, 128, 20)])
def test_paged_bf16_launch_rule(ie, B, P, start, H, d, bs):
    Q, kc, vc, table = case(P + start + H + bs, B, P, start, H, 1, d, bs, 1)
    kd, vd = dev(kc), dev(vc)
    whole = host(ie.prefill_attn(dev(Q), kd, vd, dev(table), start, bs, H, kv_dtype=ie.KV_BF16))
    for b in {0, B - 1}:
        for t in sorted({0, 1, 15, P // 2, P - 1}):
            one = host(ie.prefill_attn(dev(Q[b:b + 1, t:t + 1]), kd, vd, dev(table[b:b + 1]), start + t, bs, H,
                                       kv_dtype=ie.KV_BF16))
            assert np.array_equal(one[0, 0], whole[b, t]), (b, t)
    k, v = (from_bf16(x)[table[0]].reshape(-1, H, d)[:start + P] for x in (kc, vc))
    for h in {0, H - 1}:
        s = Q[0, :, h].astype(np.float64) @ k[:, h].T / d ** 0.5
        s[np.arange(start + P)[None] > start + np.arange(P)[:, None]] = -np.inf
        w = np.exp(s - s.max(1, keepdims=True))
        want = w @ v[:, h] / w.sum(1, keepdims=True)
        assert np.abs(whole[0, :, h] - want).max() <= REL * np.abs(want).max()


# The launch rule's lines for contiguous problems, a shape on each side: 64 tiles of 576 keys (d = 128), 128 / 64 and
# 256 / 144 tiles of 768 (d = 128, causal or not), 128 / 300 / 384 and any number of 1500 keys (d = 64).
@pytest.mark.parametrize("H,N,d,causal", [(6, 576, 128, True), (7, 600, 128, True), (6, 575, 128, False),
                                          (9, 800, 128, True), (10, 800, 128, True), (20, 800, 128, True),
                                          (4, 1000, 128, False), (5, 1000, 128, False), (11, 800, 128, False),
                                          (12, 800, 128, False), (9, 800, 64, True), (10, 800, 64, True),
                                          (23, 800, 64, True), (24, 800, 64, False), (12, 1500, 64, True),
                                          (16, 1500, 64, True), (16, 1500, 64, False)])
def test_flash_launch_rule(ie, H, N, d, causal):
    import torch

    g = torch.Generator().manual_seed(H + N + d)
    Q, K, V = (torch.randn(1, H, N, d, generator=g) for _ in range(3))
    got = ie.flash_attn(Q.cuda(), K.cuda(), V.cuda(), causal=causal).cpu().double()
    for h in {0, H - 1}:
        want = attention64(Q[0, h], K[0, h], V[0, h], causal)
        assert ((got[0, h] - want).abs() <= REL * want.abs().max()).all()


def from_bf16(bits):
    """bf16 bit patterns as 64-bit floats."""
    return (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)

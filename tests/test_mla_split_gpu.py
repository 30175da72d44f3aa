"""The work split of the MLA decode: the balanced split (a full round of CTAs
shares the batch's 64-token tiles, several requests to a CTA and several CTAs
to a request) at its edges, against the CPU oracle, and its arithmetic on the
CPU. Tolerance: the oracle's 1-ULP rule of test_mla_gpu."""
import ctypes

import numpy as np
import pytest
import torch

import moonmath_attention as ma
from moonmath_attention import _lib
from mla_inputs import KV_SCALE, QK, SCALE_576, fp8_bits, paged_pool, ragged_lens, rand_kv_rows, rand_q
from test_mla_gpu import DEV, _check, _d


def _split(lens, H, q_len, parts, tokens=0):
    """(unit, request, part, parts, record, first token, end token) of every segment,
    as the launchers' plan gives them; [] for equal parts within the parts budget."""
    arr = (ctypes.c_int * len(lens))(*lens)
    n = _lib.lib.moonmath_mla_split(len(lens), arr, H, q_len, parts, tokens, (ctypes.c_int * 7)(), 0)
    assert n >= 0
    out = (ctypes.c_int * (7 * n + 1))()
    assert _lib.lib.moonmath_mla_split(len(lens), arr, H, q_len, parts, tokens, out, n) == n
    return [tuple(out[7 * i:7 * i + 7]) for i in range(n)]


@pytest.mark.parametrize("H,q_len,tokens,units", [
    (16, 1, 0, 256), (5, 3, 9000, 256), (64, 1, 0, 256), (64, 1, 1, 128), (11, 3, 327680, 128), (64, 1, 327681, 256),
    (128, 1, 1, 128), (96, 2, 0, 80), (128, 2, 0, 64), (128, 8, 0, 16)])
def test_balanced_split_covers_every_tile_once(H, q_len, tokens, units):
    """Every token of every request in one segment, in order; parts consecutive, on
    whole tiles and not empty (but the one of an empty request); records distinct,
    consecutive per request and within the B * parts of the workspace; units within
    a round. At the fewest parts the launchers run it with: one fewer leaves the
    records of a round short."""
    rng = np.random.default_rng(units)
    cases = [rng.integers(0, 9000, size=int(rng.integers(1, 400))).tolist() for _ in range(60)]
    cases += [[0] * 300, [1] * 70, [100000] + [0] * 90, [64] * 256, [8192] * 64, [5], [-3, 70, 5000], [2048] * 128]
    for lens in cases:
        B = len(lens)
        if tokens and 32 < H * q_len <= 64 and B > 128:
            continue  # row groups of 64
        parts = 1 + -(-(units - 1) // B)
        if _lib.lib.moonmath_mla_effective_parts(B, H, parts, q_len, 1) != parts:
            continue  # more records than a workspace holds
        assert parts == 1 or _split(lens, H, q_len, parts - 1, tokens) == []
        at, first, recs, last = [0] * B, {}, [], 0
        for u, b, part, nparts, rec, lo, hi in _split(lens, H, q_len, parts, tokens):
            assert last <= u < units and lo == at[b] and (hi > lo or lens[b] <= 0 and lo == hi == 0)
            assert 0 <= part < nparts and (hi % 64 == 0 or hi == lens[b])
            assert part == 0 or rec == first[b] + part
            first.setdefault(b, rec)
            recs.append(rec)
            at[b], last = hi, u
        assert at == [max(0, n) for n in lens] and sorted(first) == list(range(B))
        assert recs == sorted(set(recs)) and recs[-1] < B * parts


def test_contiguous_parts():
    """Never more than the planners reserve records for; whole requests where they
    fill most of a round, parts where a round has room for two of each."""
    lib = _lib.lib
    rng = np.random.default_rng(5)
    for _ in range(2000):
        B, H, S, q_len = (int(rng.integers(1, m)) for m in (600, 129, 9000, 9))
        assert 1 <= lib.moonmath_mla_slab_parts(B, H, S, q_len) <= lib.mla_decode_a16w8_multiq_plan_parts_q(B, S, q_len, H)
    for B, H, S, whole in [(256, 16, 2048, True), (200, 16, 2048, True), (230, 32, 1000, True), (128, 128, 1500, True),
                           (150, 16, 2000, False), (80, 128, 3000, False), (100, 16, 2048, False), (1, 16, 4097, False)]:
        assert (lib.moonmath_mla_slab_parts(B, H, S, 1) == 1) == whole, (B, H, S)


LENS = [0, 1, 2, 63, 64, 65, 127, 128, 129, 511, 512, 513, 700, 1500, 2100, 9000]


@pytest.mark.gpu
@pytest.mark.parametrize("H,q_len,page", [(16, 1, 64), (16, 1, 1), (5, 3, 5), (17, 1, 64), (33, 1, 1), (64, 1, 64),
                                          (65, 1, 5), (128, 1, 64), (16, 4, 3), (128, 2, 64), (96, 8, 64)])
def test_balanced_split_matches_oracle(H, q_len, page):
    """Enough parts for the balanced split on 16 requests: an empty request and
    lengths at the edges of tiles, of a CTA's share and of its index batches;
    row groups of 64 with 1 to 64 rows; pages of consecutive slots, single
    scattered slots, and runs that straddle a wave's 8 or 16 tokens."""
    B = len(LENS)
    # The oracle has no empty requests: their rows are zero.
    pool, idx, indptr = paged_pool(LENS, 91, page=page)
    q_lat, q_pe = rand_q(B, q_len, H, 91)
    o = torch.full((B, q_len, H, 512), float("nan"), dtype=torch.bfloat16, device=DEV)
    op = ma.mla_decode_a16w8_paged_dev
    op(_d(q_lat), _d(q_pe), _d(pool), o, _d(torch.tensor(LENS, dtype=torch.int32)), None, _d(idx), _d(indptr), 20,
       SCALE_576, KV_SCALE)
    torch.cuda.synchronize()
    assert torch.all(o[0] == 0)
    o[0] = 0
    _check(o, q_lat, q_pe, fp8_bits(pool), LENS, SCALE_576, kv_indices=idx.numpy(), kv_indptr=indptr.numpy(),
           batches=list(range(1, B)))


@pytest.mark.gpu
@pytest.mark.parametrize("H,q_len,B,S", [
    (16, 1, 5, 3001), (64, 1, 130, 100), (128, 1, 3, 1025), (32, 4, 2, 4097),
    (16, 1, 256, 600), (16, 1, 200, 1000), (128, 2, 64, 700)])  # whole requests where paged ones are split
def test_balanced_split_contiguous(H, q_len, B, S):
    kv = rand_kv_rows(B * S, 93).view(B, S, QK)
    q_lat, q_pe = rand_q(B, q_len, H, 93)
    if q_len == 1:
        q_lat, q_pe = q_lat[:, 0].contiguous(), q_pe[:, 0].contiguous()
    o = torch.full(q_lat.shape, float("nan"), dtype=torch.bfloat16, device=DEV)
    (ma.mla_decode_a16w8 if q_len == 1 else ma.mla_decode_a16w8_multiq)(_d(q_lat), _d(q_pe), _d(kv), o, SCALE_576,
                                                                        KV_SCALE)
    torch.cuda.synchronize()
    pick = [b for b in range(B) if B <= 5 or b in (0, 1, 63, 64, B // 2, B - 1)]
    _check(o, q_lat, q_pe, fp8_bits(kv), [S] * B, SCALE_576, batches=pick)


@pytest.mark.gpu
@pytest.mark.parametrize("H,q_len", [(33, 1), (16, 3), (64, 1), (16, 4)])
def test_row_groups_of_32_and_64(H, q_len):
    """Calls of 33..64 rows as one 64-row group (kv_bytes 0: unknown) and as two of
    32: the same sums for whole requests, bit for bit, and both within the oracle's
    rule when split."""
    lens = [1, 64, 200, 1000, 3000]
    B = len(lens)
    pool, idx, indptr = paged_pool(lens, 113)
    q_lat, q_pe = rand_q(B, q_len, H, 113)
    t = [_d(x) for x in (q_lat, q_pe, pool, torch.tensor(lens, dtype=torch.int32), idx, indptr)]
    lib, p = _lib.lib, _lib.ptr
    for parts in (1, 60):
        ws = torch.empty(lib.mla_decode_a16w8_multiq_workspace_for(B, H, parts, q_len), dtype=torch.uint8, device=DEV)
        outs = []
        for kv_bytes in (0, idx.numel() * QK):
            o = torch.full((B, q_len, H, 512), float("nan"), dtype=torch.bfloat16, device=DEV)
            assert lib.launch_mla_decode_a16w8_paged_dev(p(t[0]), p(t[1]), p(t[2]), p(o), p(t[3]), None, p(t[4]), p(t[5]), B,
                                                         H, parts, 512, 64, SCALE_576, KV_SCALE, 1.0, p(ws),
                                                         _lib.stream_ptr(DEV), kv_bytes, q_len) == 0
            torch.cuda.synchronize()
            _check(o, q_lat, q_pe, fp8_bits(pool), lens, SCALE_576, kv_indices=idx.numpy(), kv_indptr=indptr.numpy())
            outs.append(o)
        assert parts > 1 or torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.gpu
def test_balanced_split_many_requests():
    """More requests than a round of CTAs: several whole requests to a CTA."""
    B, H = 700, 8
    lens = ragged_lens(B, 0, 300, 95)
    pool, idx, indptr = paged_pool(lens, 95)
    q_lat, q_pe = rand_q(B, 1, H, 95)
    o = torch.full((B, 1, H, 512), float("nan"), dtype=torch.bfloat16, device=DEV)
    ma.mla_decode_a16w8_paged_dev(_d(q_lat), _d(q_pe), _d(pool), o, _d(torch.tensor(lens, dtype=torch.int32)), None,
                                  _d(idx), _d(indptr), 2, SCALE_576, KV_SCALE)
    torch.cuda.synchronize()
    pick = [b for b in range(0, B, 13) if lens[b] > 0] + [b for b in range(B - 3, B) if lens[b] > 0]
    _check(o, q_lat, q_pe, fp8_bits(pool), lens, SCALE_576, kv_indices=idx.numpy(), kv_indptr=indptr.numpy(),
           batches=pick)
    assert not torch.isnan(o.float()).any()


@pytest.mark.gpu
@pytest.mark.parametrize("H,parts", [(16, 1), (16, 70), (64, 1), (64, 70)])
def test_block_table_clamps_pages_and_lengths(H, parts):
    """The table is read by the decode itself: page ids outside the pool and
    lengths outside the table give what the clamped table and lengths give, bit
    for bit, in both kernels and both splits."""
    B, max_blocks, num_blocks = 4, 9, 20
    g = torch.Generator().manual_seed(97)
    pool = rand_kv_rows(num_blocks * 64, 97).view(num_blocks, 64, QK)
    table = torch.randint(-5, num_blocks + 5, (B, max_blocks), generator=g, dtype=torch.int32)
    lens = torch.tensor([-3, 577, 130, 100000], dtype=torch.int32)
    q_lat, q_pe = (t[:, 0].contiguous() for t in rand_q(B, 1, H, 97))
    outs = []
    for t, n in ((table, lens), (table.clamp(0, num_blocks - 1), lens.clamp(0, max_blocks * 64))):
        o = torch.full((B, H, 512), float("nan"), dtype=torch.bfloat16, device=DEV)
        ma.mla_decode_a16w8_paged_blocks(_d(q_lat), _d(q_pe), _d(pool), o, _d(n), _d(t), parts, SCALE_576, KV_SCALE)
        torch.cuda.synchronize()
        outs.append(o)
    assert not torch.isnan(outs[0].float()).any()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.gpu
def test_noalloc_shares_its_array_beyond_64_parts():
    """300 parts of 256 rows: the size limit of the allocation-free entry counts
    64 of them (accepted); the call then uses the 128 that its array holds."""
    H, q_len, S = 128, 2, 20000
    pool, idx, indptr = paged_pool([S], 99)
    q_lat, q_pe = rand_q(1, q_len, H, 99)
    t = [_d(x) for x in (q_lat, q_pe, pool)]
    n = torch.tensor([S], dtype=torch.int32, device=DEV)
    idx, indptr = _d(idx), _d(indptr)
    lib, p, st = _lib.lib, _lib.ptr, _lib.stream_ptr(DEV)
    outs = []
    for noalloc in (True, False):
        o = torch.full((1, q_len, H, 512), float("nan"), dtype=torch.bfloat16, device=DEV)
        parts = 300 if noalloc else 128
        head = (p(t[0]), p(t[1]), p(t[2]), p(o), p(n), None, p(idx), p(indptr), 1, H, parts, 512, 64, SCALE_576,
                KV_SCALE, 1.0)
        if noalloc:
            rc = lib.launch_mla_decode_a16w8_paged_dev_noalloc(*head, st, 0, q_len)
        else:
            ws = torch.empty(lib.mla_decode_a16w8_multiq_workspace_for(1, H, parts, q_len), dtype=torch.uint8,
                             device=DEV)
            rc = lib.launch_mla_decode_a16w8_paged_dev(*head, p(ws), st, 0, q_len)
        torch.cuda.synchronize()
        assert rc == 0
        outs.append(o)
    assert not torch.isnan(outs[0].float()).any()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [1, 70])
@pytest.mark.parametrize("H,q_len", [(16, 1), (4, 4), (32, 1), (64, 1), (16, 4), (128, 1)])
def test_no_row_outside_the_requests_is_read(H, q_len, parts):
    """Every cache row that no token owns holds NaN codes (a pool from
    torch.empty, a recycled page): the rest of a request's last page, and pages
    of no request. Block tables and flat slots give the same bits, with no NaN,
    at lengths around each wave's 8 or 16 tokens of a last tile."""
    lens = [1, 7, 8, 9, 15, 16, 17, 47, 48, 49, 56, 57, 63, 64, 65, 130, 177, 700, 1025]
    B, most = len(lens), -(-max(lens) // 64)
    num_blocks = sum(-(-n // 64) for n in lens) + 3
    g = torch.Generator().manual_seed(101)
    order = torch.randperm(num_blocks, generator=g).tolist()
    bits = torch.full((num_blocks * 64, QK), 0x7F, dtype=torch.uint8)
    rows = rand_kv_rows(sum(lens), 101).view(torch.uint8)
    table = torch.full((B, most), order[-1], dtype=torch.int32)
    slots = []
    for b, n in enumerate(lens):
        pages = [order.pop(0) for _ in range(-(-n // 64))]
        table[b, :len(pages)] = torch.tensor(pages, dtype=torch.int32)
        slots += [pages[t // 64] * 64 + t % 64 for t in range(n)]
    bits[torch.tensor(slots)] = rows
    pool = _d(bits.view(torch.float8_e4m3fn).view(num_blocks, 64, QK))
    idx = _d(torch.tensor(slots, dtype=torch.int32))
    indptr = _d(torch.tensor([0] + np.cumsum(lens).tolist(), dtype=torch.int32))
    n = _d(torch.tensor(lens, dtype=torch.int32))
    q_lat, q_pe = (_d(t) for t in rand_q(B, q_len, H, 101))
    flat, blocks = (torch.full((B, q_len, H, 512), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ma.mla_decode_a16w8_paged_dev(q_lat, q_pe, pool.view(-1, 1, QK), flat, n, None, idx, indptr, parts, SCALE_576,
                                  KV_SCALE)
    ma.mla_decode_a16w8_paged_blocks(q_lat, q_pe, pool, blocks, n, _d(table), parts, SCALE_576, KV_SCALE)
    torch.cuda.synchronize()
    assert not torch.isnan(flat.float()).any()
    assert torch.equal(blocks.view(torch.int16), flat.view(torch.int16))


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [1, 70])
@pytest.mark.parametrize("H", [16, 32, 64, 128])
def test_scores_of_minus_infinity_before_finite_ones(H, parts):
    """Scores that overflow to -inf over a part's first tiles weigh nothing: the
    result is that of the tokens after them. (Queries of 2^120 in one dim, where
    those tokens hold -448, and 0 elsewhere in it.)"""
    S, cut = 700, 150
    kv = rand_kv_rows(S, 103).float()
    kv[:, 5] = 0.0
    kv[:cut, 5] = -448.0
    q_lat, q_pe = (t[:, 0].contiguous() for t in rand_q(1, 1, H, 103))
    q_lat[..., 5] = 2.0 ** 120
    pool = _d(kv.to(torch.float8_e4m3fn).view(S, 1, QK))
    outs = []
    for lo in (0, cut):
        o = torch.full((1, H, 512), float("nan"), dtype=torch.bfloat16, device=DEV)
        idx = _d(torch.arange(lo, S, dtype=torch.int32))
        n, indptr = (_d(torch.tensor(t, dtype=torch.int32)) for t in ([S - lo], [0, S - lo]))
        ma.mla_decode_a16w8_paged_dev(_d(q_lat), _d(q_pe), pool, o, n, None, idx, indptr, parts, SCALE_576, KV_SCALE)
        outs.append(o.float())
    torch.cuda.synchronize()
    # The two place tiles differently: fp32 sums in another order, then one bf16
    # rounding each (2^-8 of a value, both sides), P's rounding unchanged up to
    # the row max's power of two.
    a, b = outs
    assert torch.isfinite(a).all()
    assert ((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["q_lat", "q_pe", "both"])
@pytest.mark.parametrize("H,q_len", [(5, 1), (16, 1), (33, 1), (128, 1), (16, 5)])
def test_queries_off_a_16_byte_boundary(H, q_len, which):
    """Views that start one element into their buffers: read by plain loads, the
    bits are those of aligned copies."""
    lens = [130, 1000, 64, 2500]
    B = len(lens)
    pool, idx, indptr = paged_pool(lens, 107)
    q = [_d(t) for t in rand_q(B, q_len, H, 107)]

    def off(t):
        v = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)[1:].view(t.shape)
        return v.copy_(t)

    moved = [off(t) if which in (name, "both") else t for name, t in zip(("q_lat", "q_pe"), q, strict=True)]
    n, pool, idx, indptr = _d(torch.tensor(lens, dtype=torch.int32)), _d(pool), _d(idx), _d(indptr)
    slab = _d(rand_kv_rows(B * 300, 109).view(B, 300, QK))
    outs = []
    for ql, qp in (q, moved):
        o = torch.full((3, B, q_len, H, 512), float("nan"), dtype=torch.bfloat16, device=DEV)
        for i, parts in enumerate((1, 20)):
            ma.mla_decode_a16w8_paged_dev(ql, qp, pool, o[i], n, None, idx, indptr, parts, SCALE_576, KV_SCALE)
        if q_len == 1:
            ma.mla_decode_a16w8(ql[:, 0], qp[:, 0], slab, o[2, :, 0], SCALE_576, KV_SCALE)
        else:
            ma.mla_decode_a16w8_multiq(ql, qp, slab, o[2], SCALE_576, KV_SCALE)
        torch.cuda.synchronize()
        outs.append(o)
    assert not torch.isnan(outs[0].float()).any()
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16))

"""GPU-free decision tables of the split policies (host code of the C ABI).

The reference pins its GEMM split decision in a CPU test
(fxpr_vllm/_tests/test_gemm_warmup.py:16-62: cached choice, forced override,
clamps); its attention policy is closed-form (_pick_num_splits,
fxpr_vllm/_triton/attention.py:664-689). This build's policies are its own
static tables, in C (fxpr_attention_splits, fxpr_gemm_splits); these tests
pin them case by case. That a split count never changes the bits is the GPU
tests' part (tests/test_hip_attention.py, tests/test_hip_gemm.py).
"""

from __future__ import annotations

import ctypes

import pytest

from fxpr_vllm import _hip


@pytest.fixture(scope="module")
def lib():
    return _hip.load()


def attn_splits(lib, requests, kv_heads, group, max_q, keys, page=16, requested=0):
    return lib.fxpr_attention_splits(requests, kv_heads, group, max_q, -(-keys // page), page, requested)


def test_attention_explicit_request_wins(lib):
    # decode rows of 8192 keys hold 16 chunks of 512 keys
    for r in (1, 2, 3, 4, 8, 16):
        assert attn_splits(lib, 64, 8, 4, 1, 8192, requested=r) == r
    # an explicit request splits even where the automatic policy would not
    assert attn_splits(lib, 4, 8, 4, 1, 1024, requested=2) == 2          # short context
    assert attn_splits(lib, 1024, 8, 4, 1, 8192, requested=4) == 4      # oversubscribed
    assert attn_splits(lib, 4, 8, 4, 2048, 2048, requested=3) == 3       # prefill


def test_attention_explicit_request_beyond_chunks(lib):
    # splits past the row's chunk count would hold no keys: the launch runs
    # one per chunk (more than the automatic cap of 64 when rows are long)
    assert attn_splits(lib, 64, 8, 4, 1, 8192, requested=100) == 16
    assert attn_splits(lib, 2, 8, 4, 1, 65536, requested=100) == 100     # 128 chunks
    assert attn_splits(lib, 2, 8, 4, 1, 65536, requested=1000) == 128
    assert attn_splits(lib, 2, 8, 4, 1, 100, requested=5) == 1           # one chunk
    # the grid's z dimension bounds it
    assert attn_splits(lib, 1, 1, 1, 1, 512 * 70000, page=512, requested=70000) == 65535


def test_attention_auto_short_context(lib):
    # up to 32 key tiles of 64 (2048 keys): unsplit
    for keys in (1, 64, 512, 2048):
        assert attn_splits(lib, 4, 8, 4, 1, keys) == 1
    # 33 tiles: 5 chunks of 8 tiles, one split each
    assert attn_splits(lib, 4, 8, 4, 1, 2049) == 5


def test_attention_auto_one_chunk_per_split(lib):
    assert attn_splits(lib, 64, 8, 4, 1, 8192) == 16      # the bench decode shape
    assert attn_splits(lib, 64, 8, 4, 1, 4096) == 8
    assert attn_splits(lib, 1, 8, 4, 1, 20000) == 40      # ragged: 313 tiles, 40 chunks
    assert attn_splits(lib, 1, 8, 4, 1, 65536) == 64      # capped at 64
    assert attn_splits(lib, 1, 8, 4, 1, 1 << 20) == 64


def test_attention_auto_oversubscribed(lib):
    # (request, kv head, 16-row query tile) workgroups above 8 x 256: unsplit
    assert attn_splits(lib, 256, 8, 4, 1, 8192) == 16     # 2048 workgroups: still splits
    assert attn_splits(lib, 257, 8, 4, 1, 8192) == 1      # 2056
    # GQA groups share a query tile: 4 rows per (query, kv head) at group 4
    assert attn_splits(lib, 64, 8, 4, 4, 8192) == 16      # 16 rows: one tile
    assert attn_splits(lib, 64, 8, 4, 5, 8192) == 16      # 20 rows: 2 tiles, 1024 workgroups
    assert attn_splits(lib, 64, 8, 4, 17, 8192) == 1      # 68 rows: 5 tiles, 2560 workgroups
    # prefill: 4 requests x 8 kv heads x 512 query tiles
    assert attn_splits(lib, 4, 8, 4, 2048, 8192) == 1


def test_attention_policy_is_static(lib):
    # the same arguments always give the same count (graph capture bakes it in)
    first = [attn_splits(lib, b, 8, 4, 1, 8192) for b in (1, 8, 64, 300)]
    assert first == [attn_splits(lib, b, 8, 4, 1, 8192) for b in (1, 8, 64, 300)]


# kernels of fxpr_attention_plan: 16-row workgroups by register loads / LDS DMA,
# long requests apart by register loads / LDS DMA
ROWS16, ROWS16_DMA, LONG, LONG_DMA = range(4)


def attn_plan(lib, requests, tokens, max_q, keys, dt=1, heads=32, kv_heads=8, d=128, page=16, bits=32, stride=None,
              requested=0, window=0, causal=1):
    """(kernels, splits of long requests, of short ones, record rows per request, workspace bytes)"""
    plan = (ctypes.c_int32 * 4)()
    stride = kv_heads * d if stride is None else stride
    n = lib.fxpr_attention_plan(dt, requests, tokens, heads, kv_heads, d, page, max_q, -(-keys // page), stride, stride,
                                causal, window, bits, requested, plan)
    return (*plan, n)


def record_bytes(rows, keys, heads=32, d=128, acc=4):
    """Split records of `rows` workspace rows over a table of `keys` (heads and d as attn_plan's)."""
    slots = -(-keys // 512)
    up = lambda n: -(-n // 256) * 256  # noqa: E731
    return sum(map(up, (rows * heads * 8, rows * heads * slots * 4, rows * heads * slots * acc,
                        rows * heads * slots * d * acc)))


def test_attention_workspace_is_the_running_launchs(lib):
    # a 120-token chunk beside 20 decode steps, contexts up to 3040 keys: the
    # DMA kernels keep records of the split prefill rows; launches they do not
    # take (fp32 inputs, pages of 8 or 48 keys, a key stride of 2^20 elements,
    # 64-bit sums) run unsplit without any
    mixed = dict(requests=21, tokens=140, max_q=120, keys=3040)
    want = record_bytes(140, 3040)
    assert attn_plan(lib, **mixed) == (LONG_DMA, 6, 6, 0, want)
    assert attn_plan(lib, dt=F16, **mixed)[-1] == want
    assert attn_plan(lib, dt=F32, **mixed) == (ROWS16, 1, 1, 0, 0)
    assert attn_plan(lib, page=8, **mixed) == (LONG, 1, 1, 0, 0)
    assert attn_plan(lib, page=48, **mixed) == (LONG, 1, 1, 0, 0)
    assert attn_plan(lib, stride=1 << 20, **mixed) == (LONG, 1, 1, 0, 0)
    assert attn_plan(lib, d=96, **mixed) == (LONG, 1, 1, 0, 0)
    assert attn_plan(lib, d=256, **mixed) == (ROWS16, 1, 1, 0, 0)
    assert attn_plan(lib, bits=64, **mixed) == (ROWS16_DMA, 1, 1, 0, 0)
    # the query without type and strides covers any of them
    assert lib.fxpr_attention_workspace_bytes(21, 140, 32, 8, 128, 32, 0, 120, 190, 16) == want
    assert lib.fxpr_attention_workspace_bytes(21, 140, 32, 8, 128, 32, 0, 120, 380, 8) == 0
    # a decode batch: the plain policy's splits, with either kernel
    decode = dict(requests=64, tokens=64, max_q=1, keys=8192)
    assert attn_plan(lib, **decode) == (ROWS16_DMA, 16, 16, 0, record_bytes(64, 8192))
    assert attn_plan(lib, dt=F32, **decode) == (ROWS16, 16, 16, 0, record_bytes(64, 8192))
    # one plan's records only: 128 tokens at 16 splits by register loads
    assert attn_plan(lib, 1, 128, 128, 8192, dt=F32) == (ROWS16, 16, 16, 0, record_bytes(128, 8192))
    assert attn_plan(lib, 0, 128, 128, 8192) == (0, 0, 0, 0, 0)


def test_attention_long_requests_over_wide_tables_stay_split(lib):
    # 512 MiB of records, 1 GiB with fewer than 128 prefill workgroups
    half, full = 1 << 29, 1 << 30
    for tokens, keys, splits in ((128, 131072, 16), (130, 131072, 16), (250, 131072, 9)):
        n = record_bytes(tokens, keys)
        assert half < n <= full
        assert attn_plan(lib, 1, tokens, tokens, keys) == (LONG_DMA, splits, 1, 0, n), tokens
        # (the register-load kernels: as many records, 64 splits)
        assert attn_plan(lib, 1, tokens, tokens, keys, dt=F32) == (ROWS16, 64, 64, 0, n), tokens
    assert attn_plan(lib, 1, 64, 64, 131072)[1] == 32                          # 260 MiB
    for tokens, keys in ((256, 65536), (512, 32768)):
        assert half < record_bytes(tokens, keys) <= full
        assert attn_plan(lib, 1, tokens, tokens, keys) == (LONG_DMA, 1, 1, 0, 0), tokens
    # past 1 GiB nothing of it is split
    assert record_bytes(254, 262144) > full
    assert attn_plan(lib, 1, 254, 254, 262144) == (LONG_DMA, 1, 1, 0, 0)
    assert attn_plan(lib, 1, 256, 256, 131072) == (LONG_DMA, 1, 1, 0, 0)
    assert attn_plan(lib, 1, 256, 256, 131072, dt=F32) == (ROWS16, 1, 1, 0, 0)
    # and only where the 16-row kernels would split the batch as well
    assert half < record_bytes(130, 131072) <= full
    assert attn_plan(lib, 80, 130, 12, 131072)[1:] == (16, 1, 0, record_bytes(130, 131072))
    assert attn_plan(lib, 90, 130, 12, 131072)[1:] == (1, 1, 0, 0)
    # a chunk beside 31 decode steps; above the cap the decode steps keep
    # records of their own tokens only
    assert attn_plan(lib, 32, 543, 512, 28672) == (LONG_DMA, 4, 2, 0, record_bytes(543, 28672))
    assert half < record_bytes(543, 30720) <= full
    assert attn_plan(lib, 32, 543, 512, 30720) == (LONG_DMA, 1, 2, 11, record_bytes(32 * 11, 30720))


def test_attention_batches_of_equal_long_requests_keep_no_short_records(lib):
    # nothing for short requests where every request has the longest one's
    # tokens; the prefill rows' own splits are not affected
    assert attn_plan(lib, 4, 4 * 2048, 2048, 131072) == (LONG_DMA, 1, 1, 0, 0)
    assert attn_plan(lib, 1, 512, 512, 131072) == (LONG_DMA, 1, 1, 0, 0)     # records of 512 tokens: 2 GiB
    assert attn_plan(lib, 1, 64, 64, 32768) == (LONG_DMA, 32, 1, 0, record_bytes(64, 32768))
    # one token less (some request is shorter), and one more (padding)
    for tokens in (4 * 2048 - 1, 4 * 2048 + 1):
        assert attn_plan(lib, 4, tokens, 2048, 16384) == (LONG_DMA, 1, 32, 11, record_bytes(4 * 11, 16384))
        # a wide table: long on average is taken for all long
        assert attn_plan(lib, 4, tokens, 2048, 131072) == (LONG_DMA, 1, 1, 0, 0)
    assert attn_plan(lib, 4, 500 + 599, 500, 16400)[1:3] == (1, 32)    # others of 199.7 tokens on average
    assert attn_plan(lib, 4, 500 + 600, 500, 16400)[1:3] == (1, 1)     # of 200


def test_attention_short_requests_splits(lib):
    # a 100-token chunk beside decode steps, 7 chunks: runs of chunks while the
    # short requests' workgroups number 512 or fewer, unsplit from there on
    for requests, splits in ((2, 7), (16, 7), (64, 7), (65, 1), (300, 1)):
        assert attn_plan(lib, requests, requests + 99, 100, 3584)[2] == splits, requests
    assert attn_plan(lib, 64, 163, 100, 16384)[2] == 16                # 32 chunks, runs of two
    # beyond 16384 keys: 512 workgroups (1024 for up to 64), at most 64 splits
    for requests, splits in ((2, 64), (8, 16), (9, 8), (16, 4), (33, 2), (63, 2), (64, 1), (300, 1)):
        assert attn_plan(lib, requests, requests + 99, 100, 65536)[2] == splits, requests


def test_attention_few_rows_take_the_16_row_split(lib):
    # up to 256 rows (tokens x group) and 3000 units over tables of up to 16384
    # keys, where the plain policy splits: its launch, long requests included
    assert attn_plan(lib, 3, 28, 26, 2528) == (ROWS16_DMA, 5, 5, 0, record_bytes(28, 2528))
    assert attn_plan(lib, 1, 64, 64, 4096)[0] == ROWS16_DMA             # 256 rows
    assert attn_plan(lib, 1, 65, 65, 4096)[0] == LONG_DMA
    assert attn_plan(lib, 1, 64, 64, 11264)[0] == ROWS16_DMA            # 8 x 17 x 22 = 2992 units
    assert attn_plan(lib, 1, 64, 64, 11264 + 16)[0] == LONG_DMA         # 23 chunks: 3128
    assert attn_plan(lib, 3, 28, 26, 2048)[0] == LONG_DMA               # nothing splits
    assert attn_plan(lib, 3, 28, 26, 32768)[0] == LONG_DMA              # wide
    assert attn_plan(lib, 3, 28, 26, 2528, requested=2)[0] == LONG_DMA  # explicit


def test_attention_small_windows(lib):
    # windows of up to 2048 keys leave 3 chunks (of 1024 keys) per row: prefill
    # rows split below 141 workgroups, short requests below 128
    w = dict(window=1024)
    assert attn_plan(lib, 1, 118, 118, 2112, **w) == (LONG_DMA, 3, 1, 0, record_bytes(118, 2112))
    assert attn_plan(lib, 1, 280, 280, 8192, **w)[1:3] == (3, 1)        # 140 workgroups
    assert attn_plan(lib, 1, 282, 282, 8192, **w)[1:3] == (1, 1)
    assert attn_plan(lib, 15, 300, 250, 8192, **w)[2] == 3              # 120 short workgroups
    assert attn_plan(lib, 16, 300, 250, 8192, **w)[2] == 1
    # a table that splits nothing, a wider window, and one without causality
    assert attn_plan(lib, 1, 118, 118, 2048, **w)[1:3] == (1, 1)
    plain = attn_plan(lib, 2, 282, 281, 8192)
    assert attn_plan(lib, 2, 282, 281, 8192, window=2049) == plain
    assert attn_plan(lib, 2, 282, 281, 8192, causal=0, **w) == plain
    # the bound without the window covers every plan
    for requests, tokens, max_q in ((1, 118, 118), (3, 28, 26), (15, 300, 250), (40, 128, 89), (2, 282, 281)):
        for keys in (2112, 8192, 16384, 65536, 131072):
            bound = lib.fxpr_attention_workspace_bytes(requests, tokens, 32, 8, 128, 32, 0, max_q, -(-keys // 16), 16)
            for kw in (dict(), w, dict(window=100), dict(window=4096), dict(causal=0, **w), dict(dt=F32)):
                assert attn_plan(lib, requests, tokens, max_q, keys, **kw)[-1] <= bound, (requests, keys, kw)


def test_attention_kernels_by_the_longest_requests_rows(lib):
    # 64-row workgroups from 48 rows per kv head on; the 33 to 47 rows that fill
    # three 16-row tiles as well stay on the 16-row kernels: by LDS DMA at
    # head_dim 128 (or when split), by register loads at 64
    for heads, kv_heads, below, first in ((32, 8, (9, 10, 11), 12), (16, 16, (33, 40, 47), 48), (24, 8, (11, 15), 16),
                                          (28, 4, (5, 6), 7)):
        for d in (64, 128):
            shape = dict(heads=heads, kv_heads=kv_heads, d=d, keys=2048)
            for n in (1, 32 * kv_heads // heads, *below):
                want = ROWS16 if d == 64 and n in below else ROWS16_DMA
                assert attn_plan(lib, 8, 8 * n, n, **shape)[0] == want, (heads, d, n)
                assert attn_plan(lib, 8, 8 * n, n, requested=2, **shape)[0] == ROWS16_DMA, (heads, d, n)
                assert attn_plan(lib, 8, 8 * n, n, bits=64, **shape)[0] == ROWS16_DMA, (heads, d, n)
                assert attn_plan(lib, 8, 8 * n, n, page=8, **shape)[0] == ROWS16, (heads, d, n)
            assert attn_plan(lib, 8, 8 * first, first, **shape)[0] == LONG_DMA, heads
            assert attn_plan(lib, 8, 8 * first, first, page=8, **shape)[0] == LONG, heads


BF16, F16, F32 = 1, 0, 2


def gemm_splits(lib, m, n, k, dt=BF16, requested=0, bits=32):
    return lib.fxpr_gemm_splits(m, n, k, dt, bits, requested)


def test_gemm_explicit_request_wins(lib):
    # forced counts (the reference's _SPLITK_FORCE): honoured, clamped to the
    # K-tiles (128 wide for 16-bit inputs, 64 for fp32)
    assert gemm_splits(lib, 32, 4096, 4096, requested=4) == 4
    assert gemm_splits(lib, 1, 4096, 4096, requested=2) == 2          # even on a stream shape
    assert gemm_splits(lib, 8192, 128256, 4096, requested=3) == 3     # and a large one
    assert gemm_splits(lib, 32, 4096, 4096, requested=100) == 32      # 32 K-tiles
    assert gemm_splits(lib, 32, 4096, 4096, F32, requested=100) == 64
    assert gemm_splits(lib, 32, 4096, 128, requested=4) == 1          # one K-tile: never split
    assert gemm_splits(lib, 32, 4096, 0, requested=4) == 1
    assert gemm_splits(lib, 32, 4096, 129, requested=4) == 2          # a partial second tile


def test_gemm_auto_decode_shapes_stream(lib):
    # 16-bit, M <= 16, N <= 8192: the streaming kernel, never split
    for m in (1, 8, 16):
        for n in (1024, 4096, 6144, 8192):
            for k in (4096, 14336):
                assert gemm_splits(lib, m, n, k) == 1
                assert gemm_splits(lib, m, n, k, F16) == 1


def test_gemm_auto_split_fills_the_gpu(lib):
    # elsewhere: 512 / (output tiles) splits, at most 16, when the tiles do
    # not reach 256 (16 x 256 tiles for M <= 16; from M = 17 to 64 64 x 256
    # with 16- / 32-bit sums and 128 x 128 with 64-bit ones; 128 x 128 from
    # M = 65)
    assert gemm_splits(lib, 16, 8193, 4096) == 15        # 33 tiles
    assert gemm_splits(lib, 1, 28672, 4096) == 4         # 112 tiles
    assert gemm_splits(lib, 1, 128256, 4096) == 1        # 501 tiles
    assert gemm_splits(lib, 32, 4096, 4096) == 16        # 16 tiles
    assert gemm_splits(lib, 32, 6144, 4096) == 16        # 24 tiles
    assert gemm_splits(lib, 32, 28672, 4096) == 4        # 112 tiles
    assert gemm_splits(lib, 64, 28672, 4096, bits=16) == 4
    assert gemm_splits(lib, 32, 28672, 4096, bits=64) == 2    # 224 tiles
    assert gemm_splits(lib, 32, 6144, 4096, bits=64) == 10    # 48 tiles
    assert gemm_splits(lib, 65, 28672, 4096) == 2        # 224 tiles
    assert gemm_splits(lib, 256, 4096, 4096) == 8        # 64 tiles
    assert gemm_splits(lib, 32, 128256, 4096) == 1       # 501 tiles
    assert gemm_splits(lib, 8192, 128256, 4096) == 1
    assert gemm_splits(lib, 32, 4096, 256) == 2          # capped at the 2 K-tiles
    # fp32 inputs up to M = 32 (tiles of 256 columns, 64-wide K-tiles), and a
    # shape that fills the GPU unsplit
    assert gemm_splits(lib, 1, 4096, 4096, F32) == 16
    assert gemm_splits(lib, 32, 14336, 4096, F32) == 9   # 56 tiles
    assert gemm_splits(lib, 8192, 14336, 4096, F32) == 1


def test_gemm_workspace_follows_the_split(lib):
    # integer partials [splits, M, N] (4 or 8 bytes), none when unsplit
    assert lib.fxpr_gemm_workspace_bytes(32, 4096, 4096, BF16, 32, 0) == 16 * 32 * 4096 * 4
    assert lib.fxpr_gemm_workspace_bytes(32, 4096, 4096, BF16, 64, 0) == 16 * 32 * 4096 * 8
    assert lib.fxpr_gemm_workspace_bytes(1, 4096, 4096, BF16, 32, 0) == 0
    assert lib.fxpr_gemm_workspace_bytes(1, 4096, 4096, BF16, 32, 3) == 3 * 4096 * 4
    assert lib.fxpr_gemm_workspace_bytes(8192, 128256, 4096, BF16, 32, 0) == 0


def test_gemm_f32_split_fills_whole_rounds(lib):
    # fp32 beyond M = 32: the count whose 32- or 64-row tiles fall most evenly
    # on 256 CUs (f32_plan); rows that cannot be 16-byte aligned (K not a
    # multiple of 4) keep 512 / (output tiles)
    assert gemm_splits(lib, 256, 4096, 4096, F32) == 4       # 256 tiles of 32 rows: 4 on every CU
    assert gemm_splits(lib, 64, 6144, 4096, F32) == 8        # 96: 3 on every CU
    assert gemm_splits(lib, 130, 4096, 14336, F32) == 8      # 160: 5 on every CU
    assert gemm_splits(lib, 777, 14336, 4096, F32) == 1
    assert gemm_splits(lib, 130, 4096, 4098, F32) == 8       # 64 tiles of 128 x 128
    assert gemm_splits(lib, 130, 4096, 100, F32) <= 2        # 2 K-tiles


def test_gemm_layout_splits(lib):
    def layout(m, n, k, dt=BF16, bits=32, frac=16, lda=None, row_major=False, ldb=None):
        lda, ldb = lda or k, ldb or (n if row_major else k)
        bk, bn = (ldb, 1) if row_major else (1, ldb)
        return lib.fxpr_gemm_layout_splits(m, n, k, dt, bits, frac, lda, bk, bn)

    # K-contiguous operands: the shape's own count
    for m, n, k in ((1, 4096, 4096), (16, 8193, 4096), (32, 28672, 4096), (130, 4096, 14336)):
        for dt in (BF16, F32):
            assert layout(m, n, k, dt) == gemm_splits(lib, m, n, k, dt)
    # a row-major B at M <= 16: a row of the large-M kernel's tiles (32 of them)
    assert layout(1, 4096, 4096, row_major=True) == 16 and gemm_splits(lib, 1, 4096, 4096) == 1
    assert layout(16, 28672, 4096, row_major=True) == 4
    assert layout(17, 4096, 4096, row_major=True) == gemm_splits(lib, 17, 4096, 4096)
    # 64-bit sums at f = 32 beyond 8192 columns: the skinny tile's (56 tiles of 256)
    assert layout(16, 14336, 4096, bits=64, frac=32, row_major=True) == 9
    assert layout(16, 14336, 4096, bits=64, frac=16, row_major=True) == 4
    assert layout(16, 8192, 4096, bits=64, frac=32, row_major=True) == 8
    # fp32: the DMA kernel's plan, or 512 / (tiles of 128 x 128) where rows cannot
    # be 16-byte aligned
    assert layout(1852, 500, 856, F32, row_major=True) == gemm_splits(lib, 1852, 500, 856, F32)
    assert layout(1852, 499, 856, F32, row_major=True) == 8          # 60 tiles
    assert layout(1852, 500, 856, F32, row_major=True, ldb=501) == 8
    assert layout(1852, 499, 856, F32, ldb=857) == 8
    assert layout(1852, 499, 856, F32, lda=858) == 8
    assert layout(1852, 499, 856, F32) == gemm_splits(lib, 1852, 499, 856, F32)
    assert layout(0, 4, 4) == 1


def test_gemm_auto_decode_shapes_with_a_k_tail(lib):
    # the streaming kernel takes whole K-tiles only; other K split the skinny tile
    assert gemm_splits(lib, 1, 4096, 4096 + 16) == 16     # 16 tiles of 16 x 256
    assert gemm_splits(lib, 16, 8192, 10848) == 16        # 32 tiles
    assert gemm_splits(lib, 1, 4096, 136) == 2            # 2 K-tiles

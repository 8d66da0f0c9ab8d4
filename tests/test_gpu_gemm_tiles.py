"""The fp32 product's block tiles (32 x 32 with k over four wavefronts, 64 x 64 with k over two, 128 x 64, 128 x 128), k cut
into slices, 16-byte and single-value loads, all four storage orders: integer operands, whose sums are exact in fp32 in any
order.  The operands lie between NaNs, so that a value read from outside them and used shows."""
import ctypes

import numpy as np
import pytest

from altius_amd._lib import AltiusHipError
from conftest import assert_bits_equal

pytestmark = pytest.mark.gpu

# Sizes around the tiles' edges and k around the steps of 16, 32 and 64 values; in the second row few tiles with a long k (slices of
# 32 x 32 blocks), in the third enough tiles for the 64 x 64, 128 x 64 and 128 x 128 blocks, last ones ragged, in the fourth slices
# of 64 x 64 and of 128 x 128 blocks.
SIZES = [(1, 1, 1), (31, 33, 15), (32, 32, 64), (33, 31, 65), (65, 63, 17), (40, 36, 44),
         (1, 1000, 1024), (77, 768, 3072), (5, 130, 2052), (100, 40, 1031),
         (1024, 3072, 48), (1025, 3071, 33), (6304, 2300, 20), (6300, 3073, 37), (3300, 3200, 33),
         (551, 2305, 1481), (1411, 2516, 6162)]


def padded(rng, rows, cols, pad, offset):
    """A [rows, cols] matrix of small integers with pitch cols + pad, `offset` floats into a buffer of NaNs."""
    x = rng.integers(-3, 4, size=(rows, cols)).astype(np.float32)
    ld = cols + pad
    buf = np.full(offset + rows * ld + 64, np.nan, np.float32)
    buf[offset:offset + rows * ld].reshape(rows, ld)[:, :cols] = x
    return x, buf, ld


@pytest.mark.parametrize("trans_a", [False, True])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("pad,offset", [(0, 0), (8, 16), (3, 1)])
def test_every_tile_and_storage_order(ctx, case, trans_a, trans_b, pad, offset):
    rng = np.random.default_rng(5)
    for m, n, k in SIZES:
        case(f"gemm [{m},{k}] x [{k},{n}] trans {trans_a} {trans_b} pad {pad} offset {offset}")
        a, abuf, lda = padded(rng, *((k, m) if trans_a else (m, k)), pad, offset)
        b, bbuf, ldb = padded(rng, *((n, k) if trans_b else (k, n)), pad, offset)
        bias = rng.integers(-3, 4, size=n).astype(np.float32)
        da, db, dbias = ctx.upload(abuf), ctx.upload(bbuf), ctx.upload(bias)
        ldc = n + pad
        dc = ctx.upload(np.full(m * ldc, 7.0, np.float32))
        try:
            for _ in range(2):  # a cut tile's counters are ready for the next launch
                ctx.gemm_raw(dc.ptr, da.ptr + 4 * offset, db.ptr + 4 * offset, dbias.ptr, 1, m, n, k, trans_a, trans_b, lda, ldb, ldc,
                             c0_rs=0, c0_cs=1, alpha=2.0, beta=1.0)
                got = ctx.download(dc, (m, ldc))
                want = 2.0 * np.matmul((a.T if trans_a else a).astype(np.float64), (b.T if trans_b else b).astype(np.float64)) + bias
                assert_bits_equal(np.ascontiguousarray(got[:, :n]), want.astype(np.float32), "product")
                assert np.all(got[:, n:] == 7.0), "a store outside the result"
        finally:
            for x in (da, db, dc, dbias):
                ctx.free(x)


def test_batches_with_two_strides_and_infinities(ctx, case):
    case("gemm batches [3, 4] of [70, 20] x [20, 40], an infinity against zeros past k")
    rng = np.random.default_rng(6)
    bo, bi, m, n, k = 3, 4, 70, 40, 20
    a = rng.integers(-3, 4, size=(bo, m, bi, k)).astype(np.float32)  # heads side by side in a row
    b = rng.integers(-3, 4, size=(bi, k, n)).astype(np.float32)      # shared by the outer axis
    a[0, 0, 0, 0], a[0, 1, 0, k - 1] = np.inf, np.inf
    b[:, 0, :] = np.abs(b[:, 0, :]) + 1
    b[:, k - 1, :] = np.abs(b[:, k - 1, :]) + 1
    da, db, dc = ctx.upload(a), ctx.upload(b), ctx.alloc(4 * bo * bi * m * n)
    S = ctypes.c_size_t * 2
    try:
        rc = ctx.L.ahip_gemm_batch2(ctx.handle, dc.ptr, da.ptr, db.ptr, None, bo, bi, m, n, k, 0, 0, bi * k, n, n, S(m * bi * k, k), S(0, k * n),
                                    S(bi * m * n, m * n), 0, 0, 1.0, 0.0)
        assert rc == 0
        want = np.matmul(a.transpose(0, 2, 1, 3).astype(np.float64), b.astype(np.float64)).astype(np.float32)
        assert_bits_equal(ctx.download(dc, want.shape), want, "product")
    finally:
        for x in (da, db, dc):
            ctx.free(x)


@pytest.mark.parametrize("axis", ["m", "k"])
def test_rows_too_far_apart_for_32_bit_offsets(ctx, case, axis):
    """Rows 2 GiB apart: taken a few at a time (m), or summed in parts (k)."""
    case(f"gemm rows 2 GiB apart along {axis}")
    rows, w, n = 3, 6, 5
    ld = (1 << 29) + 64
    da = ctx.alloc(4 * ((rows - 1) * ld + w))
    rng = np.random.default_rng(7)
    x = rng.integers(-3, 4, size=(rows, w)).astype(np.float32)
    m, k, trans = (rows, w, False) if axis == "m" else (w, rows, True)
    b = rng.integers(-3, 4, size=(k, n)).astype(np.float32)
    c0 = rng.integers(-3, 4, size=(m, n)).astype(np.float32)
    db, dc0, dc = ctx.upload(b), ctx.upload(c0), ctx.alloc(4 * m * n)
    try:
        for r in range(rows):
            row = np.ascontiguousarray(x[r])
            assert ctx.L.ahip_h2d_async(ctx.handle, da.ptr + 4 * r * ld, row.ctypes.data, row.nbytes) == 0
            ctx.sync()
        ctx.gemm_raw(dc.ptr, da.ptr, db.ptr, dc0.ptr, 1, m, n, k, trans, False, ld, n, n, c0_rs=n, c0_cs=1, alpha=1.0, beta=1.0)
        want = np.matmul((x.T if trans else x).astype(np.float64), b.astype(np.float64)) + c0
        assert_bits_equal(ctx.download(dc, (m, n)), want.astype(np.float32), "product")
    finally:
        for d in (da, db, dc0, dc):
            ctx.free(d)


def test_more_products_than_a_grid_holds_are_refused(ctx, case):
    """A block of 256 threads at least for each: 2^24 of them are 2^32 threads, one more than a grid holds.  Eight fewer (one for each XCD) run."""
    batch = 1 << 24
    case(f"gemm batch of {batch} [1,1] x [1,1]")
    x = np.arange(batch, dtype=np.float32)
    da, dc = ctx.upload(x), ctx.upload(np.zeros(batch, np.float32))
    try:
        with pytest.raises(AltiusHipError, match="more tiles than a grid holds"):
            ctx.gemm_raw(dc.ptr, da.ptr, da.ptr, None, batch, 1, 1, 1, True, False, a_bs=1, b_bs=0, c_bs=1, alpha=2.0)
        ctx.gemm_raw(dc.ptr, da.ptr, da.ptr + 4, None, batch - 8, 1, 1, 1, True, False, a_bs=1, b_bs=0, c_bs=1, alpha=2.0)
        got = ctx.download(dc, (batch,))
        assert np.array_equal(got[:-8], 2.0 * x[:-8]) and not got[-8:].any()
    finally:
        ctx.free(da)
        ctx.free(dc)


def test_more_columns_than_a_grid_of_small_tiles_holds(ctx, case):
    """2^29 columns are 2^24 tiles of 32 x 32, 2^32 threads: one more than a grid holds."""
    n, period = 1 << 29, 1 << 22
    case(f"gemm [1,1] x [1,{n}]")
    x = np.random.default_rng(8).integers(-9, 10, size=period).astype(np.float32)
    da, db, dc = ctx.upload(np.full(1, 3.0, np.float32)), ctx.alloc(4 * n), ctx.alloc(4 * n)
    try:
        for start in range(0, n, period):
            assert ctx.L.ahip_h2d_async(ctx.handle, db.ptr + 4 * start, x.ctypes.data, x.nbytes) == 0
        ctx.sync()
        ctx.gemm_raw(dc.ptr, da.ptr, db.ptr, None, 1, 1, n, 1, False, False, 1, n, n, c0_rs=0, c0_cs=0, alpha=1.0, beta=0.0)
        for start in (0, n // 2 - period, n // 2, n - period):
            assert_bits_equal(ctx.download(dc, (period,), offset_bytes=4 * start), 3.0 * x, f"columns from {start}")
    finally:
        for d in (da, db, dc):
            ctx.free(d)


# The tiles that the sizes above leave out, ragged, and k around as many steps as a block has stages (3 of 64 x 64: 32 values each, of
# 128 x 64: 16; 4 of 128 x 128: 16): fewer, as many, one more, each with and without a rest.
TURNS = ([(1646, 132, k) for k in (15, 31, 32, 64, 96, 97, 128, 140)] + [(2300, 1300, k) for k in (16, 32, 48, 50, 64)] +
         [(325, 3735, 2506), (834, 3482, 700), (9001, 2500, 64), (9001, 2500, 83)])


@pytest.mark.parametrize("trans_a", [False, True])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("pad,offset", [(0, 0), (3, 1)])
def test_stages_in_turn(ctx, case, trans_a, trans_b, pad, offset):
    rng = np.random.default_rng(8)
    for m, n, k in TURNS:
        case(f"gemm [{m},{k}] x [{k},{n}] trans {trans_a} {trans_b} pad {pad} offset {offset}")
        a, abuf, lda = padded(rng, *((k, m) if trans_a else (m, k)), pad, offset)
        b, bbuf, ldb = padded(rng, *((n, k) if trans_b else (k, n)), pad, offset)
        da, db, dc = ctx.upload(abuf), ctx.upload(bbuf), ctx.alloc(4 * m * n)
        try:
            ctx.gemm_raw(dc.ptr, da.ptr + 4 * offset, db.ptr + 4 * offset, None, 1, m, n, k, trans_a, trans_b, lda, ldb, n)
            want = np.matmul(a.T if trans_a else a, b.T if trans_b else b)  # whole numbers below 2^24: exact in any order
            assert_bits_equal(ctx.download(dc, (m, n)), want, "product")
        finally:
            for x in (da, db, dc):
                ctx.free(x)


def test_more_steps_than_32_bit_offsets_reach(ctx, case):
    """Rows of k next to each other that take 4.3 GB, in two batches so that k stays whole: the offsets are counted from a later tile again."""
    block_rows, n, m = 4096, 1028, 3
    k = 257 * block_rows - 13
    case(f"gemm [{m},{k}] x [{k},{n}]")
    rng = np.random.default_rng(9)
    block = rng.integers(-1, 2, size=(block_rows, n)).astype(np.float32)
    a = rng.integers(-1, 2, size=(2 * m, k)).astype(np.float32)
    da, db, dc = ctx.upload(a), ctx.alloc(4 * k * n), ctx.alloc(8 * m * n)
    try:
        want = np.zeros((2 * m, n))
        for r in range(0, k, block_rows):
            rows = min(block_rows, k - r)
            assert ctx.L.ahip_h2d_async(ctx.handle, db.ptr + 4 * r * n, block.ctypes.data, 4 * rows * n) == 0
            want += np.matmul(a[:, r:r + rows], block[:rows])
        ctx.sync()
        ctx.gemm_raw(dc.ptr, da.ptr, db.ptr, None, 2, m, n, k, a_bs=m * k, c_bs=m * n)
        assert_bits_equal(ctx.download(dc, (2 * m, n)), want.astype(np.float32), "product")
    finally:
        for x in (da, db, dc):
            ctx.free(x)


# whole rounds of tiles and a last one that is cut along k, in two to eight slices and for every tile, ragged; then sizes that are one cut round
@pytest.mark.parametrize("m,n,k", [(1536, 1536, 1536), (2500, 2000, 1000), (2499, 1999, 1001), (3152, 768, 3072), (1100, 1000, 4100), (4200, 2100, 2050), (9000, 300, 1030),
                                   (197, 768, 3072), (77, 768, 3072), (300, 200, 1100)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_last_round_cut_along_k(ctx, case, m, n, k, trans_b):
    case(f"gemm [{m},{k}] x [{k},{n}] trans_b {trans_b}")
    rng = np.random.default_rng(m)
    a, b = (rng.integers(-3, 4, size=s).astype(np.float32) for s in ((m, k), (n, k) if trans_b else (k, n)))
    res = rng.integers(-3, 4, size=(m, n)).astype(np.float32)
    da, db, dr, dc = ctx.upload(a), ctx.upload(b), ctx.upload(res), ctx.upload(np.full((m, n), 7.0, np.float32))
    # float32 products of integers below 2^24 are exact in any order, BLAS's too
    want = np.matmul(a, b.T if trans_b else b)
    try:
        for _ in range(3):
            ctx.gemm_raw(dc.ptr, da.ptr, db.ptr, dr.ptr, 1, m, n, k, trans_b=trans_b, c0_rs=n, c0_cs=1, alpha=1.0, beta=1.0)
            assert_bits_equal(ctx.download(dc, (m, n)), want + res, "product and residual")
    finally:
        for x in (da, db, dr, dc):
            ctx.free(x)


@pytest.mark.parametrize("trans_a", [False, True])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("m,n", [(1, 1), (33, 70), (1646, 132), (1025, 3071), (6300, 3073)])
def test_sums_of_nothing(ctx, case, m, n, trans_a, trans_b):
    """k = 0: no operand is read (there is none), and the result is beta C0, or zeros."""
    case(f"gemm [{m},0] x [0,{n}] trans {trans_a} {trans_b}")
    c0 = np.random.default_rng(m).integers(-9, 10, size=(m, n)).astype(np.float32)
    d0, dc = ctx.upload(c0), ctx.upload(np.full((m, n), 7.0, np.float32))
    try:
        ctx.gemm_raw(dc.ptr, None, None, d0.ptr, 1, m, n, 0, trans_a, trans_b, m if trans_a else 1, 1 if trans_b else n, n, c0_rs=n, c0_cs=1, alpha=3.0, beta=2.0)
        assert_bits_equal(ctx.download(dc, (m, n)), 2.0 * c0, "C0")
        ctx.gemm_raw(dc.ptr, None, None, None, 1, m, n, 0, trans_a, trans_b, m if trans_a else 1, 1 if trans_b else n, n)
        assert_bits_equal(ctx.download(dc, (m, n)), np.zeros((m, n), np.float32), "zeros")
    finally:
        ctx.free(d0)
        ctx.free(dc)

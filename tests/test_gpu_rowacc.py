"""The row accumulator (short rows sorted in groups, long rows summed slab by
slab, one-owner rows copied) at the sizes where its kernels change course,
against the CPU oracle: indices bit-exact, values within REL_TOL of FP64
(relative to the sum of |products| when signed); count-only runs give the same
counts and value sum."""
import numpy as np
import pytest

from gsparc_amd import sptc
from gsparc_amd.coo import COOTensor
from helpers import compare_with_oracle

pytestmark = pytest.mark.gpu


def build(rng, K, rows, signed=False):
    """X (rows x C) and Y (C x K) such that row r has len(rows[r]) owners, the
    i-th with a segment of rows[r][i] random distinct columns; one more
    contract index, which X does not use, holds every column once, so that the
    column ranks are exactly K."""
    segs = [n for r in rows for n in r]
    C = len(segs) + 1
    yc = np.concatenate([np.full(n, c, np.uint32) for c, n in enumerate(segs)] +
                        [np.full(K, C - 1, np.uint32)])
    yj = np.concatenate([rng.choice(K, size=n, replace=False) for n in segs] +
                        [np.arange(K)]).astype(np.uint32)
    xr = np.concatenate([np.full(len(r), i, np.uint32) for i, r in enumerate(rows)])
    def vals(n):
        v = (rng.random(n) + 0.05).astype(np.float32)
        return v * np.where(rng.random(n) < 0.5, -1, 1).astype(np.float32) if signed else v
    o = rng.permutation(len(yc))
    X = COOTensor((len(rows), C), [xr, np.arange(C - 1, dtype=np.uint32)], vals(C - 1))
    Y = COOTensor((C, K), [yc[o], yj[o]], vals(len(yc)))
    return X, Y


def check(X, Y, accumulator=0):
    res = sptc.SpTC(X, Y, [1], [0], dense_accumulator=-1)
    assert res.info.accumulator == accumulator
    compare_with_oracle(X, Y, [1], [0], res)
    assert res.verify()[1] == 0
    c = sptc.SpTC(X, Y, [1], [0], dense_accumulator=-1, count_only=True)
    assert c.nnz == res.nnz and c.ir_nnz == res.ir_nnz
    scale = abs(res.info.value_sum) + 1.0
    assert abs(c.info.value_sum - res.info.value_sum) <= 1e-12 * scale * max(1, res.ir_nnz) ** 0.5
    return res


SHORT = [[1], [1, 1], [2, 3], [127, 128], [128, 128], [128, 129], [255], [256], [257], [1] * 256,
         [1] * 257, [300, 200], [768, 768], [767, 768, 1], [768, 769], [500, 500, 536],
         [500, 500, 537], [3], [1500, 36], [1500, 37]]


@pytest.mark.parametrize("K", [2, 64, 3000, 32768, 32769, 200_000])
def test_short_rows_and_group_edges(gpu, K):
    """Rows on both sides of the short limit (256 products up to 2^15 columns,
    K / 128 to 1536 above) and groups cut at multiples of 1536 products."""
    rng = np.random.default_rng(K)
    rows = [[min(n, K) for n in r] for r in SHORT * 3]
    check(*build(rng, K, rows, signed=K % 2 == 1))


@pytest.mark.parametrize("K", [65535, 65536, 65537, 98305, 131_073, (1 << 20) - 1, 1 << 20,
                               (1 << 20) + 1])
def test_long_rows_at_slab_edges(gpu, K):
    """Column spaces around one slab's 2^16 columns, up to the widest that is
    cut into slabs (2^20) and one wider (its long rows take the product sort); rows on both sides
    of the even and the product-following cut (12288 products) and of
    multiples of an item's 7168."""
    rng = np.random.default_rng(K)
    rows = [[2000, 100], [6144, 6144], [6144, 6145], [7168, 7168], [9000, 9000, 9000], [64] * 80,
            [30_000, 5, 5], [1700], [20_000]]
    check(*build(rng, K, rows, signed=True))


def test_windows_of_a_slab(gpu):
    """Slabs with more outputs than slots (5632): whole columns, then windows
    of them; a slab whose outputs fill the slots exactly."""
    rng = np.random.default_rng(3)
    rows = [[10_000, 10_000], [30_000, 12_000], [5632, 1], [5631, 1], [40_000, 40_000, 40_000]]
    check(*build(rng, 60_000, rows))


@pytest.mark.parametrize("owners,per", [(511, 20), (512, 20), (513, 20), (1300, 20), (3000, 3),
                                        (4000, 1), (255, 60), (257, 60)])
def test_many_owners(gpu, owners, per):
    """Owners in several batches of 512 (sum) and 256 (count), runs of one to
    some products per owner (units of 2 to 16 lanes)."""
    rng = np.random.default_rng(owners)
    rows = [[per] * owners, [int(n) for n in rng.integers(1, 2 * per + 1, owners)], [5, 900]]
    check(*build(rng, 30_000, rows, signed=owners % 2 == 1))


def test_bitmaps_not_kept(gpu):
    """Few products per row over 2^20 columns: the slabs' bitmaps would take
    more memory than the products are worth and are marked again."""
    rng = np.random.default_rng(8)
    check(*build(rng, 1 << 20, [[900, 900], [1000, 600, 700]] * 60))


def test_heavy_row_goes_to_the_product_sort(gpu):
    """270,000 products of one row over 1000 columns: too much for one
    workgroup, the chunk takes the product sort."""
    rng = np.random.default_rng(9)
    check(*build(rng, 1000, [[900] * 300, [5, 6], [700]]))


@pytest.mark.parametrize("rows,owners,per,K,sorted_", [
    (1, 6000, 1, 40, False), (1, 8000, 1, 40, True), (1, 75, 1000, 1000, False),
    (1, 85, 1000, 1000, True), (30, 85, 1000, 1000, False), (30, 135, 1000, 1000, True),
    (2, 12_000, 2, 40, True),
    (1, 3000, 8, 70_000, False), (1, 20_000, 2, 70_000, True)])
def test_heavy_items_on_both_sides_of_the_line(gpu, rows, owners, per, K, sorted_):
    """An item's weight is its products and 11 per owner: above 81920 and a 64th of
    the chunk's products the chunk takes the product sort, as above 2^17 products."""
    rng = np.random.default_rng(owners)
    X, Y = build(rng, K, [[per] * owners] * rows + [[5, 6]], signed=True)
    check(X, Y)
    st = sptc.SpTC(X, Y, [1], [0], dense_accumulator=-1, kernel_timing=True).kernel_stats()
    assert (st["sort_products"][0] + st["sort_products_wide"][0] > 0) == sorted_


def test_fallback_chunk_beside_others_under_a_budget(gpu):
    """A budget that cuts the products into chunks; the first holds a row that
    sends it to the product sort, the others take the row accumulator.  The
    sort's buffers and the accumulator's tables do not fit together.  Results as
    without a budget."""
    import torch

    class Dev:
        pass

    def dev(dims, idx, val):
        t = Dev()
        t.dims, t.order, t.nnz = dims, len(dims), len(val)
        t.idx = [torch.from_numpy(i.astype(np.int32)).cuda() for i in idx]
        t.val = torch.from_numpy(val.astype(np.float32)).cuda()
        return t

    rng = np.random.default_rng(12)
    K, heavy, C, N, per = 1000, 300, 300, 1_500_000, 8
    xr = np.concatenate([np.zeros(heavy, np.int64), 1 + np.repeat(np.arange(N), 2)])
    xc = np.concatenate([np.arange(heavy), heavy + rng.integers(0, C, 2 * N)])
    yc = np.concatenate([np.repeat(np.arange(heavy), 900), heavy + np.repeat(np.arange(C), per)])
    yj = np.concatenate([rng.choice(K, 900, replace=False) for _ in range(heavy)] +
                        [rng.choice(K, per, replace=False) for _ in range(C)])
    X = dev((N + 1, heavy + C), [xr, xc], rng.random(len(xr)) + 0.1)
    Y = dev((heavy + C, K), [yc, yj], rng.random(len(yc)) + 0.1)
    run = lambda **kw: sptc.SpTC(X, Y, [1], [0], dense_accumulator=-1, on_device=True, **kw)
    free = run()
    want = free.to_host()
    chunks = set()
    for f in (0.8, 0.9, 1.0, 1.1):
        r = run(mem_budget_bytes=int(f * 35 * free.ir_nnz) + 44 * len(xr), kernel_timing=True)
        chunks.add(r.info.nchunks)
        st = r.kernel_stats()
        assert st["sort_products"][0] + st["sort_products_wide"][0] > 0  # the first chunk
        for a, b in zip(r.to_host(), want):
            np.testing.assert_array_equal(a, b)
    assert min(chunks) > 1 and max(chunks) > 2


def test_duplicate_columns_of_one_owner(gpu):
    """Y with duplicate coordinates: one-owner rows are summed like others."""
    rng = np.random.default_rng(10)
    X, Y = build(rng, 4000, [[1], [40], [300], [3000], [20, 30], [2500, 700]])
    d = rng.choice(Y.nnz, 3000, replace=False)
    Y = COOTensor(Y.dims, [np.concatenate([a, a[d]]) for a in Y.idx],
                  np.concatenate([Y.val, Y.val[d] * np.float32(0.5)]))
    check(X, Y)


def test_signed_zero_infinity_and_nan(gpu):
    """A product of -0 is emitted as +0 (a sum starts at +0); infinities and
    NaN arrive as the FP64 sum of the products gives them, in one-owner, short
    and long rows."""
    rng = np.random.default_rng(11)
    X, Y = build(rng, 3000, [[50], [60, 60], [1500, 1500]])
    X.val[:] = -1.0
    Y.val[rng.random(Y.nnz) < 0.3] = 0.0
    Y.val[rng.random(Y.nnz) < 0.05] = np.inf
    Y.val[rng.random(Y.nnz) < 0.05] = -np.inf
    Y.val[rng.random(Y.nnz) < 0.02] = np.nan
    xf, yf, v = sptc.SpTC(X, Y, [1], [0], dense_accumulator=-1).to_host()
    want = {}
    by_c = {}
    for c, j, y in zip(Y.idx[0], Y.idx[1], Y.val):
        by_c.setdefault(int(c), []).append((int(j), y))
    with np.errstate(invalid="ignore"):
        for r, c, x in zip(X.idx[0], X.idx[1], X.val):
            for j, y in by_c[int(c)]:
                want[(int(r), j)] = want.get((int(r), j), 0.0) + np.float64(np.float32(x * y))
    keys = sorted(want)
    np.testing.assert_array_equal(np.stack([xf, yf], 1).astype(np.int64), np.array(keys))
    w = np.array([want[k] for k in keys]).astype(np.float32)
    np.testing.assert_array_equal(v, w)  # NaN where NaN
    assert not np.signbit(v[v == 0]).any()


@pytest.mark.parametrize("K", [40, 1 << 20, (1 << 20) + 1, 1 << 21, (1 << 21) + 1, (1 << 22) + 5])
def test_wide_columns_and_sparse_rows(gpu, K):
    """Short and one-owner rows over column spaces that are not cut into slabs
    (keys of 32 and of 64 bits in the groups), found among rows without
    products (more rows than active X nonzeros, then fewer); and one row too
    long for such a space, which takes the chunk to the product sort."""
    rng = np.random.default_rng(K)
    rows = [[min(n, K) for n in r] for r in SHORT * 2]
    for empty in (3000, 0):
        mixed = rows + [[0]] * empty
        mixed = [mixed[i] for i in rng.permutation(len(mixed))]
        check(*build(rng, K, mixed, signed=True))
    check(*build(rng, K, rows + [[min(1536, K)] * 2, [0]], signed=True))

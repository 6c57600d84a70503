"""SpGEMM at the edges of its tiers: 16 lanes per row, a wave, a dense
accumulator of each size, the tables beyond it; rows with empty partners, hubs
of more than a staged chunk, more than 32,768 products in a row."""
import numpy as np
import pytest
import scipy.sparse as sp

import apspie_amd as A

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with A.Context(0) as c:
        yield c


def _rows(lengths, n, rng):
    """CSR with rows of these lengths, sorted distinct columns, values 1..4."""
    ind = [np.sort(rng.choice(n, k, replace=False)) for k in lengths]
    ptr = np.concatenate([[0], np.cumsum(lengths)])
    col = np.concatenate(ind).astype(np.int32)
    return sp.csr_matrix((rng.integers(1, 5, len(col)).astype(np.float64), col, ptr),
                         shape=(len(lengths), n))


def _product(ctx, a, b):
    ga, gb = (ctx.upload(x.indptr.astype(np.int32), x.indices.astype(np.int32),
                         x.data.astype(np.float32), n=x.shape[1]) for x in (a, b))
    gc = ctx.spgemm(ga, gb)
    got = gc.download(values=True)
    for g in (ga, gb, gc):
        g.close()
    return got


def _same(got, want):
    want.sort_indices()
    assert np.array_equal(got[0], want.indptr)
    assert np.array_equal(got[1], want.indices)
    assert np.array_equal(got[2], want.data.astype(np.float32))


@pytest.mark.parametrize("n", [5, 17, 1000, 4096, 4097, 8192, 8193, 16384, 16385, 32768, 32769])
def test_tiers_exact(ctx, n):
    rng = np.random.default_rng(n)
    k = 2100
    # B: empty rows, single entries, short rows and a few long ones
    lens = np.minimum(n, rng.choice([0, 1, 2, 4, 16, 100], k))
    lens[:12] = min(n, 5000)
    b = _rows(lens, n, rng)
    # A: row lengths round the 16 lanes, the wave's 64 entries and the chunk of
    # 1024, each over random partners and over the long ones first
    lengths = [0, 1, 2, 3, 8, 15, 16, 17, 18, 33, 63, 64, 65, 130, 1023, 1024, 1025, 2100] * 6
    a = _rows(lengths, k, rng)
    _same(_product(ctx, a, b), (a @ b).tocsr())


@pytest.mark.parametrize("entries", [1, 4, 15, 16, 17])
def test_tiny_rows_with_shared_columns(ctx, entries):
    """Rows of `entries` partners with one product each, or none, all products
    of a row on few columns; 15 to 18 and 63 to 66 products in a row."""
    rng = np.random.default_rng(entries)
    b = sp.vstack([_rows([1] * 40, 3, rng), _rows([0] * 20, 3, rng)]).tocsr()
    b.resize(60, 40)
    a = _rows([entries] * 333, 60, rng)
    _same(_product(ctx, a, b), (a @ b).tocsr())
    for total in (15, 16, 17, 18, 63, 64, 65, 66):
        wide = _rows([total - 1, 1, 0], 90, rng)
        rows = _rows([3, 2, 1, 1] * 9, 3, rng)
        _same(_product(ctx, rows, wide), (rows @ wide).tocsr())


@pytest.mark.parametrize("n", [3000, 16384, 32768])
def test_float_sums_against_64_bits(ctx, n):
    """Positive terms: T rounded products added one by one in 32 bits, in any
    order, are within (T + 1) 2^-24 of the exact sum."""
    rng = np.random.default_rng(n + 1)
    b = _rows(np.minimum(n, rng.choice([3, 40, 2500], 900)), n, rng)
    a = _rows([2, 5, 30, 200, 900] * 5, 900, rng)
    for x in (a, b):
        x.data = (1.0 - rng.random(x.nnz)).astype(np.float32).astype(np.float64)
    got = _product(ctx, a, b)
    want = (a @ b).tocsr()
    want.sort_indices()
    ones = [sp.csr_matrix((np.ones(x.nnz), x.indices, x.indptr), shape=x.shape) for x in (a, b)]
    terms = (ones[0] @ ones[1]).tocsr()
    terms.sort_indices()
    assert np.array_equal(got[0], want.indptr) and np.array_equal(got[1], want.indices)
    err = np.abs(got[2].astype(np.float64) - want.data) / want.data
    assert np.all(err <= (terms.data + 1) * 2.0 ** -24)


def test_autotune_leaves_bounds_that_move_no_row():
    """4096 vertices: the bit-per-vertex triangle count and the dense accumulator
    take all rows the bounds would bin, so their values stay the caller's."""
    rp, c = A.gen_rmat(12)
    with A.Context(0) as ctx:
        G = ctx.upload(rp, c, np.ones(len(c), np.float32))
        mine = {"tc_medium_row": 700, "spgemm_wave_ub": 100, "spgemm_block_ub": 3000}
        for name, v in mine.items():
            ctx.set_option(name, v)
        ctx.autotune_hash(G)
        assert ctx.get_option("tc_medium_row") == 700
        if ctx.get_option("spgemm_dense"):  # else the tables win, and are tuned
            assert {k: ctx.get_option(k) for k in mine} == mine
        ctx.set_option("spgemm_dense", 0)
        ctx.autotune_hash(G)
        assert ctx.get_option("spgemm_wave_ub") in (64, 128, 256)
        assert ctx.get_option("spgemm_block_ub") in (1024, 2048, 4096)
        G.close()

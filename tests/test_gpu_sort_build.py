"""Scan, radix sort and the graph build at the edges of their tiles, and the
build's row starts over long runs of empty rows: exact against numpy and the
oracle."""
import ctypes as C

import numpy as np
import pytest

import apspie_amd as A
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with A.Context(0) as c:
        yield c


# tiles of 1024 elements up to 65,536, of 4096 above
@pytest.mark.parametrize("n", [1023, 1024, 1025, 65_535, 65_536, 65_537, 69_632, 4096 * 70 + 3])
@pytest.mark.parametrize("shift", [0, 1])
def test_scan_tiles_and_alignment(ctx, n, shift):
    """shift 1: device arrays 4 bytes off a 16-byte line."""
    x = np.random.default_rng(n).integers(-50, 100, n).astype(np.int32)
    din, dout = ctx.dev_alloc(4 * n + 16), ctx.dev_alloc(4 * n + 16)
    L, tot = A.lib(), C.c_int64()
    A._check(L.apspie_memcpy(ctx.h, din.ptr + 4 * shift, x.ctypes.data, x.nbytes, 0), ctx.h)
    A._check(L.apspie_scan_exclusive(ctx.h, din.ptr + 4 * shift, dout.ptr + 4 * shift, n,
                                     C.byref(tot), A.DEVICE), ctx.h)
    out = np.empty(n, np.int32)
    A._check(L.apspie_memcpy(ctx.h, out.ctypes.data, dout.ptr + 4 * shift, out.nbytes, 1), ctx.h)
    want = np.cumsum(x, dtype=np.int64) - x
    assert np.array_equal(out, want.astype(np.int32)) and tot.value == int(x.sum())
    din.free()
    dout.free()


# tiles of 4096 pairs, dealt out by XCD from 8 tiles on
@pytest.mark.parametrize("n", [2, 511, 4095, 4096, 4097, 8 * 4096, 9 * 4096 + 1, 4096 * 37 - 5])
@pytest.mark.parametrize("bits", [1, 8, 9, 20, 32])
def test_sort_tiles(ctx, n, bits):
    rng = np.random.default_rng(n + bits)
    hi = 1 << bits
    keys = np.minimum(rng.integers(0, hi, n), rng.integers(0, hi, n)).astype(np.uint32)
    keys[rng.integers(0, n, n // 3)] = hi - 1  # a digit that most lanes share
    order = np.argsort(keys, kind="stable")
    vals = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    k, v = ctx.sort_pairs(keys, vals, bits)
    assert np.array_equal(k, keys[order]) and np.array_equal(v, vals[order])
    assert np.array_equal(ctx.sort_pairs(keys, None, bits)[0], keys[order])


@pytest.mark.parametrize("m,ne", [(1, 3), (2, 1), (70, 2), (200, 300), (5000, 4096),
                                  (100_000, 5), (40_000, 30_000), (300, 20_000)])
@pytest.mark.parametrize("weighted", [False, True])
def test_build_row_starts(ctx, m, ne, weighted):
    """Loops, repeats with other values, and runs of empty rows before, between
    and after the entries (more than 64 and more than 16,384 rows long)."""
    rng = np.random.default_rng(m + ne)
    lo, hi = m // 3, max(m // 3 + 1, m - m // 4)  # empty rows at both ends
    r = rng.integers(lo, hi, ne).astype(np.int32)
    c = np.where(rng.random(ne) < 0.1, r, rng.integers(lo, hi, ne)).astype(np.int32)
    w = rng.random(ne).astype(np.float32)
    pad = np.zeros(ne, np.int32)
    r2, c2, w2 = O.symmetrize(np.concatenate([r, pad]), np.concatenate([c, pad]),
                              np.concatenate([w, np.zeros(ne, np.float32)]), ne)
    want = [O.coo_to_csr(m, r2, c2, w2), O.coo_to_csr(m, r, c, w)]
    for sym, (wrp, wc, wv) in zip((True, False), want):
        G = ctx.from_coo(m, r, c, w if weighted else None, symmetrize=sym)
        rp, cc, vv = G.download(values=True)
        assert np.array_equal(rp, wrp) and np.array_equal(cc, wc)
        assert np.array_equal(vv, wv if weighted else np.ones_like(wv))
        Tr = G.transpose()
        back = Tr.transpose()
        rt, ct, vt = back.download(values=True)
        if sym:  # rows sorted already: the double transpose is the same graph
            assert np.array_equal(rt, rp) and np.array_equal(ct, cc) and np.array_equal(vt, vv)
        else:    # rows come back sorted by column, repeats in input order
            rows = np.repeat(np.arange(m), np.diff(rp))
            order = np.lexsort((np.arange(len(cc)), cc, rows))
            assert np.array_equal(rt, rp) and np.array_equal(ct, cc[order])
            assert np.array_equal(vt, vv[order])
        for x in (back, Tr, G):
            x.close()


def test_build_refuses_an_index_out_of_range(ctx):
    for r, c in ((5, 0), (0, 5), (-1, 0), (0, -1)):
        for sym in (True, False):
            with pytest.raises(A.ApspieError):
                ctx.from_coo(5, [1, r, 2], [2, c, 3], symmetrize=sym)


@pytest.mark.parametrize("n", [1, 1024, 1025, 2048, 5000, 65_536, 65_537, 400_001])
@pytest.mark.parametrize("lo,hi", [(-100, 0), (-100, 100), (-(1 << 31), -(1 << 30))])
def test_scan_of_negative_values(n, lo, hi):
    """Prefixes that are negative at a tile's edge: the 64-bit total and the
    low words of the prefixes."""
    x = np.random.default_rng(n).integers(lo, hi, n).astype(np.int32)
    want = np.cumsum(x, dtype=np.int64)
    with A.Context(0) as ctx:
        out, total = ctx.scan_exclusive(x)
        assert total == want[-1]
        assert np.array_equal(out, np.concatenate([[0], want[:-1]]).astype(np.int32))

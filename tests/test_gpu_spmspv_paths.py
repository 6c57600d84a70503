"""The SpMSpV's choice of path and its sizes: products on and around one
block's sort, the sort path's limit, repeated frontier entries, and scratch
that holds no dense row.  The sort path is a sequential fold, so it is
bit-identical to the oracle on any values."""
import numpy as np
import pytest

import apspie_amd as A
from oracle import oracle as O

pytestmark = pytest.mark.gpu

N = 600_000  # so that 65,536 products still sort (products * 8 < N)
ROWS = 70_000


@pytest.fixture(scope="module")
def thin():
    """One entry in each of the first ROWS rows, many in a few columns."""
    rng = np.random.default_rng(11)
    col = np.where(rng.random(ROWS) < 0.5, rng.integers(0, 40, ROWS),
                   rng.integers(0, N, ROWS)).astype(np.int32)
    rp = np.concatenate([np.arange(ROWS + 1), np.full(N - ROWS, ROWS)]).astype(np.int64)
    return rp, col, rng.random(ROWS).astype(np.float32)


@pytest.mark.parametrize("nx", [1, 64, 2048, 2049, 4095, 4096, 4097, 12_289, 65_536, 65_537])
@pytest.mark.parametrize("sr", [A.SR_PLUS_TIMES, A.SR_BOOL, A.SR_MIN_PLUS, A.SR_MAX_FIRST])
def test_products_around_the_limits(thin, nx, sr):
    rp, col, a = thin
    rng = np.random.default_rng(nx)
    # empty rows among the entries, before, between and after
    x = np.sort(np.concatenate([rng.choice(ROWS, nx, replace=False),
                                ROWS + rng.choice(N - ROWS, 300, replace=False)]))
    xv = (rng.random(len(x)) - 0.3).astype(np.float32)
    mask = (rng.random(N) < 0.2).astype(np.int32)
    with A.Context(0) as ctx:
        G = ctx.upload(rp.astype(np.int32), col, a)
        for mk in (None, mask):
            wi, wv = O.spmspv(N, rp, col, a, sr, x, xv, mk)
            for path in (A.PATH_AUTO, A.PATH_SORT, A.PATH_ATOMIC):
                yi, yv = ctx.spmspv(G, sr, x, xv, mk, path)
                assert np.array_equal(yi, wi)
                fold = path == A.PATH_SORT or (path == A.PATH_AUTO and nx <= 65_536)
                if fold or sr != A.SR_PLUS_TIMES:
                    assert np.array_equal(yv, wv)
                else:  # up to about 1,000 values below 0.7 a column, in any order:
                    # 1,000 roundings of a sum below 700
                    assert np.allclose(yv, wv, rtol=0, atol=1000 * 700 * 2.0 ** -24)
        G.close()


@pytest.mark.parametrize("path", [A.PATH_AUTO, A.PATH_SORT, A.PATH_ATOMIC])
def test_repeated_frontier_entries(path):
    """More expanded edges than the matrix has entries."""
    m, d = 5000, 50
    rp = np.concatenate([[0], np.full(m, d)]).astype(np.int64)  # row 0 only
    col = np.sort(np.random.default_rng(1).choice(m, d, replace=False)).astype(np.int32)
    a = np.arange(1, d + 1, dtype=np.float32)
    x = np.zeros(3000, np.int32)
    xv = np.ones(3000, np.float32)
    with A.Context(0) as ctx:
        G = ctx.upload(rp.astype(np.int32), col, a)
        yi, yv = ctx.spmspv(G, A.SR_PLUS_TIMES, x, xv, None, path)
        assert np.array_equal(yi, col) and np.array_equal(yv, 3000 * a)
        G.close()


def test_scratch_without_room_for_a_dense_row(thin):
    """An AUTO call that sorts needs no dense row; one that does not is
    refused when the row does not fit."""
    rp, col, a = thin
    with A.Context(0) as ctx:
        G = ctx.upload(rp.astype(np.int32), col, a)
        ctx.reserve_arena(2 * 4 * N + (2 << 20))  # the host call's outputs and little more
        x = np.arange(0, 3000, dtype=np.int32)
        yi, yv = ctx.spmspv(G, A.SR_PLUS_TIMES, x)
        wi, wv = O.spmspv(N, rp, col, a, A.SR_PLUS_TIMES, x)
        assert np.array_equal(yi, wi) and np.array_equal(yv, wv)
        with pytest.raises(A.ApspieError) as e:
            ctx.spmspv(G, A.SR_PLUS_TIMES, np.arange(66_000, dtype=np.int32))
        assert e.value.status == -4
        G.close()


def test_a_sorting_call_leaves_a_budget_alone(thin):
    """Under a budget with room for the dense row, a call that sorts does not
    take it: what fitted beside it before still does.  A call that needs the row
    gets it, and those after it find it there."""
    rp, col, a = thin
    rng = np.random.default_rng(5)
    x = np.sort(rng.choice(ROWS, 50, replace=False))
    xv = rng.random(len(x)).astype(np.float32)
    every = np.arange(ROWS, dtype=np.int32)
    with A.Context(0) as ctx:
        G = ctx.upload(rp.astype(np.int32), col, a)
        ctx.spmspv(G, A.SR_BOOL, every, path=A.PATH_SORT)  # every other buffer
        want = ctx.spmspv(G, A.SR_PLUS_TIMES, x, xv, path=A.PATH_SORT)
        used = ctx.hbm_used()
        ctx.set_hbm_budget(used + 5 * N)
        for _ in range(2):
            got = ctx.spmspv(G, A.SR_PLUS_TIMES, x, xv)
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
            assert ctx.hbm_used() < used + N
        H = ctx.upload(np.arange(N + 1, dtype=np.int32) // 8, np.zeros(N // 8, np.int32))
        H.close()
        ctx.set_hbm_budget(used + 5 * N)
        for _ in range(2):
            yi, yv = ctx.spmspv(G, A.SR_MIN_PLUS, every, None)
            wi, wv = O.spmspv(N, rp, col, a, A.SR_MIN_PLUS, every, np.ones(ROWS, np.float32), None)
            assert np.array_equal(yi, wi) and np.array_equal(yv, wv)
            assert ctx.hbm_used() > used + 4 * N
        got = ctx.spmspv(G, A.SR_PLUS_TIMES, x, xv)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        G.close()

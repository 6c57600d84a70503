"""MIS with its last rounds in one block: candidate counts and entries round
the block's limits (2048 and 16,384), one round per vertex on chains, rows of
a graph that is not symmetric."""
import numpy as np
import pytest

import apspie_amd as A

pytestmark = pytest.mark.gpu


def _rounds(m, rp, col, prio):
    """Luby rounds: who beats every undecided row entry joins, its undecided
    entries leave (ties to the lower id)."""
    key = (prio.astype(np.uint64) << np.uint64(32)) | (0x7fffffff - np.arange(m)).astype(np.uint64)
    row = np.repeat(np.arange(m), np.diff(rp))
    state = np.where(np.diff(rp) == 0, 1, -1)
    live = np.where(state == -1, key, 0).astype(np.uint64)
    while (state == -1).any():
        und = state == -1
        lost = np.zeros(m, bool)
        lost[row[live[col] > live[row]]] = True
        win = und & ~lost
        state[win] = 1
        live[win] = 0
        out = col[win[row]]
        out = out[state[out] == -1]
        state[out] = 0
        live[out] = 0
    return state


def _symmetric(m, u, v):
    pairs = np.unique(np.concatenate([np.stack([u, v], 1), np.stack([v, u], 1)]), axis=0)
    rp = np.concatenate([[0], np.cumsum(np.bincount(pairs[:, 0], minlength=m))]).astype(np.int32)
    return rp, pairs[:, 1].astype(np.int32)


def _check(m, rp, col, prio):
    with A.Context(0) as c:
        g = c.upload(rp, col)
        want = _rounds(m, rp, col, prio)
        for _ in range(2):
            assert np.array_equal(c.mis(g, prio), want)
        g.close()


@pytest.mark.parametrize("m", [2, 63, 1000, 2047, 2048, 2049, 40_000])
def test_rising_chain(m):
    """Priorities rise along a path: every round decides two vertices."""
    u = np.arange(m - 1)
    rp, col = _symmetric(m, u, u + 1)
    prio = np.arange(m, dtype=np.uint32)
    if m == 40_000:  # rising in runs of 500
        prio = ((np.arange(m) % 500) * 100 + np.arange(m) // 500).astype(np.uint32)
    _check(m, rp, col, prio)


@pytest.mark.parametrize("m,deg", [(2048, 8), (2048, 7), (1500, 11), (1500, 10), (600, 27),
                                   (600, 100), (9000, 4), (100_000, 6), (300_000, 5)])
def test_random_graphs_at_the_limits(m, deg):
    rng = np.random.default_rng(m + deg)
    u, v = rng.integers(0, m, (2, m * deg // 2))
    rp, col = _symmetric(m, u[u != v], v[u != v])
    _check(m, rp, col, rng.integers(0, 50 if deg % 2 else 1 << 32, m).astype(np.uint32))


@pytest.mark.parametrize("m,deg", [(1800, 9), (5000, 7), (50_000, 12)])
def test_rows_that_are_not_symmetric(m, deg):
    rng = np.random.default_rng(m)
    rp = (np.arange(m + 1) * deg).astype(np.int32)
    col = rng.integers(0, m, m * deg).astype(np.int32)
    _check(m, rp, col, rng.integers(0, 1 << 32, m).astype(np.uint32))

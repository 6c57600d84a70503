"""Triangle counts at the lengths where a row changes kernels (16, 128 lower
neighbours; chunks of 512) and at the vertex counts where the long rows do
(2^18, 2^20).  Totals and per-row counts equal the oracle's."""
import numpy as np
import pytest

import apspie_amd as A
from oracle import oracle as O
from tests import graphs as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1500, 1 << 18, (1 << 18) + 1, 1 << 20, (1 << 20) + 1])
@pytest.mark.parametrize("lens", [(1, 2, 3, 15, 16, 17), (127, 128, 129), (511, 512, 513),
                                  (1023, 1024, 1025)])
def test_rows_at_tier_edges(m, lens):
    """Row h near the top has lens[h] lower neighbours, spread over all the
    vertices below; those are joined among each other at random."""
    rng = np.random.default_rng(m + sum(lens))
    hubs = m - 1 - np.arange(len(lens))
    below = m - len(lens) - 1
    pool = np.unique(np.concatenate([[0, 31, 32, below],
                                     rng.choice(below, 1100, replace=False)]))
    u, v = [], []
    for h, d in zip(hubs, lens):
        u.append(np.full(d, h))
        v.append(rng.choice(pool, d, replace=False))
    a, b = rng.choice(pool, 30_000), rng.choice(pool, 30_000)
    u.append(a[a != b])
    v.append(b[a != b])
    rp, c = O.edges_to_csr(m, np.concatenate(u).astype(np.int32),
                           np.concatenate(v).astype(np.int32))
    want, want_rows = O.tc(m, rp, c)
    assert want > 0
    with A.Context(0) as ctx:
        G = ctx.upload(rp.astype(np.int32), c)
        for _ in range(2):
            total, rows = ctx.tc(G)
            assert total == want and np.array_equal(rows, want_rows)
        assert ctx.tc(G, per_row=False)[0] == want
        G.close()


@pytest.mark.parametrize("key", ["lattice", "rmat"])
def test_rows_counted(key):
    """vertices_reached is the number of rows with two lower neighbours or
    more, whichever kernel takes them."""
    rp, c = A.gen_lattice(60) if key == "lattice" else A.gen_rmat(12)
    rows = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    lower = np.bincount(rows[c < rows], minlength=len(rp) - 1)
    with A.Context(0) as ctx:
        G = ctx.upload(rp, c)
        ctx.tc(G)
        assert ctx.stats()["vertices_reached"] == int((lower >= 2).sum())
        G.close()


def _wheel():
    """Two hubs, the second one in the middle: 19,998 and 9,000 lower neighbours."""
    n = 20000
    rim = np.arange(n - 2)
    u = np.concatenate([rim[:-1], rim, np.full(9000, 9000)])
    v = np.concatenate([rim[1:], np.full(n - 2, n - 1), np.arange(9001, 18001)])
    return n, *O.edges_to_csr(n, u.astype(np.int32), v.astype(np.int32))


def _hubs():
    """300 hubs joined to 4,700 others and to each other: 4,700 to 4,999 lower
    neighbours each."""
    n = 5000
    a, b = np.triu_indices(300, 1)
    u = np.concatenate([np.repeat(np.arange(n - 300, n), n - 300), a + n - 300])
    v = np.concatenate([np.tile(np.arange(n - 300), 300), b + n - 300])
    return n, *O.edges_to_csr(n, u.astype(np.int32), v.astype(np.int32))


@pytest.mark.parametrize("medium_row", [128, 256, 512, 1024, 2048])
@pytest.mark.parametrize("key", ["rmat14", "wheel", "hubs"])
def test_hash_tables_above_the_bits(key, medium_row):
    """With more than 2^20 vertices (most of them isolated, above the others)
    the long rows take the hash tables: in LDS for the 256- and the 1024-thread
    blocks, and above 16,384 lower neighbours in global memory."""
    if key == "rmat14":
        g = T.rmat(14)
        n, rp, c = g.m, g.rowptr, g.col
    else:
        n, rp, c = _wheel() if key == "wheel" else _hubs()
    m = (1 << 20) + 1
    rp = np.concatenate([rp, np.full(m - n, rp[-1])]).astype(np.int64)
    rows = np.repeat(np.arange(m), np.diff(rp))
    longest = np.bincount(rows[c < rows], minlength=m).max()
    assert longest > {"rmat14": 1024, "wheel": 16_384, "hubs": 4096}[key]
    want, want_rows = O.tc(m, rp, c)
    with A.Context(0) as ctx:
        ctx.set_option("tc_medium_row", medium_row)
        G = ctx.upload(rp.astype(np.int32), c)
        total, got = ctx.tc(G)
        assert total == want > 0 and np.array_equal(got, want_rows)
        assert ctx.tc(G, per_row=False)[0] == want
        G.close()

"""Triangle counts at the lengths where a row changes kernels (16, 128 lower
neighbours; chunks of 512) and at the vertex counts where the long rows do
(2^18, 2^20).  Totals and per-row counts equal the oracle's."""
import numpy as np
import pytest

import apspie_amd as A
from oracle import oracle as O

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

"""The load-balanced expansion at the edges of its shares: frontiers whose
expanded edge count falls on, just under and just over a share, a tile and
what fills the grid, against the oracle (bit-exact)."""
import numpy as np
import pytest

import apspie_amd as A
from oracle import oracle as O
from tests import graphs as T

pytestmark = pytest.mark.gpu


def broom(k, d, extra):
    """Vertex 0 joined to k others, each with d leaves (the first of them
    `extra` more); the second level then expands k * (d + 1) + extra edges."""
    mids = np.arange(1, k + 1, dtype=np.int32)
    n = 1 + k + k * d + extra
    u = np.concatenate([np.zeros(k, np.int32), np.repeat(mids, d), np.ones(extra, np.int32)])
    v = np.concatenate([mids, np.arange(1 + k, n, dtype=np.int32)])
    rp, c = O.edges_to_csr(n, u, v)
    return T.G(f"broom{k}_{d}_{extra}", n, rp, c)


# shares of 256, 512 and 1024 edges and whole tiles of 2048, on 512 blocks
@pytest.mark.parametrize("k,d", [(1, 255), (1, 2047), (5, 50), (64, 31), (128, 1023),
                                 (256, 1023), (700, 1), (2048, 0)])
@pytest.mark.parametrize("extra", [0, 1])
def test_shares_of_a_level(k, d, extra):
    g = broom(k, d, extra)
    with A.Context(0) as ctx:
        G = ctx.upload(g.rowptr32, g.col, g.w)
        want, _ = O.bfs(g.m, g.rowptr, g.col, 0)
        wd = O.sssp(g.m, g.rowptr, g.col, g.w, 0)
        wd = np.where(wd == -1, A.SSSP_INF, wd).astype(np.float32)
        for direction in (0, 1):
            ctx.set_option("bfs_direction", direction)
            assert np.array_equal(ctx.bfs(G, 0), want)
        for delta in (0, 64):
            ctx.set_option("sssp_delta", delta)
            assert np.array_equal(ctx.sssp(G, 0), wd)
        assert np.array_equal(ctx.bfs_batch(G, [0, 1])[0], want)
        assert np.array_equal(ctx.sssp_batch(G, [0, 1])[0], wd)
        G.close()


@pytest.mark.parametrize("ahead", [1, 2, 8, 64])
@pytest.mark.parametrize("key", ["lattice64", "rmat12", "path300", "one"])
def test_loops_at_any_run_ahead(ahead, key):
    """Level loops whose host side runs 1 to 24 levels ahead of the device,
    from a single vertex (no level has work) to hundreds of levels, call after
    call on one context."""
    g = {"lattice64": lambda: T.lattice(64), "rmat12": lambda: T.rmat(12),
         "path300": lambda: T.path_graph(300), "one": lambda: T.empty_graph(1)}[key]()
    with A.Context(0) as ctx:
        ctx.set_option("bfs_levels_per_sync", ahead)
        G = ctx.upload(g.rowptr32, g.col, g.w)
        for src in (0, g.m // 2, g.m - 1):
            want, _ = O.bfs(g.m, g.rowptr, g.col, src)
            wd = O.sssp(g.m, g.rowptr, g.col, g.w, src)
            wd = np.where(wd == -1, A.SSSP_INF, wd).astype(np.float32)
            for direction in (1, 0):
                ctx.set_option("bfs_direction", direction)
                assert np.array_equal(ctx.bfs(G, src), want)
            for delta in (0, 32, 200):
                ctx.set_option("sssp_delta", delta)
                assert np.array_equal(ctx.sssp(G, src), wd)
        G.close()

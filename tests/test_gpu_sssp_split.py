"""Light / heavy splits that move most vertices of a graph without isolated
ones: the frontier gets one entry per vertex, which is all it has room for."""
import numpy as np
import pytest

import apspie_amd as A
from oracle import oracle as O
from tests.test_nearfar_entries import hub_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [1024, 2048, 4096])
@pytest.mark.parametrize("m", [65, 1000, 70_001])
def test_split_moves_every_vertex(m, tile):
    rp, c, w = hub_graph(m, 4)
    with A.Context(0) as ctx:
        ctx.set_option("bfs_tile", tile)
        ctx.set_option("sssp_delta", 100)
        G = ctx.upload(rp.astype(np.int32), c, w)
        for src in (0, 1, m - 1):
            assert np.array_equal(ctx.sssp(G, src), O.sssp(m, rp, c, w, src))
            if src == 0:  # the hub, then every other vertex once
                assert ctx.stats()["vertices_reached"] == m
        G.close()


@pytest.mark.parametrize("delta", [72, 80, 96])
def test_uniform_rows(delta):
    """Rows of about 32 entries, weights 1..255: splits that move a large part
    of the vertices, all of them with light and heavy entries."""
    m = 1 << 14
    rng = np.random.default_rng(delta)
    rp, c = O.edges_to_csr(m, rng.integers(0, m, 16 * m).astype(np.int32),
                           rng.integers(0, m, 16 * m).astype(np.int32))
    w = O.assign_weights(m, rp, c)
    with A.Context(0) as ctx:
        ctx.set_option("sssp_delta", delta)
        G = ctx.upload(rp.astype(np.int32), c, w)
        for src in (0, m // 2):
            assert np.array_equal(ctx.sssp(G, src), O.sssp(m, rp, c, w, src))
        G.close()


@pytest.mark.parametrize("m,near_far", [((3 << 18) - 1, False), (3 << 18, True)])
def test_default_width_of_longer_rows(m, near_far):
    """Graphs whose weights split into light and heavy take near-far rounds
    from 3 * 2^18 vertices on.  Bellman-Ford rounds from the hub are two (the hub,
    then all others once); a split is a round more."""
    rp, c, w = hub_graph(m, 4)
    with A.Context(0) as ctx:
        G = ctx.upload(rp.astype(np.int32), c, w)
        assert np.array_equal(ctx.sssp(G, 0), np.where(np.arange(m) == 0, 0, 200))
        assert (ctx.stats()["iterations"] != 2) == near_far
        G.close()


@pytest.mark.parametrize("mean,most", [(4, 0.7), (8, 0.5)])
def test_default_width_of_large_random_graphs(mean, most):
    """2^22 vertices, short rows, short paths: a bucket as wide as the paths
    would re-expand what Bellman-Ford rounds do (at most 0.4 of it at the
    weights' own width)."""
    m = 1 << 22
    rng = np.random.default_rng(mean)
    u, v = rng.integers(0, m, (2, m * mean // 2), dtype=np.int32)
    w = rng.integers(1, 256, len(u)).astype(np.float32)
    with A.Context(0) as ctx:
        G = ctx.from_coo(m, u, v, w)
        got = ctx.sssp(G, int(u[0]))
        edges = ctx.stats()["edges_traversed"]
        ctx.set_option("sssp_delta", 0)
        assert np.array_equal(got, ctx.sssp(G, int(u[0])))
        assert edges < most * ctx.stats()["edges_traversed"]
        G.close()


@pytest.mark.parametrize("kind", ["lattice", "rmat"])
def test_default_width_gives_way_to_a_budget(kind):
    """Where only Bellman-Ford rounds fit the budget the default takes those; a
    width that was asked for is refused."""
    rp, c = A.gen_lattice(900) if kind == "lattice" else A.gen_rmat(20)
    w = A.gen_weights(rp, c)
    m, src = len(rp) - 1, int(np.argmax(np.diff(rp)))
    with A.Context(0) as ctx:
        G = ctx.upload(rp, c, w)
        out = ctx.dev_alloc(4 * m)
        ctx.set_option("sssp_delta", 0)
        ctx.sssp(G, src, out=out.ptr, mem=A.DEVICE)
        want = out.to_host(np.float32, m)
        need = ctx.hbm_used()
        ctx.trim()
        ctx.set_hbm_budget(need)
        ctx.set_option("sssp_delta", 64)
        with pytest.raises(A.ApspieError):
            ctx.sssp(G, src, out=out.ptr, mem=A.DEVICE)
        ctx.trim()
        ctx.set_option("sssp_delta", -1)
        for _ in range(2):
            out.from_host(np.zeros(m, np.float32))
            ctx.sssp(G, src, out=out.ptr, mem=A.DEVICE)
            assert np.array_equal(out.to_host(np.float32, m), want)
        out.free()
        G.close()

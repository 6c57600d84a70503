"""Batched traversals where the frontier changes its place: pulled levels that
keep their rows in snapshots, run out of them, and go back to pushing; and
batched SSSP with source-major distances (short rows, symmetric weights, known
only after a check when the graph was built symmetrized) against vertex-major
ones.  Every source equals the single-source call, which the oracle pins."""
import numpy as np
import pytest

import apspie_amd as A
from oracle import oracle as O
from tests import graphs as T

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with A.Context(0) as c:
        yield c


@pytest.mark.parametrize("nsrc", [1, 33, 70, 200, 300])
@pytest.mark.parametrize("cap_levels", [0, 1, 3, 1000])
@pytest.mark.parametrize("key", ["lattice96", "rmat11", "comb"])
def test_bfs_levels_change_form(ctx, key, cap_levels, nsrc):
    """comb: a long path with a clique in the middle, so that levels push, pull
    and push again; the snapshot room holds cap_levels of them."""
    if key == "comb":
        k, side = 60, 200
        u, v = np.triu_indices(k, 1)
        path = np.arange(2 * side + 1)
        a = np.concatenate([u + side, path[:-1] + np.where(path[:-1] >= side, k - 1, 0)])
        b = np.concatenate([v + side, path[1:] + np.where(path[1:] > side, k - 1, 0)])
        n = 2 * side + k
        g = T.G("comb", n, *O.edges_to_csr(n, a.astype(np.int32), b.astype(np.int32)))
    else:
        g = T.lattice(96) if key == "lattice96" else T.rmat(11)
    W = next(w for w in (1, 2, 4, 8, 16) if nsrc <= 32 * w)
    rng = np.random.default_rng(nsrc)
    src = rng.integers(0, g.m, nsrc)
    G = ctx.upload(g.rowptr32, g.col)
    # whole megabytes only: the room is set through the budget left instead
    try:
        for div in (4, 1 << 20):
            ctx.set_option("batch_pull_div", div)
            with A.Context(0) as c2:
                c2.set_option("batch_pull_div", div)
                c2.set_option("batch_snapshot_mb", 0 if cap_levels == 0 else 24576)
                if 0 < cap_levels < 1000:  # a budget whose half holds cap_levels rows
                    G2 = c2.upload(g.rowptr32, g.col)
                    c2.bfs_batch(G2, src)  # every other buffer is there
                    used = c2.hbm_used()
                    row = 4 * W * g.m
                    c2.trim()
                    c2.set_hbm_budget(used + 2 * (cap_levels * row + row // 2))
                else:
                    G2 = c2.upload(g.rowptr32, g.col)
                got = c2.bfs_batch(G2, src)
                for i in range(0, nsrc, 7):
                    assert np.array_equal(got[i], ctx.bfs(G, int(src[i]))), (div, i)
    finally:
        ctx.set_option("batch_pull_div", 4)
        G.close()


@pytest.mark.parametrize("nsrc", [1, 20, 50, 128, 300])
@pytest.mark.parametrize("kind", ["symmetric", "asymmetric", "unknown"])
def test_sssp_distance_layouts(ctx, kind, nsrc):
    """A lattice uploaded with symmetric or asymmetric weights, or built
    symmetrized from triples (symmetry of the weights not known)."""
    g = T.lattice(72)
    rows = np.repeat(np.arange(g.m, dtype=np.int32), g.deg)
    w = np.asarray(g.w, np.float32)
    if kind == "unknown":
        up = rows < g.col
        G = ctx.from_coo(g.m, rows[up], g.col[up], w[up], symmetrize=True)
    else:
        if kind == "asymmetric":
            w = np.where(rows < g.col, w, w % 97 + 1).astype(np.float32)
        G = ctx.upload(g.rowptr32, g.col, w)
    rng = np.random.default_rng(nsrc)
    src = rng.integers(0, g.m, nsrc)
    try:
        for delta in (-1, 64, 3000):
            for div in (4, 0, 1 << 20):
                ctx.set_option("batch_sssp_delta", delta)
                ctx.set_option("batch_sssp_pull_div", div)
                got = ctx.sssp_batch(G, src)
                for i in range(0, nsrc, 9):
                    wd = O.sssp(g.m, g.rowptr, g.col, w, int(src[i]))
                    wd = np.where(wd == -1, A.SSSP_INF, wd).astype(np.float32)
                    assert np.array_equal(got[i], wd), (delta, div, i)
    finally:
        ctx.set_option("batch_sssp_delta", -1)
        ctx.set_option("batch_sssp_pull_div", 4)
        G.close()


@pytest.mark.parametrize("nsrc", [128, 129, 200, 260])
def test_groups_of_a_large_graph(nsrc):
    """From 2^20 vertices on, source-major SSSP splits a batch in groups of
    128: every row equals the single-source call's."""
    w = 1024
    ids = np.arange(w * w).reshape(w, w)
    u = np.concatenate([ids[:, :-1].ravel(), ids[:-1].ravel()]).astype(np.int32)
    v = np.concatenate([ids[:, 1:].ravel(), ids[1:].ravel()]).astype(np.int32)
    rng = np.random.default_rng(nsrc)
    keep = rng.random(len(u)) >= 0.1
    u, v = u[keep], v[keep]
    val = rng.integers(1, 256, len(u)).astype(np.float32)
    src = rng.choice(w * w, nsrc, replace=False).astype(np.int32)
    with A.Context(0) as c:
        G = c.from_coo(w * w, u, v, val)
        got = c.sssp_batch(G, src)
        for i in {0, 1, 127, nsrc - 1, min(128, nsrc - 1), min(256, nsrc - 1)}:
            assert np.array_equal(got[i], c.sssp(G, int(src[i])))
        G.close()


@pytest.mark.parametrize("hi", [1, 255])
def test_only_near_far_batches_are_grouped(hi):
    """Equal weights mean Bellman-Ford rounds: a batch then stays one pass, and
    300 copies of a source expand what the source alone does.  With weights
    1..255 the batch is split in three."""
    w, nsrc = 1024, 300
    ids = np.arange(w * w).reshape(w, w)
    u = np.concatenate([ids[:, :-1].ravel(), ids[:-1].ravel()]).astype(np.int32)
    v = np.concatenate([ids[:, 1:].ravel(), ids[1:].ravel()]).astype(np.int32)
    val = np.random.default_rng(1).integers(1, hi + 1, len(u)).astype(np.float32)
    src = int(ids[w // 2, w // 2])
    with A.Context(0) as c:
        G = c.from_coo(w * w, u, v, val)
        out = c.dev_alloc(4 * nsrc * w * w)
        c.sssp_batch(G, [src], out=out.ptr, mem=A.DEVICE)
        alone = c.stats()["vertices_reached"]
        c.sssp_batch(G, [src] * nsrc, out=out.ptr, mem=A.DEVICE)
        if hi == 1:
            assert alone == w * w and c.stats()["vertices_reached"] == alone
        else:
            assert c.stats()["vertices_reached"] > 2 * alone
        out.free()
        G.close()

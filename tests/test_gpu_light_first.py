"""The light-first copy of a graph's rows (near-far SSSP) at the lengths where
its row kernels change: a lane group's row, one step and several steps of a
wave, and rows for whole blocks, with all-light and all-heavy rows among them,
and weight ranges that end on the last entry.  Distances equal the oracle's."""
import numpy as np
import pytest

import apspie_amd as A
from oracle import oracle as O
from tests import graphs as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [(1, 15, 16, 17, 63, 64, 65), (255, 256, 257, 512, 513),
                                  (2047, 2048, 2049), (8191, 8192, 8193, 20_001)])
@pytest.mark.parametrize("kind", ["mixed", "light", "heavy", "last"])
def test_rows_split_by_weight(lens, kind):
    """A chain of hubs, hub h joined to lens[h] vertices of its own."""
    n = len(lens) + sum(lens)
    u, v, at = [], [], len(lens)
    for h, d in enumerate(lens):
        u.append(np.full(d, h))
        v.append(np.arange(at, at + d))
        at += d
    u.append(np.arange(len(lens) - 1))
    v.append(np.arange(1, len(lens)))
    # leaves of one hub joined to the next one's: paths that beat the hubs'
    rng = np.random.default_rng(sum(lens))
    u.append(rng.integers(len(lens), n, n))
    v.append(rng.integers(len(lens), n, n))
    rp, c = O.edges_to_csr(n, np.concatenate(u).astype(np.int32),
                           np.concatenate(v).astype(np.int32))
    g = T.G("hubs", n, rp, c)
    w = np.asarray(g.w)
    if kind == "light":
        w = np.minimum(w, 40.0)
    elif kind == "heavy":
        w = np.maximum(w, 70.0)
    elif kind == "last":  # the whole range sits in the last row
        w = np.where(np.arange(len(w)) >= g.rowptr[-2], w * 1000.0, 5.0)
    # symmetric values are not needed: the CSR is what is walked
    w = w.astype(np.float32)
    with A.Context(0) as ctx:
        G = ctx.upload(g.rowptr32, g.col, w)
        for delta in (64, 100, -1):
            ctx.set_option("sssp_delta", delta)
            for src in (0, n - 1):
                wd = O.sssp(n, g.rowptr, g.col, w, src)
                assert np.array_equal(ctx.sssp(G, src),
                                      np.where(wd == -1, A.SSSP_INF, wd).astype(np.float32))
        G.close()


@pytest.mark.parametrize("m,kind", [(887 ** 2, "lattice"), (1 << 20, "rmat")])
def test_default_width_at_its_gates(m, kind):
    """The first sizes at which the default picks near-far rounds give the
    Bellman-Ford rounds' distances."""
    rp, c = (A.gen_lattice(887) if kind == "lattice" else A.gen_rmat(20))
    w = A.gen_weights(rp, c)
    with A.Context(0) as ctx:
        G = ctx.upload(rp, c, w)
        src = int(np.argmax(np.diff(rp)))
        got = ctx.sssp(G, src)
        rounds = ctx.stats()["iterations"]
        ctx.set_option("sssp_delta", 0)
        assert np.array_equal(got, ctx.sssp(G, src))
        assert rounds != ctx.stats()["iterations"]  # the default took other rounds
        G.close()

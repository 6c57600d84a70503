"""How many entries a light / heavy split appends to the frontier, on the CPU.

The frontier of the SSSP rounds (sssp.hip k_sssp_nf_round) holds m + 1
entries.  A split moves pending vertices, each with its light and its heavy
entries, and adds the heavy entries of the marked ones.  The parts of a row
adjoin, so a moved vertex is one entry (its whole row) and a split appends at
most one entry per vertex; an entry per part would not fit on graphs where a
split moves most vertices.  The schedule is run here round by round with all
relaxations of a round at once, and both countings are taken at every split."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_nearfar_model import F32_INF, next_threshold, oracle


def split_entries(m, rowptr, col, w, src, delta):
    """(distances, most entries of a split: one per vertex, one per part)."""
    w = np.asarray(w, np.float32)
    rows = np.repeat(np.arange(m), np.diff(rowptr))
    light = w < np.float32(delta)
    has_light = np.bincount(rows[light], minlength=m) > 0
    has_heavy = np.bincount(rows[~light], minlength=m) > 0
    dist = np.full(m, F32_INF, np.float32)
    dist[src] = 0
    pend = np.zeros(m, bool)
    marked = np.zeros(m, bool)
    T = step = np.float32(delta)
    edges = np.nonzero(rows == src)[0]  # expanded this round
    split_last, left_prev, min_prev = False, 0, None
    most = parts = 0
    for _ in range(10_000):
        if edges.size:
            nd = np.full(m, F32_INF, np.float32)
            np.minimum.at(nd, col[edges], dist[rows[edges]] + w[edges])
            down = nd < dist
            dist[down] = nd[down]
            pend |= down & (nd >= T)
            near = down & (nd < T)
            marked |= near
            edges = np.nonzero(near[rows] & light)[0]
            split_last = False
            continue
        if split_last and left_prev == 0:
            return dist, most, parts
        tn, step = next_threshold(T, step, split_last and min_prev is not None, min_prev)
        take = pend & (dist >= T) & (dist < tn)
        left = pend & (dist >= tn)
        most = max(most, int(((take & (has_light | has_heavy)) | (marked & has_heavy)).sum()))
        parts = max(parts, int((take & has_light).sum() + ((take | marked) & has_heavy).sum()))
        edges = np.nonzero(take[rows] | (marked[rows] & ~light))[0]
        left_prev = int(left.sum())
        min_prev = dist[left].min() if left_prev else None
        pend, T, split_last = left, tn, True
        marked[:] = False
    raise AssertionError("did not converge")


def hub_graph(m, deg, seed=0):
    """Vertex 0 joined to all at 200; the others in a ring at 20 with deg
    chords each at 150: from 0, one split moves every other vertex."""
    rng = np.random.default_rng(seed)
    ids = np.arange(1, m)
    ring = np.r_[ids[1:], ids[0]]
    u = np.concatenate([np.zeros(m - 1, int), ids, np.repeat(ids, deg)])
    v = np.concatenate([ids, ring, rng.integers(1, m, (m - 1) * deg)])
    rp, c = O.edges_to_csr(m, u.astype(np.int32), v.astype(np.int32))
    rows = np.repeat(np.arange(m), np.diff(rp))
    near = np.abs(rows - c)
    w = np.where((rows == 0) | (c == 0), 200, np.where((near == 1) | (near == m - 2), 20, 150))
    return rp, c, w.astype(np.float32)


@pytest.mark.parametrize("kind", ["hub", "uniform"])
def test_one_entry_per_vertex(kind):
    if kind == "hub":
        m, delta = 2000, 100.0
        rp, c, w = hub_graph(m, 4)
    else:  # no isolated vertices, weights 1..255
        m, delta = 1 << 14, 80.0
        rng = np.random.default_rng(3)
        rp, c = O.edges_to_csr(m, rng.integers(0, m, 16 * m).astype(np.int32),
                               rng.integers(0, m, 16 * m).astype(np.int32))
        w = O.assign_weights(m, rp, c)
    dist, most, parts = split_entries(m, rp, c, w, 0, delta)
    assert np.array_equal(dist, oracle(m, rp, c, w, 0))
    assert most <= m
    assert parts > m + 1  # what an entry per part would append

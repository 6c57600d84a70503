"""Entry offsets at the top of their 32 bits: graphs of more than 2^30 entries,
made on the GPU, whose results are known or compared between two ways."""
import ctypes as C

import numpy as np
import pytest

import apspie_amd as A

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _from_coo(ctx, m, row, col, val):
    torch.cuda.synchronize()
    h = C.c_void_p()
    coo = A._Coo(m, m, row.numel(), row.data_ptr(), col.data_ptr(), val.data_ptr())
    A._check(A.lib().apspie_graph_from_coo(ctx.h, C.byref(coo), A.DEVICE, 1, C.byref(h)), ctx.h)
    return A.Graph(ctx, h)


def test_symmetric_weights_beyond_2_30_entries():
    """The check of a built graph's mirror values searches rows whose offsets
    pass 2^30; with it, Bellman-Ford rounds pull, and reach what pushed ones do."""
    m, k = 1 << 20, 600
    rng = np.random.default_rng(1)
    step = torch.from_numpy(rng.choice(m // 2 - 1, k, replace=False).astype(np.int32) + 1).cuda()
    row = torch.arange(m, dtype=torch.int32, device="cuda").repeat(k)
    col = (row + step.repeat_interleave(m)) % m
    val = ((row * 31 + col) % 255 + 1).float()
    with A.Context(0) as ctx:
        G = _from_coo(ctx, m, row, col, val)
        del row, col, val, step
        torch.cuda.empty_cache()
        assert G.nnz == 2 * k * m > 1 << 30
        ctx.set_option("sssp_delta", 0)
        pushed = ctx.sssp(G, 5)
        assert ctx.stats()["edges_checked"] == ctx.stats()["edges_traversed"]
        ctx.set_option("sssp_pull_div", 1 << 20)
        assert np.array_equal(ctx.sssp(G, 5), pushed)
        # pulled: the weights were found symmetric
        assert ctx.stats()["edges_checked"] != ctx.stats()["edges_traversed"]
        assert pushed[5] == 0 and pushed.max() < 255 * 8
        G.close()


TOP = (1 << 31) - 2  # the most entries a graph may have


def _wrap(ctx, m, n, rowptr, col, val=None):
    torch.cuda.synchronize()
    h = C.c_void_p()
    csr = A._Csr(m, n, col.numel(), rowptr.data_ptr(), col.data_ptr(),
                 None if val is None else val.data_ptr())
    A._check(A.lib().apspie_graph_wrap(ctx.h, C.byref(csr), C.byref(h)), ctx.h)
    return A.Graph(ctx, h)


def _long_rows(length):
    """2^31 / length rows of `length` entries, the last one two shorter: row
    (j, a) = j * stride + a leads to (j', (a * length + j) mod stride) for all
    j'.  Values 10 for the first half of a row, 200 for the second, and 3 in the
    last row."""
    m = (1 << 31) // length
    stride = m // length
    r = torch.arange(m, dtype=torch.int64, device="cuda")
    to = (((r % stride) * length + r // stride) % stride).int()
    j = torch.arange(length, dtype=torch.int32, device="cuda")
    col = (j[None, :] * stride + to[:, None]).view(-1)[:TOP]
    w = torch.where(j < length // 2, 10.0, 200.0).float()
    val = w[None, :].expand(m, length).contiguous().view(-1)[:TOP]
    val[(m - 1) * length:] = 3.0
    rowptr = torch.arange(m + 1, dtype=torch.int64, device="cuda") * length
    rowptr[m] = TOP
    return m, stride, to, w, rowptr.int(), col, val


@pytest.mark.parametrize("length", [64, 2048, 4096])
def test_light_first_rows_at_the_top(length):
    """The kernels of the light-first copy (a lane group's rows, a wave's, a
    block's) up to the last offset, by the distances of near-far rounds."""
    m, stride, to, w, rowptr, col, val = _long_rows(length)
    inf = torch.tensor(float(A.SSSP_INF), device="cuda")
    want = torch.full((m,), float(A.SSSP_INF), device="cuda")
    want[0] = 0
    last = col[(m - 1) * length:].long()
    for _ in range(100):
        into = torch.full((stride,), float(A.SSSP_INF), device="cuda")
        into.scatter_reduce_(0, to[:-1].long(), want[:-1], "amin")
        new = torch.minimum(want, torch.where(into[None, :] < inf, into[None, :] + w[:, None],
                                              inf).view(-1))
        if new[m - 1] < inf:
            new[last] = torch.minimum(new[last], new[m - 1] + 3)
        if torch.equal(new, want):
            break
        want = new
    else:
        raise AssertionError("no fixed point")
    with A.Context(0) as ctx:
        ctx.set_option("sssp_delta", 100)
        G = _wrap(ctx, m, m, rowptr, col, val)
        assert G.nnz == TOP
        out = torch.empty(m, device="cuda")
        torch.cuda.synchronize()
        ctx.sssp(G, 0, out=out.data_ptr(), mem=A.DEVICE)
        assert torch.equal(out, want)
        G.close()
    del col, val, out, want, new
    torch.cuda.empty_cache()


@pytest.mark.parametrize("width", [1, 33])
def test_product_of_rows_at_the_top(width):
    """A * B where B has entries in two rows of every A row: `width` columns
    each (the wave tier's rows, or the dense accumulator's)."""
    length = 2048
    m, stride, _, _, rowptr, col, val = _long_rows(length)
    k = np.arange(m) // stride  # the entry of A's rows that meets row k of B
    size = np.where((k == 5) | (k == 2045), width, 0)
    brp = np.concatenate([[0], np.cumsum(size)]).astype(np.int32)
    bcol = np.concatenate([np.arange(width) * 3 + 1 + (q == 2045) for q in k[size > 0]])
    with A.Context(0) as ctx:
        G = _wrap(ctx, m, m, rowptr, col, val)
        B = ctx.upload(brp, bcol.astype(np.int32), np.ones(len(bcol), np.float32), n=128)
        P = ctx.spgemm(G, B)
        rp, c, x = P.download(values=True)
        assert np.array_equal(rp, np.arange(m + 1) * 2 * width)
        one = np.sort(np.concatenate([np.arange(width) * 3 + 1, np.arange(width) * 3 + 2]))
        assert np.array_equal(c.reshape(m, -1), np.broadcast_to(one, (m, 2 * width)))
        x = x.reshape(m, -1)
        assert (x[:-1] == np.where(one % 3 == 1, 10, 200)).all() and (x[-1] == 3).all()
        for g in (P, B, G):
            g.close()
    del col, val
    torch.cuda.empty_cache()


def test_triangles_of_rows_at_the_top():
    """The lower half's rows lead to the upper half and have no lower
    neighbours; the last three have 300, about 520,000 and 200 of them."""
    m, half, length = 1 << 20, 1 << 19, 4095
    rng = np.random.default_rng(3)
    a = np.sort(rng.choice(half, 300, replace=False))
    c = np.sort(rng.choice(half, 198, replace=False))
    L = {m - 3: a, m - 1: np.concatenate([c, [m - 3, m - 2]])}
    rest = TOP - half * length - len(a) - 2 - len(L[m - 1]) - 1
    L[m - 2] = np.concatenate([np.sort(rng.choice(half, rest - 1, replace=False)), [m - 3]])
    tail = np.concatenate([L[m - 3], [m - 2, m - 1], L[m - 2], [m - 1], L[m - 1]])
    want = np.zeros(m, np.int64)
    for r in (m - 2, m - 1):
        want[r] = sum(len(np.intersect1d(L[r], L[k])) for k in (m - 3, m - 2) if k < r)
    lens = np.zeros(m, np.int64)
    lens[:half] = length
    lens[-3:] = len(a) + 2, rest + 1, len(L[m - 1])
    rowptr = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).cuda()
    r = torch.arange(half, dtype=torch.int32, device="cuda")
    j = torch.arange(length, dtype=torch.int32, device="cuda")
    col = torch.empty(TOP, dtype=torch.int32, device="cuda")
    col[:half * length] = (half + j[None, :] * 128 + (r % 128)[:, None]).view(-1)
    col[half * length:] = torch.from_numpy(tail.astype(np.int32)).cuda()
    with A.Context(0) as ctx:
        G = _wrap(ctx, m, m, rowptr, col)
        total, rows = ctx.tc(G)
        assert total == want.sum() > 0 and np.array_equal(rows, want)
        G.close()
    del col
    torch.cuda.empty_cache()

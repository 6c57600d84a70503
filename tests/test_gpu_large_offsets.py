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

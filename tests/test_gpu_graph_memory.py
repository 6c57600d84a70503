"""Arrays of destroyed graphs are kept for the next ones: the accounting, the
budget and the results are those of arrays freed at once."""
import ctypes as C
import time

import numpy as np
import pytest

import apspie_amd as A

pytestmark = pytest.mark.gpu


def _csr(m, k, seed):
    rng = np.random.default_rng(seed)
    col = np.sort(rng.integers(0, m, (m, k)), axis=1).astype(np.int32).reshape(-1)
    return (np.arange(m + 1) * k).astype(np.int32), col, rng.random(m * k, dtype=np.float32)


def _check(g, csr):
    rp, col, val = g.download(values=True)
    assert np.array_equal(rp, csr[0]) and np.array_equal(col, csr[1])
    assert np.array_equal(val, csr[2])


def test_reuse_keeps_contents_and_accounting():
    with A.Context(0) as c:
        base = c.hbm_used()
        for i, (m, k) in enumerate([(100_000, 8), (100_000, 8), (100_000, 7), (90_000, 8),
                                    (1000, 4), (100_000, 9), (262_144, 1), (100_000, 8)]):
            csr = _csr(m, k, i)
            a, b = c.upload(*csr), c.upload(*csr)
            _check(a, csr)
            a.close()
            other = _csr(m, k, 100 + i)
            a = c.upload(*other)  # on the blocks of the first
            _check(a, other)
            _check(b, csr)
            a.close()
            b.close()
            assert c.hbm_used() == base
        c.trim()
        assert c.hbm_used() == base


def test_budget_and_other_contexts():
    csr = _csr(200_000, 16, 1)  # 26 MB
    small = _csr(150_000, 2, 2)
    with A.Context(0) as c, A.Context(0) as other:
        g = c.upload(*csr)
        size = c.hbm_used()
        g.close()
        c.set_hbm_budget(size + 1000)  # kept blocks do not count against a new graph
        s = c.upload(*small)
        _check(s, small)
        with pytest.raises(A.ApspieError):
            c.upload(*csr)
        s.close()
        g = c.upload(*csr)
        h = other.upload(*csr)
        _check(g, csr)
        g.close()
        _check(h, csr)
        h.close()
    g = None
    with A.Context(0) as c:
        keep = c.upload(*csr)
        c.upload(*csr).close()
        g = c.upload(*csr)  # outlives its context, on a block given out twice
        keep.close()
    g.close()


def test_upload_refuses_without_arrays():
    """A refused upload has nothing to release: no description at all, none of
    the arrays, or a column out of range."""
    csr = _csr(100, 3, 5)
    with A.Context(0) as c:
        base = c.hbm_used()
        h = C.c_void_p()
        for arg in (None, C.byref(A._Csr(4, 4, 0, None, None, None))):
            assert A.lib().apspie_graph_upload(c.h, arg, C.byref(h)) != 0
            assert not h
        with pytest.raises(A.ApspieError):
            c.upload(csr[0], np.full_like(csr[1], 100), csr[2])
        assert c.hbm_used() == base
        g = c.upload(*csr)
        _check(g, csr)
        g.close()


@pytest.mark.parametrize("kind", ["from_coo", "transpose", "spgemm"])
@pytest.mark.parametrize("room", [0, 1, 2])
def test_refused_results_give_their_arrays_back(kind, room):
    """A result whose first `room` arrays fit the budget and whose next one is
    refused: nothing stays counted, and the call passes once there is room."""
    m, k = 300_000, 8
    rp, col, val = _csr(m, k, 3)
    rows = np.repeat(np.arange(m, dtype=np.int32), k)
    eye = np.arange(m + 1, dtype=np.int32)
    with A.Context(0) as c:
        a = c.upload(rp, col, val)
        one = c.upload(eye, eye[:-1], np.ones(m, np.float32))

        def make():
            if kind == "from_coo":
                return c.from_coo(m, rows, col, val, symmetrize=False)
            return a.transpose() if kind == "transpose" else c.spgemm(one, a)

        g = make()
        nnz = len(g.download()[1])
        g.close()  # the scratch buffers stay
        used = c.hbm_used()
        c.set_hbm_budget(used + sum([4 * (m + 1), 4 * nnz, 4 * nnz][:room]) + m)
        for _ in range(2):
            with pytest.raises(A.ApspieError):
                make()
            assert c.hbm_used() == used
        c.set_hbm_budget(0)
        g = make()
        assert c.hbm_used() == used + 4 * (m + 1) + 8 * nnz
        g.close()
        assert c.hbm_used() == used
        a.close()
        one.close()


def test_edgeless_graphs_are_counted_and_uncounted_alike():
    with A.Context(0) as c:
        none = np.zeros(0, np.int32)
        a = c.upload(np.zeros(6, np.int32), none, np.zeros(0, np.float32))
        for make in (lambda: c.from_coo(5, none, none, symmetrize=True),
                     lambda: c.from_coo(5, np.arange(5), np.arange(5), symmetrize=True),
                     a.transpose, lambda: c.spgemm(a, a)):
            make().close()
            used = c.hbm_used()
            for _ in range(2):
                g = make()
                assert len(g.download()[1]) == 0 and c.hbm_used() > used
                g.close()
                assert c.hbm_used() == used
        a.close()


def test_larger_kept_blocks_do_not_narrow_a_budget():
    """A graph that fits the budget to the byte fits it too where kept blocks up
    to an eighth larger are at hand, and counts what it counts without them."""
    large, csr = _csr(220_000, 16, 1), _csr(200_000, 16, 2)
    with A.Context(0) as c:
        g = c.upload(*csr)
        size = c.hbm_used()
        g.close()
        c.trim()
        for budget in (0, size):
            c.set_hbm_budget(0)
            c.upload(*large).close()
            c.set_hbm_budget(budget)
            g = c.upload(*csr)
            assert c.hbm_used() == size
            _check(g, csr)
            g.close()
            assert c.hbm_used() == 0


def _free_bytes():
    """Free device memory, by the runtime the library has loaded."""
    free, total = C.c_size_t(), C.c_size_t()
    assert C.CDLL("libamdhip64.so").hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _settles(cond):
    """The device returns freed memory after clearing it, a moment later."""
    for _ in range(100):
        if cond():
            return True
        time.sleep(0.02)
    return False


def test_kept_blocks_are_the_devices():
    """All contexts of a device keep 512 MB together, and a request of one that
    the device cannot serve takes back what another one keeps."""
    csr = _csr(1_000_000, 40, 7)  # 320 MB
    slack = 64 << 20
    with A.Context(0) as a, A.Context(0) as b, A.Context(0) as c:
        a.upload(*csr).close()
        a.trim()
        time.sleep(0.5)
        before = _free_bytes()
        for ctx in (a, b, c):
            ctx.upload(*csr).close()
        assert _settles(lambda: before - _free_bytes() < (512 << 20) + slack)
        assert before - _free_bytes() > (200 << 20)
        p = C.c_void_p()
        assert A.lib().apspie_dev_alloc(c.h, C.c_int64(1 << 50), C.byref(p)) != 0
        assert _settles(lambda: abs(before - _free_bytes()) < slack)
        for ctx in (a, b, c):  # and the contexts go on
            g = ctx.upload(*csr)
            _check(g, csr)
            g.close()
        for ctx in (a, b, c):
            ctx.trim()
        assert _settles(lambda: abs(before - _free_bytes()) < slack)

"""Host arrays to and from the device at the sizes where transfer.hip changes:
one word, a part, a batch of 4 MiB either side of its end, more than the ring
of 32 MiB; arrays that start off a 16-byte boundary; two contexts on two
threads; an index out of range at the far end.  A diagonal matrix comes back as
it was handed over, bit for bit."""
import ctypes
import threading

import numpy as np
import pytest

from elfel_hip import _lib as L

pytestmark = pytest.mark.gpu
I64, F64 = ctypes.POINTER(ctypes.c_int64), ctypes.POINTER(ctypes.c_double)


def _off(a, words):
    """A copy of a that starts `words` words past an allocation's start."""
    b = np.empty(a.size + words, a.dtype)
    b[words:] = a
    return b[words:]


def _round_trip(ctx, n, off, seed):
    rng = np.random.default_rng(seed)
    d = _off(np.arange(1, n + 1, dtype=np.int64), off)
    V = _off(rng.standard_normal(n), off)
    nnz = ctypes.c_int64()
    rc = ctx.lib.elfel_hip_sparse(ctx.h, n, n, n, d.ctypes.data_as(I64), d.ctypes.data_as(I64), V.ctypes.data_as(F64), L.CSC,
                                  ctypes.byref(nnz))
    assert rc == 0 and nnz.value == n
    for base in (0, 1):
        ptr, ind = _off(np.full(n + 1, -9, np.int64), off), _off(np.full(n, -9, np.int64), off)
        val = _off(np.full(n, np.nan), off)
        assert ctx.lib.elfel_hip_copy_sparse(ctx.h, base, ptr.ctypes.data_as(I64), ind.ctypes.data_as(I64),
                                             val.ctypes.data_as(F64)) == 0
        assert np.array_equal(ptr, np.arange(n + 1) + base) and np.array_equal(ind, np.arange(n) + base)
        assert np.array_equal(val, V)
    # one array of the three
    val = np.full(n, np.nan)
    assert ctx.lib.elfel_hip_copy_sparse(ctx.h, 0, None, None, val.ctypes.data_as(F64)) == 0
    assert np.array_equal(val, V)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("n", [1, 2, 7, 16383, 16385, 131071, 524287, 524288, 524289, 1048577, 5000011])
def test_round_trip(ctx, n, off):
    _round_trip(ctx, n, off, n)


def test_index_out_of_range_at_the_end(ctx):
    n = 3000001
    d = np.arange(1, n + 1, dtype=np.int64)
    for bad in (n + 1, 0, 2 ** 40):
        d[-1] = bad
        with pytest.raises(L.ElfelRangeError):
            ctx.sparse(d, np.ones(n, np.int64), np.ones(n), n, 1)
        with pytest.raises(L.ElfelRangeError):
            ctx.vector(d, np.ones(n), n)
    d[-1] = n
    assert np.array_equal(ctx.vector(d, np.arange(n, dtype=np.float64), n), np.arange(n))


def test_two_contexts_on_two_threads():
    failed = []

    def one(k):
        try:
            c = L.Context(0)
            for i in range(4):
                _round_trip(c, 700001 + 300000 * k + i, k, 10 * k + i)
            c.close()
        except BaseException as e:  # noqa: BLE001
            failed.append(e)

    ts = [threading.Thread(target=one, args=(k,)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not failed, failed[0]

"""elfel_hip_sparse_noalloc with its results in the memory of its inputs: the
same pattern and values, bit for bit, as into memory of their own.  4600 entries
are one workgroup's, 300 000 and 900 000 small and large tiles, and a row of
5000 goes to the sort."""
import ctypes

import numpy as np
import pytest

from elfel_hip import _lib as L
from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu


@pytest.fixture
def hip():
    h = Hip()
    yield h
    h.free()


def _stream(n, nrow, long_row, seed):
    rng = np.random.default_rng(seed)
    I, J = rng.integers(1, nrow + 1, n), rng.integers(1, nrow + 1, n)
    I[:long_row] = 3
    I = rng.permutation(I)
    return I, J, rng.standard_normal(n)


@pytest.mark.parametrize("layout", [L.CSR, L.CSC])
@pytest.mark.parametrize("n,nrow,long_row", [(4600, 300, 0), (300000, 20000, 0), (900000, 60000, 0), (300000, 20000, 5000)])
def test_results_in_the_inputs_memory(ctx, hip, n, nrow, long_row, layout):
    I, J, V = _stream(n, nrow, long_row, n)
    nnz = ctx.sparse(I, J, V, nrow, nrow, layout=layout)
    ref = ctx.copy_sparse(base=0)[:3]

    def build(row, col, val, ptr, ind, out):
        assert ctx.sparse_noalloc(nrow, nrow, n, row, col, val, layout, ptr, ind, out) == nnz
        got = hip.get(ptr, nrow + 1, np.int32), hip.get(ind, nnz, np.int32), hip.get(out, nnz, np.float64)
        for a, b in zip(got, ref):
            assert np.array_equal(a, b)

    ptr, ind, out = hip.alloc(4 * (nrow + 1)), hip.alloc(4 * n), hip.alloc(8 * n)
    for _ in range(3):
        row, col, val = hip.put(I), hip.put(J), hip.put(V)
        build(row, col, val, ptr, ind, val)  # the values in place
    row, col, val = hip.put(I), hip.put(J), hip.put(V)
    build(row, col, val, col, row, val)  # all of them
    row, col, val = hip.put(I), hip.put(J), hip.put(V)
    build(row, col, val, ptr, val, out)  # the indices over the values
    row, col, val = hip.put(I), hip.put(J), hip.put(V)
    build(row, col, val, val + 8 * (n - nrow), ind, out)  # the pointers over the last values
    row, col = hip.put(I), hip.put(J)
    shifted = hip.put(np.concatenate([np.zeros(100), V]))
    build(row, col, shifted + 800, ptr, ind, shifted)  # the values 100 words earlier


@pytest.mark.parametrize("n,nrow", [(50, 20), (20000, 3000)])
def test_refused_call_changes_nothing(ctx, hip, n, nrow):
    """An index out of range: the count and the result arrays keep what they hold."""
    I, J, V = _stream(n, nrow, 0, n)
    J[n // 2] = nrow + 1
    ptr, ind, out = hip.put(np.full(nrow + 1, -7, np.int32)), hip.put(np.full(n, -7, np.int32)), hip.put(np.full(n, -7.0))
    nnz = ctypes.c_int64(-7)
    rc = ctx.lib.elfel_hip_sparse_noalloc(ctx.h, nrow, nrow, n, hip.put(I), hip.put(J), hip.put(V), L.CSR, ptr, ind, out,
                                          ctypes.byref(nnz))
    assert rc == L.ERANGE and nnz.value == -7
    assert np.all(hip.get(ptr, nrow + 1, np.int32) == -7) and np.all(hip.get(ind, n, np.int32) == -7)
    assert np.all(hip.get(out, n, np.float64) == -7.0)

"""Small transfers (arrays of a call up to 2 MiB on the device, transfer.hip): uploads
that nothing waits for, one after another through more memory than a context
keeps for them, from host arrays that change right after the call; coefficients
at the edges of the padded blocks (4096) and of what counts as small (131072 of
two coefficients), read back exactly: a matrix and a load of powers of two."""
import ctypes

import numpy as np
import pytest

import elfel_hip as eh
from elfel_hip import _lib as L

pytestmark = pytest.mark.gpu
I64, F64 = ctypes.POINTER(ctypes.c_int64), ctypes.POINTER(ctypes.c_double)


@pytest.mark.parametrize("nx,ny", [(1, 1), (45, 45), (63, 65), (64, 64), (241, 17), (128, 128), (256, 250), (256, 256), (65537, 1),
                                   (300, 300), (512, 256), (43691, 3)])
def test_uploads_without_waits(ctx, nx, ny):
    mesh = eh.Q4block(float(nx), float(ny), nx, ny)
    n, E = mesh.nnodes, mesh.nelements
    conn, xy, dofs = mesh.conn.copy(), mesh.xy.copy(), np.random.default_rng(E).permutation(n).reshape(-1, 1) + 1
    kappa = np.random.default_rng(3).uniform(0.5, 2.0, E)
    Q = np.random.default_rng(4).uniform(-1.0, 1.0, E)
    ctx.set_mesh(0, conn, xy)
    ctx.set_dofs(0, dofs, n)
    conn[:], xy[:], dofs[:] = 0, np.nan, 0
    for method in (L.SORT, L.REUSE):
        ctx.set_coefficients(E, kappa, Q)
        ctx.assemble(L.HEAT, L.Q4, 2, precision=L.FP64, method=method, layout=L.CSR)
        ptr, ind, val = ctx.copy_sparse(base=0)[:3]
        F = ctx.copy_vector(n)
        assert ptr[-1] == val.size and np.isfinite(val).all() and np.abs(val).max() > 0
        for k in range(24):
            a, b = kappa * 2.0 ** (k % 11), Q * 2.0 ** -(k % 7)
            ctx.set_coefficients(E, a, b)
            a[:], b[:] = np.nan, np.nan
            ctx.assemble(L.HEAT, L.Q4, 2, precision=L.FP64, method=method, layout=L.CSR, wait=k % 2 == 0)
            if k % 5 == 4:
                got = ctx.copy_sparse(base=0)[:3]
                assert np.array_equal(got[0], ptr) and np.array_equal(got[1], ind)
                assert np.array_equal(got[2], val * 2.0 ** (k % 11)) and np.array_equal(ctx.copy_vector(n), F * 2.0 ** -(k % 7))


def test_many_small_meshes_in_turn(ctx):
    """Connectivities, nodes and dof maps of changing sizes, each set over the last before it was used."""
    got = []
    for rep in range(2):
        for n in (3, 17, 40, 5, 90, 91, 92, 2):
            mesh = eh.T3block(1.0, 1.0, n, n)
            for order in (np.arange(mesh.nnodes)[::-1], np.arange(mesh.nnodes)):
                ctx.set_mesh(0, mesh.conn, mesh.xy)
                ctx.set_dofs(0, order.reshape(-1, 1) + 1, mesh.nnodes)
            ctx.set_coefficients(mesh.nelements)
            ctx.assemble(L.HEAT, L.T3, 1, precision=L.FP64, method=L.SORT, layout=L.CSC, kappa=1.0, Q=1.0)
            ptr, ind, val = ctx.copy_sparse(base=0)[:3]
            rows = np.zeros(mesh.nnodes)
            np.add.at(rows, ind, val)
            assert np.abs(rows).max() < 1e-12  # a constant has no flux
            assert abs(ctx.copy_vector(mesh.nnodes).sum() - 1.0) < 1e-12  # the load of the unit square
            got.append((ptr, ind, val))
    half = len(got) // 2
    for a, b in zip(got[:half], got[half:]):
        assert all(np.array_equal(x, y) for x, y in zip(a, b))


def test_refused_upload_then_the_next(ctx):
    mesh = eh.T3block(1.0, 1.0, 9, 9)
    conn = mesh.conn.copy()
    for bad in (0, mesh.nnodes + 1, -2 ** 40):
        conn[-1, -1] = bad
        with pytest.raises(L.ElfelRangeError):
            ctx.set_mesh(0, conn, mesh.xy)
        with pytest.raises(L.ElfelRangeError):
            ctx.vector(np.array([1, 2, bad], np.int64), np.ones(3), mesh.nnodes)
    assert np.array_equal(ctx.vector(np.array([3, 1, 3], np.int64), np.array([1.0, 2.0, 4.0]), 3), [2.0, 0.0, 5.0])


@pytest.mark.parametrize("n", [1, 8191, 8192, 8193, 8200, 131071, 131072, 131073, 262144, 262145])
@pytest.mark.parametrize("off", [0, 1])
def test_one_array_out(ctx, n, off):
    """Words as they are, one array of a call: either side of 64 KB, 1 MB and 2 MB, new memory and kept."""
    idx, val = np.arange(1, n + 1, dtype=np.int64), np.random.default_rng(n).standard_normal(n)
    for _ in range(3):
        buf = np.full(n + 2, -7.0)
        out = buf[off:off + n]
        rc = ctx.lib.elfel_hip_vector(ctx.h, n, n, idx.ctypes.data_as(I64), val.ctypes.data_as(F64), out.ctypes.data_as(F64))
        assert rc == L.OK and np.array_equal(out, val) and np.all(buf[off + n:] == -7.0) and np.all(buf[:off] == -7.0)
        val = -2.0 * val

"""elfel_hip_pcg at the sizes where its kernels change: rows either side of a
wave, of a block of 256 rows, of what one workgroup solves (1024 rows for each
of a work-item's; 2048 FP64 and 4096 mixed at most, grids in their own order),
of a workgroup of the one-launch solve (512 rows FP64, 768 mixed), of the most
rows that it takes (224 workgroups), of each count of rows a work-item of the
solve from registers (262144 rows each on 256 CUs; 1 to 3 FP64, 1 to 8 mixed)
and past its last, grids with their boundary
numbered last and ones whose slices it does not take, a matrix whose rows are
wider than the registers, and one whose columns are too far from the diagonal
for 16-bit offsets.

The solve stops on its own FP64 residual, ||b - A x|| <= tol ||b||.  The same
residual formed here differs by the rounding of its sums, at most about
(entries of a row + 2) 2^-53 times |A| |x| / ||b||, which is below 2^-52 * 64 *
4 nfree for these matrices (|x| <= nfree ||b|| / 4 and |A| <= 16 in units of the
diagonal): the bound is tol plus that.
"""
import numpy as np
import pytest
import scipy.sparse as sp

import elfel_hip as eh
from elfel_hip import _lib as L

pytestmark = pytest.mark.gpu
TOL = 1e-8


def _solve(ctx, fe, N, nfree, prec, seed=3, shuffle=False, kind=L.HEAT, order=None):
    block = {L.Q4: eh.Q4block, L.T3: eh.T3block, L.T6: eh.T6block}[fe]
    mesh = block(1.0, 1.0, N, N)
    nc = 2 if kind == L.ELAST else 1
    n = mesh.nnodes * nc
    rng = np.random.default_rng(seed)
    dn = (rng.permutation(n) if shuffle else np.arange(n) if order is None else order) + 1
    ctx.set_mesh(0, mesh.conn, mesh.xy)
    ctx.set_dofs(0, dn.reshape(-1, nc), n)
    ctx.set_coefficients(mesh.nelements)
    rule = 2 if fe == L.Q4 else 3 if fe == L.T6 else 1
    ctx.assemble(kind, fe, rule, precision=L.FP64, method=L.REUSE, layout=L.CSR, D=eh.plane_strain_D(1.0, 0.3))
    ptr, ind, val = ctx.copy_sparse(base=0)[:3]
    K = sp.csr_matrix((val, ind, ptr), shape=(n, n))
    F = rng.standard_normal(n)
    x0 = rng.standard_normal(n)
    x, it, _, rel = ctx.pcg(nfree, F, x0, precision=prec, tol=TOL, maxit=200000)
    assert np.array_equal(x[nfree:], x0[nfree:]) and rel <= TOL
    b = F[:nfree] - K[:nfree, nfree:] @ x0[nfree:]
    r = b - K[:nfree, :nfree] @ x[:nfree]
    assert np.linalg.norm(r) <= (TOL + 2.0 ** -52 * 256 * nfree) * np.linalg.norm(b), (nfree, it)
    again = ctx.pcg(nfree, F, x0, precision=prec, tol=TOL, maxit=200000)
    assert np.array_equal(again[0], x) and again[1] == it  # every run gives the same bits


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("nfree", [1, 2, 63, 64, 65, 255, 256, 257, 511, 512, 513, 767, 768, 769, 1535, 1536, 1537, 1600])
def test_small(ctx, nfree, prec):
    _solve(ctx, L.Q4, 40, nfree, prec)
    _solve(ctx, L.Q4, 40, nfree, prec, shuffle=True)


@pytest.mark.parametrize("fe", [L.T3, L.Q4])
@pytest.mark.parametrize("prec,nfree", [(L.FP64, 1023), (L.FP64, 1024), (L.FP64, 1025), (L.FP64, 2047), (L.FP64, 2048),
                                        (L.FP64, 2049), (L.MIXED, 2049), (L.MIXED, 3072), (L.MIXED, 4095), (L.MIXED, 4096),
                                        (L.MIXED, 4097)])
def test_one_workgroup(ctx, nfree, prec, fe):
    _solve(ctx, fe, 66, nfree, prec)


@pytest.mark.parametrize("prec,nfree,N", [(L.FP64, 224 * 512, 340), (L.FP64, 224 * 512 + 1, 340),
                                          (L.MIXED, 224 * 768, 416), (L.MIXED, 224 * 768 + 1, 416)])
def test_most_rows_of_one_launch(ctx, prec, nfree, N):
    _solve(ctx, L.Q4, N, nfree, prec)


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
def test_wide_rows_and_far_columns(ctx, prec):
    _solve(ctx, L.T6, 12, 1100, prec, kind=L.ELAST)  # rows of up to 38 entries
    _solve(ctx, L.T3, 200, 39000, prec, shuffle=True)
    _solve(ctx, L.T3, 30, 900, prec, shuffle=True)


@pytest.mark.parametrize("prec,fe,nfree,N", [
    (L.FP64, L.Q4, 262144, 520), (L.FP64, L.T3, 262145, 520), (L.FP64, L.T3, 524288, 730), (L.FP64, L.Q4, 524289, 730),
    (L.FP64, L.Q4, 786432, 890), (L.FP64, L.T3, 786433, 890),
    (L.MIXED, L.T3, 262144, 520), (L.MIXED, L.Q4, 262145, 520), (L.MIXED, L.Q4, 524289, 730),
    (L.MIXED, L.Q4, 786433, 890), (L.MIXED, L.T3, 1048577, 1030), (L.MIXED, L.Q4, 1310721, 1150), (L.MIXED, L.Q4, 1572865, 1260),
    (L.MIXED, L.T3, 1835009, 1360), (L.MIXED, L.Q4, 2097152, 1449), (L.MIXED, L.T3, 2097153, 1449)])
def test_rows_in_registers(ctx, prec, fe, nfree, N):
    _solve(ctx, fe, N, nfree, prec)


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("fe", [L.T3, L.Q4])
@pytest.mark.parametrize("held", ["boundary", "scattered", "swapped"])
def test_held_nodes_and_numberings(ctx, held, fe, prec):
    N = 560  # 561 x 561 nodes; the free ones first, in the mesh's order
    fixed = np.zeros((N + 1, N + 1), bool)
    fixed[[0, -1]] = fixed[:, [0, -1]] = True
    if held == "scattered":
        fixed |= np.random.default_rng(5).random(fixed.shape) < 0.01
    fixed = fixed.ravel()
    free = int((~fixed).sum())
    order = np.where(fixed, free + np.cumsum(fixed) - 1, np.cumsum(~fixed) - 1)
    if held == "swapped":  # free neighbours by twos: offsets of no three runs
        order = np.where(order < free // 2 * 2, order ^ 1, order)
    _solve(ctx, fe, N, free, prec, order=order)

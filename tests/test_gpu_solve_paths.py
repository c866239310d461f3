"""elfel_hip_pcg gives the same iterations and the same bits whether a solve runs
in one launch or in two launches an iteration (ELFEL_HIP_PCG_ONE_LAUNCH=0), and
its solution has the residual that it claims, formed here in float64: tol plus
the rounding of the sums, 2^-52 * 256 * nfree (test_gpu_solve_sizes.py)."""
import numpy as np
import pytest
import scipy.sparse as sp

import elfel_hip as eh
from elfel_hip import _lib as L

pytestmark = pytest.mark.gpu
TOL = 1e-10


def _both(ctx, monkeypatch, nfree, prec, seed=3, tol=TOL, ends=True):
    """Solves the context's CSR matrix for a random right-hand side both ways.
    ends: the iteration reaches the tolerance."""
    ptr, ind, val = ctx.copy_sparse(base=0)[:3]
    n = ptr.size - 1
    K = sp.csr_matrix((val, ind, ptr), shape=(n, n))
    rng = np.random.default_rng(seed)
    F, x0 = rng.standard_normal(n), rng.standard_normal(n)
    monkeypatch.setenv("ELFEL_HIP_PCG_ONE_LAUNCH", "0")
    x2, it2, _, rel2 = ctx.pcg(nfree, F, x0, precision=prec, tol=tol, maxit=100000)
    monkeypatch.delenv("ELFEL_HIP_PCG_ONE_LAUNCH")
    x, it, _, rel = ctx.pcg(nfree, F, x0, precision=prec, tol=tol, maxit=100000)
    assert it == it2 and np.array_equal(x, x2, equal_nan=True) and np.array_equal(rel, rel2, equal_nan=True), (it, it2, rel, rel2)
    if not ends:
        return
    assert rel <= tol
    b = F[:nfree] - K[:nfree, nfree:] @ x0[nfree:]
    r = b - K[:nfree, :nfree] @ x[:nfree]
    assert np.linalg.norm(r) <= (tol + 2.0 ** -52 * 256 * nfree) * np.linalg.norm(b)


def _heat(ctx, fe, nx, ny, fixed):
    """Heat on nx x ny cells, the fixed nodes' dofs last; the free dofs' number."""
    mesh = {L.T3: eh.T3block, L.Q4: eh.Q4block}[fe](float(nx), float(ny), nx, ny)
    x, y = np.rint(mesh.xy).astype(int).T
    fixed = fixed(x, y)
    free = int((~fixed).sum())
    order = np.where(fixed, free + np.cumsum(fixed) - 1, np.cumsum(~fixed) - 1)
    ctx.set_mesh(0, mesh.conn, mesh.xy)
    ctx.set_dofs(0, order.reshape(-1, 1) + 1, mesh.nnodes)
    ctx.set_coefficients(mesh.nelements)
    ctx.assemble(L.HEAT, fe, 2 if fe == L.Q4 else 1, precision=L.FP64, method=L.REUSE, layout=L.CSR)
    return free


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("fe,across", [(L.T3, 1), (L.T3, 2), (L.T3, 3), (L.T3, 4), (L.Q4, 2), (L.Q4, 3), (L.Q4, 4)])
@pytest.mark.parametrize("along", [2, 60, 1000, 30000, 100000])
def test_strips_with_held_sides(ctx, monkeypatch, along, fe, across, prec):
    """`across` free nodes between two held sides, numbered first along the short
    side.  (Quadrilaterals with one free node across have few distinct
    eigenvalues: the mixed iteration, by either way, runs past its end there.)"""
    nx, ny = across + 1, along + 1
    free = _heat(ctx, fe, nx, ny, lambda x, y: (x == 0) | (x == nx) | (y == 0) | (y == ny))
    assert free == across * along
    _both(ctx, monkeypatch, free, prec)


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("fe", [L.T3, L.Q4])
@pytest.mark.parametrize("cells", [1, 2, 3])
def test_strips_with_free_sides(ctx, monkeypatch, cells, fe, prec):
    free = _heat(ctx, fe, cells, 61, lambda x, y: (y == 0) | (y == 61))
    assert free == 60 * (cells + 1)
    _both(ctx, monkeypatch, free, prec)


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("n", [5, 300, 2500, 120000, 180000])
@pytest.mark.parametrize("offsets", [(1,), (2,), (1, 2), (1, 3), (1, 2, 3), (2, 3, 4), (1, 2, 3, 4)])
def test_bands(ctx, monkeypatch, offsets, n, prec):
    """Diagonally dominant bands of a COO stream: the diagonal 2.5 times the sum of its row."""
    rng = np.random.default_rng(n)
    i = np.arange(1, n + 1)
    I, J, V, diag = [], [], [], np.full(n, 0.5)
    for d in offsets:
        v = rng.uniform(0.5, 1.0, max(n - d, 0))
        I += [i[:-d], i[d:]]
        J += [i[d:], i[:-d]]
        V += [-v, -v]
        diag[: n - d] += 2.5 * v
        diag[d:] += 2.5 * v
    ctx.sparse(np.concatenate(I + [i]), np.concatenate(J + [i]), np.concatenate(V + [diag]), n, n, layout=L.CSR)
    _both(ctx, monkeypatch, n, prec)


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("N,shuffle", [(20, False), (70, False), (40, True), (200, False), (200, True)])
@pytest.mark.parametrize("where", ["last", "between", "both"])
def test_free_dofs_of_no_element(ctx, monkeypatch, where, N, shuffle, prec):
    """Free dofs that no element has, whole slices of 64 rows of them: their rows
    have no entries and their load is zero, so they keep their values.  N = 200
    shuffled has columns beyond 16-bit offsets."""
    mesh = eh.Q4block(1.0, 1.0, N, N)
    n, held = mesh.nnodes, mesh.nnodes // 10
    rng = np.random.default_rng(N)
    dof = rng.permutation(n) if shuffle else np.arange(n)
    half = (n - held) // 2
    between, last = {"last": (0, 333), "between": (200, 0), "both": (200, 333)}[where]
    dof = dof + np.where(dof >= half, between, 0) + np.where(dof >= n - held, last, 0)
    total, free = n + between + last, n - held + between + last
    ctx.set_mesh(0, mesh.conn, mesh.xy)
    ctx.set_dofs(0, dof.reshape(-1, 1) + 1, total)
    ctx.set_coefficients(mesh.nelements)
    ctx.assemble(L.HEAT, L.Q4, 2, precision=L.FP64, method=L.SORT, layout=L.CSR)
    ptr, ind, val = ctx.copy_sparse(base=0)[:3]
    K = sp.csr_matrix((val, ind, ptr), shape=(total, total))
    none = np.diff(ptr) == 0
    assert none.sum() == between + last
    F, x0 = rng.standard_normal(total), rng.standard_normal(total)
    F[none] = 0.0
    monkeypatch.setenv("ELFEL_HIP_PCG_ONE_LAUNCH", "0")
    x2, it2, _, rel2 = ctx.pcg(free, F, x0, precision=prec, tol=TOL, maxit=20000)
    monkeypatch.setenv("ELFEL_HIP_SELL_UNIFORM", "0")
    x3, it3, _, rel3 = ctx.pcg(free, F, x0, precision=prec, tol=TOL, maxit=20000)
    monkeypatch.delenv("ELFEL_HIP_PCG_ONE_LAUNCH")
    monkeypatch.delenv("ELFEL_HIP_SELL_UNIFORM")
    x, it, _, rel = ctx.pcg(free, F, x0, precision=prec, tol=TOL, maxit=20000)
    assert it == it2 == it3 and rel == rel2 == rel3 <= TOL
    assert np.array_equal(x, x2) and np.array_equal(x, x3)
    assert np.array_equal(x[none], x0[none])
    b = F[:free] - K[:free, free:] @ x0[free:]
    assert np.linalg.norm(b - K[:free, :free] @ x[:free]) <= (TOL + 2.0 ** -52 * 256 * free) * np.linalg.norm(b)


@pytest.mark.parametrize("fe", [L.T3, L.Q4])
@pytest.mark.parametrize("N,prec,sizes", [
    (70, L.FP64, (1, 64, 65, 255, 257, 1023, 1024, 1025, 2047, 2048, 2049, 3071)),
    (70, L.MIXED, (1, 64, 65, 255, 257, 1023, 1024, 1025, 2048, 2049, 3072, 4095, 4096, 4097, 4609)),
    (340, L.FP64, (224 * 512, 224 * 512 + 1)), (416, L.MIXED, (224 * 768, 224 * 768 + 1)),
    (730, L.FP64, (262144, 262145, 524288, 524289)), (890, L.FP64, (786432, 786433)),
    (730, L.MIXED, (262144, 262145, 524289)), (1030, L.MIXED, (786433, 1048577)), (1449, L.MIXED, (1572865, 2097152, 2097153))])
def test_both_ways_where_the_kernels_change(ctx, monkeypatch, N, prec, sizes, fe):
    """Rows either side of what each one-launch kernel and each number of rows a
    work-item takes (test_gpu_solve_sizes.py), grids in their own order."""
    n = (N + 1) ** 2
    for nfree in sizes:
        free = _heat(ctx, fe, N, N, lambda x, y: x + (N + 1) * y >= nfree)
        assert free == nfree < n
        # (one grid row of quadrilaterals: the strips of one free node across, above)
        _both(ctx, monkeypatch, nfree, prec, tol=1e-8, ends=prec == L.FP64 or fe == L.T3 or nfree > N + 1)


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("fe,N,shuffle", [(L.T3, 40, False), (L.Q4, 300, False), (L.T3, 300, True), (L.Q4, 700, False), (L.T6, 60, False),
                                          (L.T6, 60, True)])
def test_direction_in_the_product_or_before_it(ctx, monkeypatch, fe, N, shuffle, prec):
    """Two and three kernels an iteration (ELFEL_HIP_PCG_FUSED), heat and, on T6,
    elasticity, whose rows are wider than the registers; in a random order the
    columns lie beyond 16-bit offsets."""
    mesh = {L.T3: eh.T3block, L.Q4: eh.Q4block, L.T6: eh.T6block}[fe](1.0, 1.0, N, N)
    nc = 2 if fe == L.T6 else 1
    n = mesh.nnodes * nc
    nfree = n - 3 * N * nc
    dof = np.random.default_rng(N).permutation(n) if shuffle else np.arange(n)
    ctx.set_mesh(0, mesh.conn, mesh.xy)
    ctx.set_dofs(0, dof.reshape(-1, nc) + 1, n)
    ctx.set_coefficients(mesh.nelements)
    ctx.assemble(L.ELAST if nc == 2 else L.HEAT, fe, {L.T3: 1, L.Q4: 2, L.T6: 3}[fe], precision=L.FP64, method=L.REUSE,
                 layout=L.CSR, D=eh.plane_strain_D(1.0, 0.3))
    rng = np.random.default_rng(7)
    F, x0 = rng.standard_normal(n), rng.standard_normal(n)
    monkeypatch.setenv("ELFEL_HIP_PCG_ONE_LAUNCH", "0")
    got = []
    for fused in ("0", "1", None):
        if fused is None:
            monkeypatch.delenv("ELFEL_HIP_PCG_FUSED")
        else:
            monkeypatch.setenv("ELFEL_HIP_PCG_FUSED", fused)
        got.append(ctx.pcg(nfree, F, x0, precision=prec, tol=1e-8, maxit=20000))
    for x, it, _, rel in got:
        assert rel <= 1e-8 and it == got[0][1] and np.array_equal(x, got[0][0])

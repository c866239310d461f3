"""One-launch solves whose waits give up (ELFEL_HIP_PCG_POLLS: a wait of few
polls; every workgroup then leaves its loop and the kernel ends): the solve goes
on from the x that they left, in two launches an iteration, to the residual that
it claims, formed here in float64: tol plus the rounding of the sums, 2^-52 *
256 * nfree (test_gpu_solve_sizes.py).  A solve without the limit afterwards has
the bits of one before."""
import numpy as np
import pytest
import scipy.sparse as sp

import elfel_hip as eh
from elfel_hip import _lib as L

pytestmark = pytest.mark.gpu
TOL = 1e-9


@pytest.mark.parametrize("prec", [L.FP64, L.MIXED])
@pytest.mark.parametrize("fe,N", [(L.Q4, 80), (L.T3, 200), (L.Q4, 440)])
def test_waits_that_give_up(ctx, monkeypatch, fe, N, prec):
    """80 and 200 cells across: the small solve; 440: the one from registers."""
    mesh = {L.T3: eh.T3block, L.Q4: eh.Q4block}[fe](1.0, 1.0, N, N)
    n = mesh.nnodes
    nfree = n - 2 * (N + 1)
    ctx.set_mesh(0, mesh.conn, mesh.xy)
    ctx.set_dofs(0, np.arange(1, n + 1).reshape(-1, 1), n)
    ctx.set_coefficients(mesh.nelements)
    ctx.assemble(L.HEAT, fe, 2 if fe == L.Q4 else 1, precision=L.FP64, method=L.REUSE, layout=L.CSR)
    ptr, ind, val = ctx.copy_sparse(base=0)[:3]
    K = sp.csr_matrix((val, ind, ptr), shape=(n, n))
    rng = np.random.default_rng(N)
    F, x0 = rng.standard_normal(n), rng.standard_normal(n)
    b = F[:nfree] - K[:nfree, nfree:] @ x0[nfree:]
    before = ctx.pcg(nfree, F, x0, precision=prec, tol=TOL, maxit=50000)
    for polls in (1, 2, 3, 5, 8, 20):
        monkeypatch.setenv("ELFEL_HIP_PCG_POLLS", str(polls))
        x, it, _, rel = ctx.pcg(nfree, F, x0, precision=prec, tol=TOL, maxit=50000)
        assert rel <= TOL, (polls, it, rel)
        r = b - K[:nfree, :nfree] @ x[:nfree]
        assert np.linalg.norm(r) <= (TOL + 2.0 ** -52 * 256 * nfree) * np.linalg.norm(b), polls
        assert np.array_equal(x[nfree:], x0[nfree:])
        if polls == 1:  # no first wait is through in one poll
            assert it != before[1] or not np.array_equal(x, before[0])
    monkeypatch.delenv("ELFEL_HIP_PCG_POLLS")
    after = ctx.pcg(nfree, F, x0, precision=prec, tol=TOL, maxit=50000)
    assert np.array_equal(after[0], before[0]) and after[1:] == before[1:]

"""The row-bucket COO build (elfel_hip_sparse, elfel_hip_sparse_noalloc) at the
edges of its tiles, against the oracle's sparse(): pattern and values bit for
bit (tolerance 0, the same sums in the same order).  Up to 6144 entries and 8191
rows are one workgroup's; 1536 entries start in a tile, 3584 of a stream of more
than 393216, with rows of up to 512; with one of up to 1024, or 2048, as many;
longer ones and matrices of far more rows than entries take the sort."""
import numpy as np
import pytest

import elfel_hip as eh
import oracle as O
from elfel_hip import _lib as L
from test_gpu_general_meshes import _oracle_heat, _same, fan_mesh
from test_zz_no_alloc import Hip, _noalloc

pytestmark = pytest.mark.gpu


@pytest.fixture
def hip():
    h = Hip()
    yield h
    h.free()


def _rows(lengths, ncol, rng):
    """A stream with the given entries per row, rows interleaved, columns repeating."""
    I = rng.permutation(np.repeat(np.arange(1, len(lengths) + 1), lengths))
    return I, rng.integers(1, ncol + 1, I.size)


def _case(name, rng):
    if name.startswith("n="):
        n = int(name[2:])
        return (*_rows(rng.multinomial(n, np.full(40, 1 / 40)), 23, rng), 40, 23)
    if name.startswith("many="):
        n = int(name[5:])
        return (*_rows(rng.multinomial(n, np.full(9000, 1 / 9000)), 60, rng), 9000, 60)
    if name.startswith("rows="):
        n = int(name[5:])
        return (*_rows(rng.multinomial(6000, np.full(n, 1 / n)), 31, rng), n, 31)
    if name.startswith("tiled row="):
        k = int(name[10:])
        return (*_rows([3] * 2500 + [k] + [0] * 7 + [5] * 300, max(k // 2, 1), rng), 2808, max(k // 2, 1))
    if name.startswith("large row="):
        k = int(name[10:])
        return (*_rows([40] * 5000 + [k] + [0] * 7 + [41] * 5000, max(k // 2, 1), rng), 10008, max(k // 2, 1))
    if name.startswith("row="):  # one long row between short ones, and a tile that it straddles
        k = int(name[4:])
        return (*_rows([3] * 500 + [k] + [0] * 7 + [5] * 300, max(k // 2, 1), rng), 808, max(k // 2, 1))
    if name == "long rows side by side":  # every tile at its largest
        return (*_rows([511, 1024, 1, 512, 512, 512, 512, 511, 1][2:], 600, rng), 7, 600)
    if name == "long rows in tiles":
        return (*_rows([512, 512, 512, 511, 1] * 4 + [512] + [1] * 40, 600, rng), 61, 600)
    if name == "longest rows":
        return (*_rows([1024, 1023, 1] * 3 + [1024] * 4 + [1] * 40, 900, rng), 53, 900)
    if name == "longest rows, many":
        return (*_rows([2048, 2047, 1] * 30 + [2048] * 150 + [1] * 2000, 1500, rng), 2240, 1500)
    if name == "long rows, many":
        return (*_rows([512] * 5 + [511, 1] + [512] * 830 + [3] * 1020, 700, rng), 1857, 700)
    if name == "empty ends":
        return (*_rows([0] * 9000 + [2] * 50 + [0] * 9000, 60, rng), 18050, 60)
    if name == "one entry":
        return np.array([7]), np.array([3]), 9, 4
    if name == "one row":
        return (*_rows([400], 1, rng), 1, 1)
    if name == "two rows, all duplicates":
        return (*_rows([300, 300], 1, rng), 2, 1)
    if name == "more rows than entries":
        return (*_rows([1] * 30 + [0] * 69970, 30, rng), 70000, 30)
    if name == "last columns":  # indices next to the limit of int32
        n = 3000
        return rng.integers(1, 50, n), 2 ** 31 - 2 - rng.integers(0, 40, n), 50, 2 ** 31 - 2
    raise ValueError(name)


CASES = ["many=393216", "many=393217", "many=401408", "long rows, many", "n=1535", "n=1536", "n=1537", "n=2048", "n=3072", "n=6143", "n=6144", "n=6145", "n=7679",
         "n=7680", "n=7681", "n=9001", "rows=8190", "rows=8191", "rows=8192", "tiled row=511", "tiled row=512",
         "tiled row=513", "tiled row=1023", "tiled row=1024", "tiled row=1025", "large row=513", "large row=2047", "large row=2048",
         "large row=2049", "longest rows", "longest rows, many", "long rows in tiles", "row=511", "row=512", "row=513", "row=1600",
         "long rows side by side", "empty ends", "one entry", "one row", "two rows, all duplicates",
         "more rows than entries", "last columns"]


@pytest.mark.parametrize("csc", [False, True])
@pytest.mark.parametrize("name", CASES)
def test_bucket_build_equals_oracle(name, csc, ctx, hip):
    rng = np.random.default_rng(5)
    I, J, nrow, ncol = _case(name, rng)
    I, J = I.astype(np.int64), J.astype(np.int64)
    if csc:  # the cases describe the major rows
        I, J, nrow, ncol = J, I, ncol, nrow
    V = rng.standard_normal(I.size)
    V[::7] = -0.0
    V[3::31] = np.inf
    if csc is False and nrow >= 2 ** 31 - 2:
        pytest.skip("the oracle's pointers over 2^31 rows")
    ref = O.sparse(I, J, V, nrow, ncol, csc=csc)
    lay = L.CSC if csc else L.CSR
    for _ in range(2):
        nnz = ctx.sparse(I, J, V, nrow, ncol, layout=lay)
        got = ctx.copy_sparse(base=0)[:3]
        assert nnz == ref[0][-1]
        for a, b in zip(got, ref):
            assert np.array_equal(a, b, equal_nan=True) and np.array_equal(np.signbit(a), np.signbit(b)), name
        got = _noalloc(ctx, hip, I, J, V, nrow, ncol, lay)
        for a, b in zip(got[1:], ref):
            assert np.array_equal(a, b, equal_nan=True), name


def test_bucket_build_refuses_then_works(ctx):
    rng = np.random.default_rng(6)
    I, J = rng.integers(1, 31, 5000), rng.integers(1, 31, 5000)
    V = rng.standard_normal(5000)
    for bad in (0, 31, -5, 2 ** 40):
        K = J.copy()
        K[4321] = bad
        with pytest.raises(L.ElfelRangeError):
            ctx.sparse(I, K, V, 30, 30, layout=L.CSR)
    ctx.sparse(I, J, V, 30, 30, layout=L.CSR)
    ref = O.sparse(I, J, V, 30, 30, csc=False)
    for a, b in zip(ctx.copy_sparse(base=0)[:3], ref):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("method", [L.SORT, L.REUSE])
@pytest.mark.parametrize("layout", [L.CSR, L.CSC])
def test_element_stream_at_the_longest_row(ctx, method, layout):
    """A T3 fan's centre row has 3 K entries: 170 and 171 elements lie either
    side of 512 entries, 341 and 342 of the 1024 of a small tile.  One context, so that the answer for one
    mesh must not outlive it, with and without a wait, and a dof that two nodes
    (hence an element's two local dofs) share."""
    for K, tie in ((170, False), (171, False), (40, True), (170, False), (171, True), (30, False), (341, False), (342, True), (341, True),
                   (342, False), (30, True)):
        conn, xy = fan_mesh(K, rings=2)
        dn = np.random.default_rng(K).permutation(xy.shape[0]) + 1
        if tie:
            dn[2] = dn[1]  # neighbours on the first ring: one dof twice in an element
        n = xy.shape[0]
        ref = _oracle_heat(conn, xy, dn, n, layout)
        ctx.set_mesh(0, conn, xy)
        ctx.set_dofs(0, dn, n)
        ctx.set_coefficients(conn.shape[0])
        for wait in (True, False, False):
            ctx.assemble(L.HEAT, L.T3, 1, method=method, layout=layout, kappa=1.3, Q=-2.0, wait=wait)
            _same(ctx.copy_sparse(base=0), ref)
            assert np.array_equal(ctx.copy_vector(n), ref[3])


@pytest.mark.parametrize("layout", [L.CSR, L.CSC])
def test_element_stream_in_large_tiles(ctx, layout):
    """460 800 entries: with a dof that two nodes of an element share, and one
    that no element has (its load is zero)."""
    mesh = eh.T3block(2.0, 1.0, 160, 160)
    conn, xy = np.asarray(mesh.conn), np.asarray(mesh.xy)
    n = xy.shape[0] + 1
    dn = np.random.default_rng(8).permutation(n)[:-1] + 1
    dn[2] = dn[1]
    ref = _oracle_heat(conn, xy, dn, n, layout)
    ctx.set_mesh(0, conn, xy)
    ctx.set_dofs(0, dn, n)
    ctx.set_coefficients(conn.shape[0])
    for method in (L.SORT, L.REUSE):
        ctx.assemble(L.HEAT, L.T3, 1, method=method, layout=layout, kappa=1.3, Q=-2.0)
        _same(ctx.copy_sparse(base=0), ref)
        assert np.array_equal(ctx.copy_vector(n), ref[3])


@pytest.mark.parametrize("method", [L.SORT, L.REUSE])
@pytest.mark.parametrize("ne", [2, 682, 683])
def test_element_stream_of_one_workgroup(ctx, ne, method):
    """6138 and 6147 entries lie either side of what one workgroup takes."""
    mesh = eh.T3block(2.0, 1.0, 20, 20)
    conn, xy = np.asarray(mesh.conn)[:ne], np.asarray(mesh.xy)
    n = xy.shape[0] + 1
    dn = np.random.default_rng(ne).permutation(n)[:-1] + 1
    dn[conn[0][1]] = dn[conn[0][0]]  # one dof twice in an element
    for layout in (L.CSR, L.CSC):
        ref = _oracle_heat(conn, xy, dn, n, layout)
        ctx.set_mesh(0, conn, xy)
        ctx.set_dofs(0, dn, n)
        ctx.set_coefficients(conn.shape[0])
        ctx.assemble(L.HEAT, L.T3, 1, method=method, layout=layout, kappa=1.3, Q=-2.0)
        _same(ctx.copy_sparse(base=0), ref)
        assert np.array_equal(ctx.copy_vector(n), ref[3])

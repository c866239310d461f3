"""Transfers where no host memory can be pinned (ELFEL_HIP_PINNED=0 in a process
of its own): the same arrays come back, small ones, a batch of 4 MiB either side
of its end and more than the ring; an index out of range is still refused."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CODE = """
import numpy as np
import elfel_hip as eh
from elfel_hip import _lib as L
ctx = L.Context(0)
for n in (1, 700, 130000, 524289, 1048577, 5000011):
    d, V = np.arange(1, n + 1, dtype=np.int64), np.random.default_rng(n).standard_normal(n)
    assert ctx.sparse(d, d, V, n, n) == n
    ptr, ind, val = ctx.copy_sparse(base=1)[:3]
    assert np.array_equal(ptr, np.arange(1, n + 2)) and np.array_equal(ind, d) and np.array_equal(val, V)
    d[-1] = n + 1
    try:
        ctx.vector(d, V, n)
        raise SystemExit("an index out of range was taken")
    except L.ElfelRangeError:
        pass
mesh = eh.Q4block(1.0, 1.0, 300, 300)
ctx.set_mesh(0, mesh.conn, mesh.xy)
ctx.set_dofs(0, np.arange(1, mesh.nnodes + 1).reshape(-1, 1), mesh.nnodes)
k = np.random.default_rng(1).uniform(0.5, 2.0, mesh.nelements)
got = []
for f in (1.0, 4.0):
    ctx.set_coefficients(mesh.nelements, k * f, k)
    ctx.assemble(L.HEAT, L.Q4, 2, precision=L.FP64, method=L.REUSE, layout=L.CSR)
    got.append((ctx.copy_sparse(base=0)[2], ctx.copy_vector(mesh.nnodes)))
assert np.array_equal(got[0][0] * 4.0, got[1][0]) and np.array_equal(got[0][1], got[1][1]) and np.abs(got[0][0]).max() > 0
ctx.close()
print("OK", flush=True)
"""


@pytest.mark.gpu
def test_transfers_through_ordinary_memory():
    env = dict(os.environ, ELFEL_HIP_PINNED="0", PYTHONPATH=os.path.join(ROOT, "elfel.jl_amd"))
    r = subprocess.run([sys.executable, "-c", CODE], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.strip() == "OK", r.stdout + r.stderr

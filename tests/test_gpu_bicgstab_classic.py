"""Jacobi-BiCGStab with the reference's recurrences: alpha and omega inside the vector kernels (six
kernels per iteration) up to a bound on the partial sums read, scalar kernels of their own beyond it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [("powerlaw", 300, 6), ("powerlaw", 20001, 6), ("powerlaw", 300000, 6),
                                  ("convdiff", 61, 6), ("convdiff", 100, 8)])
def test_both_forms_solve(dev, vh, oracle, case):
    """Either form solves to its tolerance, and chunks of one iteration and graph chunks give the same x
    bit for bit."""
    kind, m, kernels = case
    rp, col, val = vh.powerlaw(m, min(512, m // 2), 2.0, 1.1, 5) if kind == "powerlaw" else vh.convection_diffusion(m, m, m)
    n = rp.size - 1
    A, b = vh.CsrMatrix(rp, col, val), vh.random_uniform(3, n)
    xs = []
    for kw in ({}, {"chunk": 1}, {"use_graph": True, "chunk": 8}):
        db, dx = vh.DeviceArray.from_numpy(b), vh.DeviceArray.zeros(n, np.float64)
        res = vh.bicgstab(A, db, dx, precond=1, tol=1e-10, max_iters=2000, **kw)
        assert res.converged and res.kernels_per_iter == kernels
        xs.append(dx.to_numpy())
    assert np.array_equal(xs[0], xs[1]) and np.array_equal(xs[0], xs[2])
    # the stop is on ||D^-1 r||, so ||r|| may be larger by the spread of the diagonal
    rows = np.repeat(np.arange(n), np.diff(rp.astype(np.int64)))
    d = np.abs(val[col.astype(np.int64) == rows])
    r = b - oracle.csr_spmv(rp, col, val, xs[0])
    assert np.linalg.norm(r) / np.linalg.norm(b) < 10 * 1e-10 * d.max() / d.min()

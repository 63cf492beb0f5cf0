"""GMRES(m) through every register width of the Gram-Schmidt kernels (m = 4,
8, 16, 24, 32), the basis lengths between them, and the separate kernels that
longer bases take, at vector lengths around a wavefront, a workgroup and the
grid's first stride.

Well-conditioned nonsymmetric systems (I plus a random sparse matrix of norm
below 1/2, condition below 3): the solver stops at a relative residual of
1e-11, so the solution is within 3e-11 of the dense solve, and a full-length
basis has to finish in one cycle."""
import numpy as np
import pytest
import torch

import cfdrs_amd as ca
from cfdrs_amd.linear_solver import gmres_exact_restart

pytestmark = pytest.mark.gpu


def system(n, seed):
    rng = np.random.default_rng(seed)
    rows, cols, vals = [], [], []
    for i in range(n):
        c = np.unique(rng.integers(0, n, 4))
        v = rng.uniform(-1.0, 1.0, c.size)
        v *= 0.45 / np.abs(v).sum()
        d = dict(zip(c.tolist(), v.tolist()))
        d[i] = d.get(i, 0.0) + 1.0
        for j in sorted(d):
            rows.append(i)
            cols.append(j)
            vals.append(d[j])
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))])
    return np.array(rows), np.array(cols), np.array(vals), rp, rng.uniform(-1.0, 1.0, n)


@pytest.mark.parametrize("m", [1, 3, 4, 5, 8, 9, 16, 17, 24, 25, 32, 33, 40, 65])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 1025])
def test_restart_widths(n, m):
    rows, cols, vals, rp, b = system(n, 100 * n + m)
    a = ca.CsrMatrix.from_parts(vals, cols, rp, n, n)
    x = np.zeros(n)
    rep = gmres_exact_restart(a, b, None, x, ca.IterativeSolverConfig.new(1e-11).with_max_iterations(2000), m)
    assert rep.termination == ca.Termination.Converged
    ax = np.bincount(rows, weights=vals * x[cols], minlength=n)
    assert np.linalg.norm(b - ax) <= 1.1e-11 * np.linalg.norm(b)
    dense = np.zeros((n, n))
    dense[rows, cols] = vals
    want = np.linalg.solve(dense, b)
    # row sums of the perturbation are 0.45; its column sums, and with them the
    # condition, are bounded by the matrix itself
    cond = np.linalg.cond(dense)
    assert np.linalg.norm(x - want) <= 1.2e-11 * cond * np.linalg.norm(want)


@pytest.mark.parametrize("n", [131071, 131073, 300001])
def test_long_vectors(n):
    # tridiagonal, diagonally dominant: past one element per lane of the grid
    rng = np.random.default_rng(n)
    lo, up = rng.uniform(-1.0, 0.0, n - 1), rng.uniform(-1.0, 0.0, n - 1)
    import scipy.sparse as sp

    m = sp.diags([lo, np.full(n, 4.0), up], [-1, 0, 1], format="csr")
    a = ca.CsrMatrix.from_scipy(m)
    b = torch.from_numpy(rng.uniform(-1.0, 1.0, n)).cuda()
    x = torch.zeros_like(b)
    rep = gmres_exact_restart(a, b, None, x, ca.IterativeSolverConfig.new(1e-12).with_max_iterations(200), 32)
    assert rep.termination == ca.Termination.Converged and rep.iterations <= 40
    r = b.cpu().numpy() - m @ x.cpu().numpy()
    assert np.linalg.norm(r) <= 1.1e-12 * np.linalg.norm(b.cpu().numpy())

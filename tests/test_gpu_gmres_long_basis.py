"""GMRES over more than 32 basis vectors (separate multi-dots and multi-axpys)
on vectors of a lane's last rows, one block's, and around the 262,144 rows at
which the multi-dots' blocks take a fifth row per lane.

The operator is a diagonally dominant tridiagonal one of condition about 40,
which needs some 45 vectors for 1e-11 within one cycle; the dots are held to
what a cycle needs, a residual estimate that the explicit residual confirms in
the same number of steps as on the smallest system, give or take 2 (the
right-hand sides are random)."""
import numpy as np
import pytest
import torch

import cfdrs_amd as ca
from cfdrs_amd.linear_solver import gmres_exact_restart

pytestmark = pytest.mark.gpu


def solve(n, precision, tol):
    import scipy.sparse as sp

    rng = np.random.default_rng(7)
    m = sp.diags([np.full(n - 1, -1.0), np.full(n, 2.1), np.full(n - 1, -0.999)], [-1, 0, 1], format="csr")
    a = ca.CsrMatrix.from_scipy(m)
    b = rng.uniform(-1.0, 1.0, n)
    x = torch.zeros(n, dtype=torch.float64, device="cuda")
    cfg = ca.IterativeSolverConfig.new(tol).with_max_iterations(400).with_precision(precision)
    rep = gmres_exact_restart(a, torch.from_numpy(b).cuda(), None, x, cfg, 128)
    assert rep.termination == ca.Termination.Converged
    assert np.linalg.norm(b - m @ x.cpu().numpy()) <= 1.01 * tol * np.linalg.norm(b)
    return rep.iterations


@pytest.mark.parametrize("precision,tol", [(ca.Precision.FP64, 1e-11), (ca.Precision.FP32_REFINED, 1e-9)])
def test_long_basis(precision, tol):
    first = solve(1025, precision, tol)
    assert precision != ca.Precision.FP64 or 34 < first <= 128
    for n in (4097, 65537, 262143, 262144, 262145, 300001):
        assert abs(solve(n, precision, tol) - first) <= (2 if precision == ca.Precision.FP64 else 8), n

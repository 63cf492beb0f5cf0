"""FP32-inner CG that stops on its recursive residual and goes on from the FP64
one: the products enqueued behind the stop must leave the direction as it was,
in every row.

The host enqueues check_every steps at a time and learns of the stop a chunk
later, so the number of skipped products, and with it the buffer that holds the
direction afterwards, depends on check_every, and nothing else may: with no
replacement in between (a reliable_interval beyond the budget) the solve runs
the same operations on the same values for every check_every.  Equal iteration
counts and equal bits are asked for.  Row counts whose 256-row tiles are not a
multiple of 8 leave blocks of the product without a tile."""
import numpy as np
import pytest

import cfdrs_amd as ca
from cfdrs_amd import problems as P

pytestmark = pytest.mark.gpu

GRIDS = [(100, 90, 1), (101, 91, 1), (200, 151, 1), (31, 33, 29), (64, 64, 1), (32, 32, 32)]


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("prec", ["jacobi", "amg"])
def test_resumes_with_the_direction_it_stopped_with(grid, prec):
    nx, ny, nz = grid
    n = nx * ny * nz
    k = np.exp(P.uniform(71, n, -1.0, 1.0))
    rp, ci, v, _ = P.varcoef(nx, ny, nz, 1.0, k, 0b000010, np.zeros(6))
    b = P.uniform(72, n)
    a = ca.CsrMatrix.from_parts(v, ci, rp, n, n)
    assert a.storage()["format"] == "dia"
    m = ca.JacobiPreconditioner(a) if prec == "jacobi" else ca.AlgebraicMultigrid(
        a, ca.AMGConfig.smoothed_aggregation())
    resumed = 0
    for tol in (1e-5, 3e-6, 1e-6, 5e-7, 3e-7, 2e-7, 1e-7, 1e-10):
        out = []
        for every in (1, 2, 3, 4, 5, 8):
            cfg = ca.IterativeSolverConfig.new(tol).with_max_iterations(4000).with_precision(
                ca.Precision.FP32_REFINED).with_reliable_interval(1 << 20)
            cfg.check_every = every
            x = np.zeros(n)
            rep = ca.cg_preconditioned(a, b, m, x, cfg)
            assert rep.termination == ca.Termination.Converged, (tol, every, rep)
            out.append((rep.iterations, rep.outer_iterations, x))
        resumed += out[0][1] > 1
        for every, o in zip((2, 3, 4, 5, 8), out[1:]):
            assert o[:2] == out[0][:2] and np.array_equal(o[2], out[0][2]), (tol, every, o[:2], out[0][:2])
    assert resumed >= 1

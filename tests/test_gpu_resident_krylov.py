"""CG and BiCGSTAB with the iterations in one launch (diagonal storage, Jacobi
or no preconditioner) against the launch per phase that the same matrix takes
in row-block storage.

After a few iterations the two iterates differ by rounding alone: sums of at
most 5e5 terms in other orders (relative 1e-13), carried through 12 iterations
of an operator whose scaled condition number is at most some hundred in that
span; 1e-9 leaves a factor of 100.  FP32 inner iterations: 1e-4 of the same.
Converged solves are held to their explicit residual and to the same number of
iterations within 2%, at least 2 (the residual falls below the threshold at one
or the next).  Sizes: the smallest diagonal storage, ragged last blocks, the
largest halo and one more, the edges of 1, 2 and 4 rows per thread, the largest
systems and one row more."""
import numpy as np
import pytest

import cfdrs_amd as ca
from cfdrs_amd import problems as P
from cfdrs_amd.linear_solver import SolveError

pytestmark = pytest.mark.gpu

GRIDS = [(64, 64, 1), (41, 103, 1), (73, 71, 1), (1023, 12, 1), (1024, 12, 1), (1025, 12, 1), (128, 128, 1),
         (256, 256, 1), (257, 256, 1), (362, 363, 1), (512, 512, 1), (513, 512, 1), (24, 25, 22), (32, 32, 32),
         (1024, 512, 1), (1024, 513, 1)]


def system(nx, ny, nz, symmetric):
    n = nx * ny * nz
    k = np.exp(P.uniform(71, n, -1.0, 1.0))
    rp, ci, v, _ = P.varcoef(nx, ny, nz, 1.0, k, 0b000011, np.zeros(6))
    if not symmetric:
        rows = np.repeat(np.arange(n), np.diff(rp))
        v = np.where(ci < rows, 1.2 * v, v)
        v = np.where(ci == rows, 1.2 * v, v)
    return rp, ci, v, P.uniform(72, n), n


def solve(a, method, precond, b, tol, its, precision):
    cfg = ca.IterativeSolverConfig.new(tol).with_max_iterations(its).with_precision(precision)
    x = np.zeros(b.size)
    if not precond:
        return (ca.cg if method == "cg" else ca.bicgstab)(a, b, x, cfg), x
    run = ca.cg_preconditioned if method == "cg" else ca.bicgstab_preconditioned
    return run(a, b, ca.JacobiPreconditioner(a), x, cfg), x


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("method,symmetric", [("cg", True), ("bicgstab", True), ("bicgstab", False)])
def test_matches_a_launch_per_phase(grid, method, symmetric):
    rp, ci, v, b, n = system(*grid, symmetric)
    pair = [ca.CsrMatrix.from_parts(v, ci, rp, n, n) for _ in range(2)]
    pair[1].set_storage("csr_rowblock")
    assert pair[0].storage()["format"] == "dia"
    for precond in (True, False):
        for precision, tol in ((ca.Precision.FP64, 1e-9), (ca.Precision.FP32_REFINED, 1e-4)):
            its = 12
            (ra, x), (rb, y) = (solve(a, method, precond, b, 1e-14, its, precision) for a in pair)
            assert ra.iterations == rb.iterations and ra.termination == rb.termination, (ra, rb)
            assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y), (precond, precision)


@pytest.mark.parametrize("grid", [(73, 71, 1), (128, 128, 1), (257, 256, 1), (32, 32, 32)])
@pytest.mark.parametrize("method,symmetric", [("cg", True), ("bicgstab", False)])
@pytest.mark.parametrize("precision", [ca.Precision.FP64, ca.Precision.FP32_REFINED])
def test_converges_like_a_launch_per_phase(grid, method, symmetric, precision):
    rp, ci, v, b, n = system(*grid, symmetric)
    rows = np.repeat(np.arange(n), np.diff(rp))
    out = []
    for storage in ("auto", "csr_rowblock"):
        a = ca.CsrMatrix.from_parts(v, ci, rp, n, n)
        a.set_storage(storage)
        rep, x = solve(a, method, True, b, 1e-10, 5000, precision)
        assert rep.termination == ca.Termination.Converged, (storage, rep)
        res = b - np.bincount(rows, weights=v * x[ci], minlength=n)
        assert np.linalg.norm(res) <= 1.001e-10 * np.linalg.norm(b), storage
        out.append(rep.iterations)
    if method == "cg" and precision == ca.Precision.FP64:
        assert abs(out[0] - out[1]) <= max(2, out[1] // 50), out


def test_stops_as_a_launch_per_phase_does():
    """A zero right-hand side, a NaN in it, an indefinite operator and a budget
    that ends the solve."""
    rp, ci, v, b, n = system(128, 128, 1, True)
    nan = b.copy()
    nan[777] = np.nan
    cases = [(v, np.zeros(n), 100), (v, nan, 100), (-v, b, 100), (v, b, 1), (v, b, 9)]
    for values, rhs, its in cases:
        got = []
        for storage in ("auto", "csr_rowblock"):
            a = ca.CsrMatrix.from_parts(values, ci, rp, n, n)
            a.set_storage(storage)
            for method in ("cg", "bicgstab"):
                try:
                    rep, _ = solve(a, method, False, rhs, 1e-10, its, ca.Precision.FP64)
                    got.append((rep.termination, rep.iterations))
                except SolveError as e:
                    got.append(str(e))
        assert got[:2] == got[2:], (its, got)

"""Resident CG and BiCGSTAB solves whose workgroups do not wait for each other
long enough: with a limit of one poll a block looks once for sums that take the
others microseconds to publish, so the first launch gives up in one of its first
exchanges, and the solve goes on with a launch per phase.

A launch that gave up has changed neither x nor the scalars, and the residual
and the directions are formed anew, so the rest is the solve that takes a launch
per phase from the start, operation for operation: equal reports and equal bits
are asked for.  A resident solve after it has to find everything as before."""
import numpy as np
import pytest

import cfdrs_amd as ca
from cfdrs_amd import problems as P
from cfdrs_amd._native import CfdlaError

pytestmark = pytest.mark.gpu

KINDS = [("cg", True, ca.Precision.FP64), ("cg", True, ca.Precision.FP32_REFINED),
         ("bicgstab", True, ca.Precision.FP64), ("bicgstab", False, ca.Precision.FP64),
         ("bicgstab", False, ca.Precision.FP32_REFINED)]


def system(nx, ny, nz, symmetric):
    n = nx * ny * nz
    k = np.exp(P.uniform(71, n, -1.0, 1.0))
    rp, ci, v, _ = P.varcoef(nx, ny, nz, 1.0, k, 0b000011, np.zeros(6))
    if not symmetric:
        rows = np.repeat(np.arange(n), np.diff(rp))
        v = np.where(ci < rows, 1.2 * v, v)
        v = np.where(ci == rows, 1.2 * v, v)
    return ca.CsrMatrix.from_parts(v, ci, rp, n, n), P.uniform(72, n), P.uniform(73, n, -0.1, 0.1)


def solve(a, method, precond, b, x0, precision):
    # (restarted refinement runs its inner solves as the FP64 one runs)
    cfg = ca.IterativeSolverConfig.new(1e-9).with_max_iterations(6000).with_precision(
        precision).with_reliable_interval(-1)
    x = x0.copy()
    if precond:
        run = ca.cg_preconditioned if method == "cg" else ca.bicgstab_preconditioned
        return run(a, b, ca.JacobiPreconditioner(a), x, cfg), x
    return (ca.cg if method == "cg" else ca.bicgstab)(a, b, x, cfg), x


@pytest.mark.parametrize("grid", [(73, 71, 1), (128, 128, 1), (257, 256, 1), (24, 25, 22)])
@pytest.mark.parametrize("method,symmetric,precision", KINDS)
@pytest.mark.parametrize("precond", [True, False])
def test_goes_on_with_a_launch_per_phase(grid, method, symmetric, precision, precond):
    a, b, x0 = system(*grid, symmetric)
    assert a.storage()["format"] == "dia"
    before, x_before = solve(a, method, precond, b, x0, precision)
    a.set_resident_polls(0)
    plain, y = solve(a, method, precond, b, x0, precision)
    a.set_resident_polls(1)
    gave_up, x = solve(a, method, precond, b, x0, precision)
    assert plain.termination == ca.Termination.Converged
    assert gave_up == plain and np.array_equal(x, y)
    a.set_resident_polls(-1)
    after, x_after = solve(a, method, precond, b, x0, precision)
    assert after == before and np.array_equal(x_after, x_before)
    assert not np.array_equal(x_after, y)  # the resident solve sums in another order


def test_limits_of_the_setting():
    a, _, _ = system(8, 8, 1, True)
    for polls in (-2, (1 << 20) + 1):
        with pytest.raises(CfdlaError):
            a.set_resident_polls(polls)
    a.set_resident_polls(1 << 20)

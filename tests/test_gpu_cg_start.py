"""The PCG update fused with the first two sweeps of the V-cycle (symmetric
diagonal storage of at most five entries per row, up to 262,144 rows) against
the recurrence written out: the residual update on the host, every V-cycle
through apply_to, which makes its own first sweeps.  Sizes: the smallest with
diagonal storage, ragged ones, one diagonal beside the main one, the largest
the fused update takes and the first above; sweep counts that end in either
buffer; the hierarchy of the same matrix and of another one.

After k <= 5 steps from zero the two differ by the rounding of a few sums per
entry and step, 1e-15 each, grown by the step lengths: 1e-10 relative."""
import numpy as np
import pytest
import torch

import cfdrs_amd as ca
from cfdrs_amd import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def system(nx, ny, seed):
    n = nx * ny
    k = np.exp(P.uniform(seed, n, -1.0, 1.0))
    rp, ci, v, _ = P.varcoef(nx, ny, 1, float(nx * nx), k, 0b0010, np.zeros(6))
    return ca.CsrMatrix.from_parts(v, ci, rp, n, n), O.Csr.from_arrays(rp, ci, v, n)


def steps(orc, m, b, k):
    def cycle(r):
        z = torch.empty(len(r), dtype=torch.float64, device="cuda")
        m.apply_to(torch.from_numpy(r).cuda(), z)
        return z.cpu().numpy()

    x, r = np.zeros_like(b), b.copy()
    z = cycle(r)
    p, rz = z.copy(), r @ z
    for _ in range(k):
        q = orc.spmv(p)
        alpha = rz / (p @ q)
        x += alpha * p
        r = r - alpha * q
        z = cycle(r)
        rz, old = r @ z, rz
        p = z + (rz / old) * p
    return x


@pytest.mark.parametrize("sweeps", [(2, 2), (2, 1), (3, 2)])
@pytest.mark.parametrize("grid", [(64, 64), (67, 65), (4999, 1), (512, 512), (513, 512)])
def test_matches_the_recurrence(grid, sweeps):
    a, orc = system(*grid, 61)
    other, _ = system(*grid, 62)
    n = grid[0] * grid[1]
    assert a.storage()["format"] == "dia"
    b = P.uniform(63, n)
    cfg = ca.AMGConfig.smoothed_aggregation()
    cfg.pre_smooth_iterations, cfg.post_smooth_iterations = sweeps
    for src in (a, other):
        m = ca.AlgebraicMultigrid(src, cfg)
        for k in (1, 2, 5):
            x = np.zeros(n)
            short = ca.IterativeSolverConfig.new(1e-14).with_max_iterations(k)
            rep = ca.cg_preconditioned(a, b, m, x, short.with_precision(ca.Precision.FP64))
            assert rep.iterations == k, rep
            ref = steps(orc, m, b, k)
            assert np.linalg.norm(x - ref) <= 1e-10 * np.linalg.norm(ref), k


def test_solves_to_the_tolerance():
    a, orc = system(131, 97, 71)
    b = P.uniform(72, 131 * 97)
    m = ca.AlgebraicMultigrid(a, ca.AMGConfig.smoothed_aggregation())
    for precision in (ca.Precision.FP64, ca.Precision.FP32_REFINED):
        x = np.zeros_like(b)
        cfg = ca.IterativeSolverConfig.new(1e-10).with_max_iterations(200).with_precision(precision)
        cfg = cfg.with_reliable_interval(-1)  # restarted refinement: the update in FP32
        rep = ca.cg_preconditioned(a, b, m, x, cfg)
        assert rep.termination == ca.Termination.Converged, rep
        assert np.linalg.norm(b - orc.spmv(x)) <= 1e-10 * np.linalg.norm(b)

"""What the statistics of a multigrid hierarchy name: the level whose pre-sweeps
and restriction are one product, and the first level of the dense operator."""
import numpy as np
import pytest

import cfdrs_amd as ca
from cfdrs_amd import problems as P

pytestmark = pytest.mark.gpu


def system(grid, seed):
    nx, ny, nz = grid
    n = nx * ny * nz
    k = np.exp(P.uniform(seed, n, -1.0, 1.0))
    rp, ci, v, _ = P.varcoef(nx, ny, nz, float(nx * nx), k, 0b0010, np.zeros(6))
    return rp, ci, v, n, k


def config(min_coarse, **more):
    cfg = ca.AMGConfig.smoothed_aggregation()
    return ca.AMGConfig(**{**cfg.__dict__, "min_coarse_size": min_coarse, **more})


def close(a, b, tol):
    return torch.linalg.norm(a.double() - b.double()) <= tol * torch.linalg.norm(b.double())


def test_statistics_name_what_runs():
    rp, ci, v, n, _ = system((24, 24, 24), 31)
    a = ca.CsrMatrix.from_parts(v, ci, rp, n, n)
    r, z = P.uniform(33, n), np.empty(n)

    def levels(cfg, gather=None):
        m = ca.AlgebraicMultigrid(a, cfg)
        assert m.statistics.fused_level == -1 and m.statistics.dense_level == -1  # not on the device yet
        if gather:
            m.set_gather(gather)
        m.apply_to(r, z)
        s = m.statistics
        return s.level_sizes, s.fused_level, s.dense_level

    sizes, fused, dense = levels(config(100))
    first = next(l for l in range(1, len(sizes)) if sizes[l] <= 2048)
    assert (fused, dense) == (len(sizes) - 2, first) and dense < len(sizes) - 1
    assert levels(config(100, separate_coarse_restriction=True))[1:] == (-1, -1)
    assert levels(config(100), "quad")[1:] == (len(sizes) - 2, -1)
    assert levels(config(100, post_smooth_iterations=1, pre_smooth_iterations=1))[1:] == (-1, -1)
    # the default hierarchy (Gauss-Seidel): the tail's levels behind its first small one
    sizes, fused, dense = levels(ca.AMGConfig.default())
    assert fused == -1 and (dense == -1 or sizes[dense] <= 2048)

"""The pre-sweeps and the restriction of the level above a dense coarsest level
as one product F, on hierarchies that build it: a level of more than 2,048 rows
above the coarsest one, or a coarsest level of more than 512 rows (smaller ones
run as one dense operator instead).  F in padded rows and in row blocks (a
forced gather layout) against the three separate products and the oracle, in
FP64 and FP32, before and after a device recompute; and what the statistics
name for each kind of hierarchy.

F's rows are cut into pieces that the coarse solve adds: a coarse entry is a sum
of at most some 2,000 products whichever way it is formed, three operators in a
row: sqrt(2000) 3 roundings are 1.5e-14 and 8e-6 of the cycle; 2e-13 and 2e-5
are allowed."""
import numpy as np
import pytest
import torch

import cfdrs_amd as ca
from cfdrs_amd import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu

FUSED = [((112, 108, 1), 400), ((130, 120, 1), 400), ((190, 185, 1), 1000), ((32, 30, 28), 400)]


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


def padded_lanes(widths):
    """Lanes per row of an operator in padded rows, 0 where it stays in row
    blocks: 4 entries per lane, at most 64 lanes, 700,000 slots, and three times
    the entries."""
    lanes = 1
    while 4 * lanes < widths.max():
        lanes *= 2
    slots = 4 * lanes * widths.size
    return lanes if lanes <= 64 and slots <= min(700000, 3 * widths.sum() + 4096) else 0


def fused_lanes(m, level):
    """The lanes of F, from the level's patterns."""
    import scipy.sparse as sp

    def pattern(which):
        rp, ci, v, nr, nc = m.level(level, which)
        return sp.csr_matrix((np.ones(v.size), ci, rp), shape=(nr, nc))

    a, r = pattern("A"), pattern("R")
    wide = np.diff((r @ a @ a).indptr)
    s = np.diff(a.indptr)
    piece = 4 * max(8, padded_lanes(s))
    parts = -(-wide.max() // piece)
    cut = np.clip(wide[:, None] - piece * np.arange(parts), 0, piece)
    return padded_lanes(np.concatenate([s, cut.ravel()])) if padded_lanes(s) else 0


@pytest.mark.parametrize("grid,min_coarse", FUSED)
def test_matches_separate_products(grid, min_coarse):
    rp, ci, v, n, _ = system(grid, 31)
    a = ca.CsrMatrix.from_parts(v, ci, rp, n, n)
    fused = ca.AlgebraicMultigrid(a, config(min_coarse))
    blocks = ca.AlgebraicMultigrid(a, config(min_coarse))
    blocks.set_gather("quad")
    plain = ca.AlgebraicMultigrid(a, config(min_coarse, separate_coarse_restriction=True))
    r = torch.from_numpy(P.uniform(33, n)).cuda()

    def check():
        for dtype, tol in ((torch.float64, 2e-13), (torch.float32, 2e-5)):
            rr = r.to(dtype)
            z, w, y = (torch.empty_like(rr) for _ in range(3))
            fused.apply_to(rr, z)
            blocks.apply_to(rr, w)
            plain.apply_to(rr, y)
            assert close(z, y, tol) and close(w, y, tol) and close(z, w, tol), dtype
            if dtype == torch.float64:
                out = z.cpu().numpy()
        return out

    z = check()
    L = fused.statistics.num_levels
    rows = fused.level(L - 2, "A")[3]
    assert L >= 3 and (rows > 2048 or fused.level(L - 1, "A")[3] > 512)
    assert fused_lanes(fused, L - 2) > 0  # in padded rows
    for m, level in ((fused, L - 2), (blocks, L - 2), (plain, -1)):
        assert m.statistics.fused_level == level and m.statistics.dense_level == -1
    cfg = config(min_coarse)
    oamg = O.Amg(O.Csr.from_arrays(rp, ci, v, n), coarsening="three_phase", interp="smoothed", smoother="jacobi",
                 omega=cfg.relaxation_factor, coarse_solve="direct", sa_omega=cfg.smoothing_omega,
                 theta=cfg.strength_threshold, min_coarse=cfg.min_coarse_size)
    zo = oamg.apply(r.cpu().numpy())
    assert np.linalg.norm(z - zo) <= 1e-11 * np.linalg.norm(zo)
    k = system(grid, 32)[4]
    a.varcoef_refresh_device(*grid, float(grid[0] ** 2), torch.from_numpy(k).cuda(), 0b0010, np.zeros(6))
    for m in (fused, blocks, plain):
        m.recompute_device(a)
    assert np.linalg.norm(check() - z) > 1e-3 * np.linalg.norm(z)


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

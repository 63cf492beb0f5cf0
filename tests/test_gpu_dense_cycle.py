"""The last levels of a V-cycle as one dense operator against the same levels
run one by one (a hierarchy that asks for separate restriction products), for
operators of up to 512, 1024, 1536 and 2048 rows and the first size above, in
FP64 and FP32; and hierarchies recomputed on the device against ones recomputed
on the host, which form the operator from the same values: equal bits.

The operator's entries are sums of at most a few hundred products per level, of
five operators in a row, and a row of it has at most 2048 terms: 1e-13 relative
to the cycle, and FP32 vectors' rounding, 1e-5."""
import numpy as np
import pytest
import torch

import cfdrs_amd as ca
from cfdrs_amd import problems as P

pytestmark = pytest.mark.gpu

GRIDS = [((53, 55), 512), ((76, 79), 1024), ((91, 96), 1536), ((110, 110), 2048), ((112, 108), 1 << 30)]


def system(nx, ny, seed):
    n = nx * ny
    k = np.exp(P.uniform(seed, n, -1.0, 1.0))
    rp, ci, v, _ = P.varcoef(nx, ny, 1, float(nx * nx), k, 0b0010, np.zeros(6))
    return ca.CsrMatrix.from_parts(v, ci, rp, n, n), n


@pytest.mark.parametrize("grid,most", GRIDS)
def test_matches_level_by_level(grid, most):
    a, n = system(*grid, 81)
    cfg = ca.AMGConfig.smoothed_aggregation()
    cfg.min_coarse_size = 60
    sep = ca.AMGConfig(**{**cfg.__dict__, "separate_coarse_restriction": True})
    m, plain = ca.AlgebraicMultigrid(a, cfg), ca.AlgebraicMultigrid(a, sep)
    rows = m.level(1, "A")[3]
    assert m.statistics.num_levels >= 3 and (most // 2 if most < 4096 else 2048) < rows <= most, rows
    for s in range(3):
        r = torch.from_numpy(P.uniform(82 + s, n)).cuda()
        for dtype, tol in ((torch.float64, 1e-13), (torch.float32, 1e-5)):
            x, y = torch.empty_like(r, dtype=dtype), torch.empty_like(r, dtype=dtype)
            m.apply_to(r.to(dtype), x)
            plain.apply_to(r.to(dtype), y)
            assert torch.linalg.norm(x.double() - y.double()) <= tol * torch.linalg.norm(y.double()), (dtype, s)


@pytest.mark.parametrize("kind", ["jacobi", "gauss-seidel"])
@pytest.mark.parametrize("grid", [(53, 55), (76, 79), (91, 96), (110, 105)])
def test_recompute_forms_the_same_operator(kind, grid):
    a, n = system(*grid, 91)
    b, _ = system(*grid, 91)
    cfg = ca.AMGConfig.smoothed_aggregation() if kind == "jacobi" else ca.AMGConfig.default()
    dev, host = ca.AlgebraicMultigrid(a, cfg), ca.AlgebraicMultigrid(b, cfg)
    for seed in (92, 93):
        v = system(*grid, seed)[0].creation_order_values()
        a.update_values_device(torch.from_numpy(np.ascontiguousarray(v)).cuda())
        dev.recompute_device(a)
        b.update_values(v)
        host.recompute(b)
        r = P.uniform(94, n)
        for dtype in (torch.float64, torch.float32):
            rr = torch.from_numpy(r).to(dtype).cuda()
            x, y = torch.empty_like(rr), torch.empty_like(rr)
            dev.apply_to(rr, x)
            host.apply_to(rr, y)
            assert torch.equal(x, y) and torch.linalg.norm(x) > 0, (dtype, seed)

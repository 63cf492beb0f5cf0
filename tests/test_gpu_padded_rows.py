"""The padded-row layout of an AMG hierarchy's small operators against the
row-block layouts of the same hierarchy (which a forced gather layout brings
back): V-cycles in FP64 and FP32 on 2D and 3D grids, so that the transfers and
coarse levels have 1 to 64 lanes per row, before and after a device recompute.

Both sum each row's products in an order of their own: rows of at most 256
entries, values of one sign pattern, so the relative difference of a V-cycle
stays within a few hundred roundings (1e-13, 2e-5)."""
import numpy as np
import pytest
import torch

import cfdrs_amd as ca
from cfdrs_amd import problems as P

pytestmark = pytest.mark.gpu

GRIDS = [(65, 63, 1), (97, 101, 1), (256, 40, 1), (300, 210, 1), (14, 15, 16), (24, 22, 20)]


def close(a, b, tol):
    return torch.linalg.norm(a.double() - b.double()) <= tol * torch.linalg.norm(b.double())


@pytest.mark.parametrize("nx,ny,nz", GRIDS)
@pytest.mark.parametrize("separate", [False, True])
def test_vcycle_matches_row_blocks(nx, ny, nz, separate):
    n = nx * ny * nz
    ks = [np.exp(P.uniform(s, n, -1.0, 1.0)) for s in (31, 32)]
    rp, ci, v, _ = P.varcoef(nx, ny, nz, float(nx * nx), ks[0], 0b0010, np.zeros(6))
    a = ca.CsrMatrix.from_parts(v, ci, rp, n, n)
    cfg = ca.AMGConfig.smoothed_aggregation()
    cfg.min_coarse_size = 60
    cfg.separate_coarse_restriction = separate
    padded, blocks = ca.AlgebraicMultigrid(a, cfg), ca.AlgebraicMultigrid(a, cfg)
    blocks.set_gather("quad")
    r = torch.from_numpy(P.uniform(33, n)).cuda()
    for k in (None, torch.from_numpy(ks[1]).cuda()):
        if k is not None:
            a.varcoef_refresh_device(nx, ny, nz, float(nx * nx), k, 0b0010, np.zeros(6))
            padded.recompute_device(a)
            blocks.recompute_device(a)
        for dtype, tol in ((torch.float64, 1e-13), (torch.float32, 2e-5)):
            rr = r.to(dtype)
            z, w = torch.empty_like(rr), torch.empty_like(rr)
            padded.apply_to(rr, z)
            blocks.apply_to(rr, w)
            assert close(z, w, tol), (dtype, k is not None)

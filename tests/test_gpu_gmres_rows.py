"""GMRES with multicolour SOR where the passes have one row per thread, the
product is formed in the first of them and the sweep starts in the scaling of
its argument: diagonal storage against the same matrix in row blocks (whose
product is a launch of its own), with 2 and 4 colours, 5 to 9 entries per row,
around a block's rows, and at the largest system of that form and the first of
the general one (which sweeps and scales apart).

The two iterates differ by the products' rounding, 1e-16 per step, carried
through at most two cycles of well-conditioned steps: 1e-11."""
import numpy as np
import pytest

import cfdrs_amd as ca
from cfdrs_amd import problems as P
from cfdrs_amd.linear_solver import gmres_exact_restart

pytestmark = pytest.mark.gpu


def stencil(nx, ny, nz, corners, seed):
    """Diagonally dominant nonsymmetric 5-, 7- or 9-point operator."""
    n = nx * ny * nz
    i = np.arange(n)
    x, y, z = i % nx, i // nx % ny, i // (nx * ny)
    steps = [(-1, 0, 0), (1, 0, 0), (0, -1, 0), (0, 1, 0)] + ([(0, 0, -1), (0, 0, 1)] if nz > 1 else [])
    if corners:
        steps += [(a, b, 0) for a in (-1, 1) for b in (-1, 1)]
    rows, cols, vals = [i], [i], [np.full(n, 1.0 + 0.1 * len(steps))]
    for k, (a, b, c) in enumerate(steps):
        ok = (x + a >= 0) & (x + a < nx) & (y + b >= 0) & (y + b < ny) & (z + c >= 0) & (z + c < nz)
        rows.append(i[ok])
        cols.append(i[ok] + a + b * nx + c * nx * ny)
        vals.append(-P.uniform(seed + k, n, 0.05, 0.95 / len(steps) + 0.1)[ok])
    r, c, v = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)
    order = np.lexsort((c, r))
    rp = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))])
    return rp, c[order], v[order], n


@pytest.mark.parametrize("grid,corners", [((64, 64, 1), False), ((65, 64, 1), False), ((79, 92, 1), False),
                                          ((17, 16, 16), False), ((70, 66, 1), True), ((512, 512, 1), False),
                                          ((513, 512, 1), False)])
@pytest.mark.parametrize("m", [1, 8, 30])
def test_matches_row_blocks(grid, corners, m):
    rp, ci, v, n = stencil(*grid, corners, 31)
    b = P.uniform(32, n)
    for precision, tol in ((ca.Precision.FP64, 1e-11), (ca.Precision.FP32_REFINED, 1e-4)):
        out = []
        for storage in ("auto", "csr_rowblock"):
            a = ca.CsrMatrix.from_parts(v, ci, rp, n, n)
            a.set_storage(storage)
            x = np.zeros(n)
            cfg = ca.IterativeSolverConfig.new(1e-13).with_max_iterations(min(2 * m, 40)).with_precision(precision)
            rep = gmres_exact_restart(a, b, ca.SuccessiveOverRelaxation(a, 1.1), x, cfg, m)
            out.append((rep.termination, x))
        assert out[0][0] == out[1][0]
        assert np.linalg.norm(out[0][1] - out[1][1]) <= tol * np.linalg.norm(out[1][1]), precision

"""The one-workgroup tail of the Gauss-Seidel V-cycle against the same cycle
in numpy on the exported hierarchy, at sizes where the tail starts on the
finest level, below it (more than 10,047 rows) and where a colour holds one
row more or less than the workgroup's threads."""
import numpy as np
import pytest
import torch

import cfdrs_amd as ca
from cfdrs_amd import problems as P

pytestmark = pytest.mark.gpu


def colours(rp, ci, n):
    """Greedy colouring in breadth-first order on the symmetrized pattern."""
    adj = [[] for _ in range(n)]
    for i in range(n):
        for j in ci[rp[i]:rp[i + 1]]:
            if j != i:
                adj[i].append(int(j))
                adj[int(j)].append(i)
    seen, order = np.zeros(n, bool), []
    for root in range(n):
        if seen[root]:
            continue
        seen[root] = True
        order.append(root)
        head = len(order) - 1
        while head < len(order):
            # neighbours in the order the library lists them: by row, then entry
            for j in adj[order[head]]:
                if not seen[j]:
                    seen[j] = True
                    order.append(j)
            head += 1
    col = np.full(n, -1)
    for i in order:
        used = {col[j] for j in adj[i]}
        c = 0
        while c in used:
            c += 1
        col[i] = c
    return col


class Cycle:
    def __init__(self, amg, cfg):
        self.cfg, self.lv = cfg, []
        L = amg.statistics.num_levels
        for q in range(L):
            rp, ci, v, n, _ = amg.level(q, "A")
            rows = np.repeat(np.arange(n), np.diff(rp))
            a = (rows, ci, v, n)
            d = np.zeros(n)
            d[rows[rows == ci]] = v[rows == ci]
            pr = []
            if q + 1 < L:
                for which in ("P", "R"):
                    r, c, w, m, _ = amg.level(q, which)
                    pr.append((np.repeat(np.arange(m), np.diff(r)), c, w, m))
            self.lv.append((a, d, colours(rp, ci, n), pr))

    @staticmethod
    def mul(a, x):
        return np.bincount(a[0], weights=a[2] * x[a[1]], minlength=a[3])

    def sweeps(self, q, b, x, k):
        a, d, col, _ = self.lv[q]
        nc = col.max() + 1
        passes = [list(range(nc))] * k
        if self.cfg.smoother_type == ca.SmootherType.SymmetricGaussSeidel:
            passes = passes + [list(range(nc - 1, -1, -1))] * k
        for one in passes:
            for c in one:
                on = col == c
                nv = (b - (self.mul(a, x) - d * x)) / d
                x = np.where(on, x + self.cfg.relaxation_factor * (nv - x), x)
        return x

    def run(self, q, b):
        a, _, _, pr = self.lv[q]
        x = np.zeros(a[3])
        if q + 1 == len(self.lv):
            if self.cfg.coarse_solver == ca.CoarseSolver.Direct:
                m = np.zeros((a[3], a[3]))
                m[a[0], a[1]] = a[2]
                return np.linalg.solve(m, b)
            return self.sweeps(q, b, self.sweeps(q, b, x, self.cfg.pre_smooth_iterations), 10)
        x = self.sweeps(q, b, x, self.cfg.pre_smooth_iterations)
        e = self.run(q + 1, self.mul(pr[1], b - self.mul(a, x)))
        return self.sweeps(q, b, x + self.mul(pr[0], e), self.cfg.post_smooth_iterations)


def config(**kw):
    c = ca.AMGConfig.default()
    for k, v in kw.items():
        setattr(c, k, v)
    return c


CASES = [
    (45, 45, {}),   # 1,012 / 1,013 rows per colour
    (64, 32, {}),   # 1,024 rows per colour
    (41, 50, {"smoother_type": ca.SmootherType.SymmetricGaussSeidel}),
    (9, 7, {"relaxation_factor": 1.2, "smoother_type": ca.SmootherType.SOR}),
    (51, 197, {"post_smooth_iterations": 1}),   # 10,047 rows: tail on the finest level
    (101, 102, {"coarse_solver": ca.CoarseSolver.Direct}),  # 10,302 rows: the finest level by launches
    (50, 37, {"coarse_solver": ca.CoarseSolver.Direct, "pre_smooth_iterations": 0}),
    (30, 30, {"max_levels": 1}),
    (25, 41, {"coarsening_strategy": ca.CoarseningStrategy.Aggregation,
              "interpolation_strategy": ca.InterpolationStrategy.Direct, "max_levels": 3}),
]


@pytest.mark.parametrize("nx,ny,options", CASES)
@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-12), (torch.float32, 2e-4)])
def test_vcycle_matches_numpy(nx, ny, options, dtype, tol):
    k = np.exp(P.uniform(5, nx * ny, -1.0, 1.0))
    rp, ci, v, _ = P.varcoef(nx, ny, 1, float(nx * nx), k, 0b0010, np.zeros(6))
    a = ca.CsrMatrix.from_parts(v, ci, rp, nx * ny, nx * ny)
    cfg = config(**options)
    amg = ca.AlgebraicMultigrid(a, cfg)
    b = P.uniform(6, nx * ny)
    want = Cycle(amg, cfg).run(0, b)
    r = torch.from_numpy(b).to("cuda", dtype)
    z = torch.empty_like(r)
    amg.apply_to(r, z)
    err = np.linalg.norm(z.double().cpu().numpy() - want) / np.linalg.norm(want)
    assert err <= tol, err


def test_device_recompute_reaches_the_tail():
    nx, ny = 40, 33
    ks = [np.exp(P.uniform(s, nx * ny, -1.0, 1.0)) for s in (7, 8)]
    rp, ci, v, _ = P.varcoef(nx, ny, 1, 1.0, ks[0], 0b0010, np.zeros(6))
    a = ca.CsrMatrix.from_parts(v, ci, rp, nx * ny, nx * ny)
    cfg = config()
    amg = ca.AlgebraicMultigrid(a, cfg)
    r = torch.from_numpy(P.uniform(9, nx * ny)).cuda()
    z = torch.empty_like(r)
    amg.apply_to(r, z)
    a.varcoef_refresh_device(nx, ny, 1, 1.0, torch.from_numpy(ks[1]).cuda(), 0b0010, np.zeros(6))
    amg.recompute_device(a)
    amg.apply_to(r, z)
    want = Cycle(amg, cfg).run(0, r.cpu().numpy())
    assert np.linalg.norm(z.cpu().numpy() - want) <= 1e-12 * np.linalg.norm(want)

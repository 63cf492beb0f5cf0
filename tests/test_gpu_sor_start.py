"""The fused start of a multicolour SOR sweep (first and second colour in one
launch) against the sweep written out in numpy, on bipartite patterns whose
second-colour rows couple to 1 .. 9 rows: every slot width of the fused
kernel, the widths between them, and the longest row that leaves the second
colour to a launch of its own; and on a three-colour pattern."""
import numpy as np
import pytest
import torch

import cfdrs_amd as ca

pytestmark = pytest.mark.gpu


def sweep(rows, cols, vals, n, colour, omega, r):
    d = np.zeros(n)
    d[rows[rows == cols]] = vals[rows == cols]
    z = np.zeros(n)
    for c in range(colour.max() + 1):
        off = rows != cols
        acc = r - np.bincount(rows[off], weights=vals[off] * z[cols[off]], minlength=n)
        z = np.where(colour == c, omega / d * acc, z)
    return z


def matrix(entries, n):
    rows = np.array([e[0] for e in entries])
    cols = np.array([e[1] for e in entries])
    vals = np.array([e[2] for e in entries])
    order = np.lexsort((cols, rows))
    rows, cols, vals = rows[order], cols[order], vals[order]
    rp = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))])
    return rows, cols, vals, ca.CsrMatrix.from_parts(vals, cols, rp, n, n)


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-13), (torch.float32, 1e-5)])
def test_bipartite_sweep(k, dtype, tol):
    # even rows are coupled to the k odd rows around them (a connected strip)
    n = 2 * 701
    rng = np.random.default_rng(k)
    e = [(i, i, 4.0 + rng.random()) for i in range(n)]
    pairs = set()
    for i in range(0, n, 2):
        for q in range(k):
            j = i + 1 + 2 * (q - k // 2)
            if 0 < j < n:
                pairs.add((i, j))
        if i + 2 < n:
            pairs.add((i + 2, i + 1))
    for i, j in pairs:
        e += [(i, j, -rng.random()), (j, i, -rng.random())]
    rows, cols, vals, a = matrix(e, n)
    sor = ca.SuccessiveOverRelaxation(a, 1.1)
    assert sor.colours == 2
    r = rng.uniform(-1.0, 1.0, n)
    want = sweep(rows, cols, vals, n, np.arange(n) % 2, 1.1, r)
    rt = torch.from_numpy(r).to("cuda", dtype)
    z = torch.empty_like(rt)
    sor.apply_to(rt, z)
    assert np.linalg.norm(z.double().cpu().numpy() - want) <= tol * np.linalg.norm(want)


def test_three_colours_follow_the_fused_start():
    # a ring of triangles: every row meets both other colours
    m = 400
    n = 3 * m
    rng = np.random.default_rng(5)
    e = [(i, i, 5.0) for i in range(n)]
    for t in range(m):
        a, b, c = 3 * t, 3 * t + 1, 3 * t + 2
        for i, j in ((a, b), (b, c), (a, c)) + (((c, a + 3),) if t + 1 < m else ()):
            v = -rng.random()
            e += [(i, j, v), (j, i, v)]
    rows, cols, vals, a = matrix(e, n)
    sor = ca.SuccessiveOverRelaxation(a, 0.9)
    assert sor.colours == 3
    # breadth-first greedy colours of this ring, row by row from row 0
    colour = np.full(n, -1)
    adj = [[] for _ in range(n)]
    for i, j in zip(rows, cols):
        if i != j:
            adj[i].append(j)
    order, seen = [0], {0}
    for i in order:
        for j in sorted(adj[i]):
            if j not in seen:
                seen.add(j)
                order.append(j)
    for i in order:
        used = {colour[j] for j in adj[i]}
        colour[i] = min(c for c in range(4) if c not in used)
    r = rng.uniform(-1.0, 1.0, n)
    z = np.empty(n)
    sor.apply_to(r, z)
    want = sweep(rows, cols, vals, n, colour, 0.9, r)
    assert np.linalg.norm(z - want) <= 1e-13 * np.linalg.norm(want)

"""The device Gauss-Jordan inverse of a coarsest level against the host's: one-
level hierarchies whose matrix needs row exchanges, at the edges of its panels
(16 columns), wavefronts (64 rows) and block sizes, recomputed on either side.
Both run the same operations in the same order: equal bits."""
import numpy as np
import pytest
import torch

import cfdrs_amd as ca
from cfdrs_amd import problems as P

pytestmark = pytest.mark.gpu


def general(n, seed):
    """A cyclic shift with large entries, a weak diagonal and a band: every
    column's pivot lies off the diagonal; some entries are exact zeros."""
    i = np.arange(n)
    cols = np.unique(np.stack([i, (i + 1) % n, (i + 3) % n, (i * 7 + 2) % n]), axis=0)
    a = np.zeros((n, n))
    for k, c in enumerate(cols):
        a[i, c] += P.uniform(seed + k, n, -0.3, 0.3)
    a[i, (i + 1) % n] += 2.0
    a[i[::5], (i[::5] + 3) % n] *= 0.0
    rp = np.concatenate([[0], np.cumsum([len(np.unique(cols[:, r])) for r in range(n)])])
    ci = np.concatenate([np.unique(cols[:, r]) for r in range(n)])
    rows = np.repeat(i, np.diff(rp))
    return rp.astype(np.int64), ci.astype(np.int64), a[rows, ci]


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 33, 63, 64, 65, 129, 255, 256, 257, 400, 512, 513, 1023, 1024, 1025])
def test_matches_host(n):
    rp, ci, v = general(n, 40)
    cfg = ca.AMGConfig.smoothed_aggregation()
    cfg.min_coarse_size = n + 1
    a = ca.CsrMatrix.from_parts(v, ci, rp, n, n)
    b = ca.CsrMatrix.from_parts(v, ci, rp, n, n)
    dev, host = ca.AlgebraicMultigrid(a, cfg), ca.AlgebraicMultigrid(b, cfg)
    assert dev.statistics.num_levels == 1
    for k in range(2):
        v2 = general(n, 50 + k)[2]
        a.update_values_device(torch.from_numpy(v2).cuda())
        b.update_values(v2)
        if not v2.any():  # one row, its entry zero: singular on either side
            for solve in (lambda: dev.recompute_device(a), lambda: (host.recompute(b), host.apply_to(v2, v2.copy()))):
                with pytest.raises(ca.CfdlaError, match="singular"):
                    solve()
            continue
        dev.recompute_device(a)
        host.recompute(b)
        for s in range(3):
            r = P.uniform(60 + s, n)
            x, y = np.empty(n), np.empty(n)
            dev.apply_to(r, x)
            host.apply_to(r, y)
            assert np.array_equal(x.view(np.int64), y.view(np.int64)), (n, k, s)
            assert s or np.abs(x).max() > 0

"""The wavefront sums behind every dot product, on integer data: all partial
sums are exact in FP64, so the norm must equal the host's to the last bit
whatever the tree, and a lane that is dropped or counted twice changes it."""
import numpy as np
import pytest

import cfdrs_amd as ca

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 63, 64, 65, 127, 255, 256, 257, 1023, 1024, 1025, 4099, 300001])
def test_initial_residual_norm_is_exact_on_integers(n):
    a = ca.CsrMatrix.from_parts(np.ones(n), np.arange(n), np.arange(n + 1), n, n)
    # distinct powers of two per lane within a wavefront, small integers across wavefronts
    b = np.where(np.arange(n) % 64 < 20, 2.0 ** (np.arange(n) % 64 % 10), 1.0 + np.arange(n) % 7)
    rep = ca.cg(a, b, np.zeros(n), ca.IterativeSolverConfig.new(1e-12))
    assert rep.initial_residual_norm == np.sqrt(np.sum(b * b))

"""Kriging weights against systems solved in extended precision: the refinement's residual
is summed in twice the precision, so the weights are rounded values of the solution."""
import numpy as np
import pytest
import scipy.linalg as sl

from oracle import kriging as okr
from test_gpu_kriging_inverse import _images, _mask

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,radius", [("full", 3.1), ("ellipsoid", 4.2), ("most", 4.2)])
def test_refined_weights_are_accurate(kind, radius):
    from dualres_amd.kriging import kriging_build
    dims, theta = (14, 12, 10), (0.806, 0.132, 1.5)
    hr, q, std, qs = _images(dims, _mask(kind, dims))
    W = kriging_build(hr, q, std, qs, theta, radius)
    rows, P, _ = okr.kriging_pattern(hr, std, q, qs, theta, radius)
    K = okr.perturbation_kernel_distances(P, q, theta, dtype=np.float32).astype(np.float64)
    checked = 0
    for i in range(0, len(rows), 2):
        _, pidx, kp = rows[i]
        if 2 * len(pidx) < len(P):
            continue  # solved directly
        A = K[np.ix_(pidx, pidx)]
        c = sl.cho_factor(A)
        x = np.zeros(len(pidx), np.longdouble)
        for _ in range(4):
            r = kp.astype(np.longdouble) - A.astype(np.longdouble) @ x
            x = x + sl.cho_solve(c, r.astype(np.float64))
        x = x / x.sum()
        w = W.data[W.indptr[i]:W.indptr[i + 1]]
        # the update, the sum and the division round each weight a few times; the sum of up to 341 weights
        # of both signs in float64 adds less than 30 eps
        assert np.linalg.norm(w - x) <= 32 * np.finfo(np.float64).eps * np.linalg.norm(x.astype(np.float64))
        checked += 1
    assert checked > 5

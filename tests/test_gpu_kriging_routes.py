"""How the kriging systems are worked on.  Few systems share a batch whatever
their sizes.  Which ones go through the inverse of the whole neighbourhood's
kernel matrix: none, and no inverse computed, where solving them directly is
the less work (few rows, rows that keep little of the neighbourhood) or the
matrix is indefinite or nearly singular.  Weights against the oracle, and the
accuracy of the direct ones."""
import numpy as np
import pytest

from oracle import kriging as okr
from test_gpu_kriging_inverse import _check, _images, _mask

pytestmark = pytest.mark.gpu


def _sizes(n_systems):
    return -(-n_systems // 512)  # batches of at least 512 systems


@pytest.mark.parametrize("dims,kind,radius", [((8, 8, 8), "full", 3.1), ((14, 12, 10), "most", 3.1),
                                              ((24, 20, 16), "most", 2.3)])
def test_few_systems_of_many_sizes_share_a_batch(dims, kind, radius):
    """Indefinite kernels: a batch of systems by Cholesky, those that fail by LU.
    The systems have from a third of the neighbourhood's offsets to all."""
    info = _check(dims, kind, radius, (1.6, 0.05, 1.8))
    assert info["n_lu"] > 0
    cut = 2 if info["n_unique_solves"] > 512 else 0  # past 512 systems a batch ends with its size
    assert info["n_batches"] <= _sizes(info["n_unique_solves"]) + _sizes(info["n_lu"]) + 2 * cut


@pytest.mark.parametrize("dims,kind,radius,built", [
    ((4, 4, 4), "full", 4.2, False),
    ((8, 8, 8), "full", 4.2, False),
    ((16, 14, 12), "most", 4.2, True),
    ((20, 18, 16), "most", 4.2, True),
    ((24, 24, 24), "most", 3.0, True),
    ((8, 8, 8), "most", 2.3, False),
    ((4, 4, 4), "full", 6.9, False),
    ((14, 12, 10), "ellipsoid", 6.9, False),
])
def test_the_inverse_is_computed_where_it_is_less_work(dims, kind, radius, built):
    info = _check(dims, kind, radius, (0.806, 0.2, 1.3))
    assert info["inverse_built"] == built
    assert (0 < info["n_inverse"] <= info["n_unique_solves"]) if built else info["n_inverse"] == 0


# largest diagonal entry of K^-1 and of 1 / L_ii^2, limit 1e4: indefinite; 1.0e6 and 7.4e5; 1.2e4 and 8.9e3
@pytest.mark.parametrize("theta,built", [((1.6, 0.05, 1.8), False), ((1.0 - 1e-6, 0.01, 2.0), False),
                                         ((1.0 - 8e-5, 0.02, 2.0), True)])
def test_no_system_goes_through_an_ill_conditioned_inverse(theta, built):
    from dualres_amd.kriging import kriging_build
    dims, radius = (16, 14, 12), 4.2
    hr, q, std, qs = _images(dims, _mask("most", dims))
    W, info = kriging_build(hr, q, std, qs, theta, radius, return_info=True)
    assert info["inverse_built"] == built and info["n_inverse"] == 0
    rp, cols, vals, *_ = okr.get_sparse_kriging_matrix_data(hr, std, q, qs, theta, radius)
    np.testing.assert_array_equal(W.indptr, rp)
    np.testing.assert_array_equal(W.indices, cols)
    _, P, _ = okr.kriging_pattern(hr, std, q, qs, theta, radius)
    if theta[0] < 1.0:
        # float64 solves of submatrices of K agree to n eps times its condition number
        K = okr.perturbation_kernel_distances(P, q, theta, dtype=np.float32).astype(np.float64)
        tol = len(P) * np.finfo(np.float64).eps * np.linalg.cond(K)
        assert np.linalg.norm(W.data - vals) <= tol * np.linalg.norm(vals)
    else:
        assert info["n_lu"] > 0


@pytest.mark.parametrize("dims,kind,radius", [((14, 12, 10), "ellipsoid", 6.9), ((14, 12, 10), "half", 4.2),
                                              ((8, 8, 8), "most", 2.3), ((4, 4, 4), "full", 6.9)])
def test_direct_weights_are_refined(dims, kind, radius):
    """As accurate as the weights that come through the inverse."""
    import scipy.linalg as sl
    from dualres_amd.kriging import kriging_build
    theta = (0.806, 0.132, 1.5)
    hr, q, std, qs = _images(dims, _mask(kind, dims))
    W, info = kriging_build(hr, q, std, qs, theta, radius, return_info=True)
    assert not info["inverse_built"]
    rows, P, _ = okr.kriging_pattern(hr, std, q, qs, theta, radius)
    K = okr.perturbation_kernel_distances(P, q, theta, dtype=np.float32).astype(np.float64)
    for i in range(0, len(rows), 3):
        _, pidx, kp = rows[i]
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

"""Kriging systems solved through the inverse of the ball's kernel matrix
against the oracle's direct solves, over masks whose rows lose from none to
most of the ball: whole tiles of absent offsets and remainders, systems with
more absent than present offsets (solved directly), and kernels for which
every system is solved directly."""
import numpy as np
import pytest

from dualres_amd import problem
from oracle import kriging as okr

pytestmark = pytest.mark.gpu


def _images(dims, mask, seed=2):
    rng = np.random.default_rng(seed)
    hr = np.where(mask, 1.0 + rng.random(mask.shape), 0.0)
    sd = tuple(d // 2 for d in dims)
    std = np.ones(sd[::-1])
    q = problem.qform_axis(1.0, dims)
    qs = problem.qform_axis(2.0, sd, origin=[q[a, 3] + 0.5 for a in range(3)])
    return hr, q, std, qs


def _mask(kind, dims):
    rng = np.random.default_rng(5)
    shape = dims[::-1]
    if kind == "full":
        return np.ones(shape, bool)
    if kind == "ellipsoid":
        return problem.ellipsoid_mask(dims, 0.4)
    return rng.random(shape) < {"most": 0.8, "half": 0.5, "few": 0.25}[kind]


def _check(dims, kind, radius, theta):
    from dualres_amd.kriging import kriging_build
    hr, q, std, qs = _images(dims, _mask(kind, dims))
    W, info = kriging_build(hr, q, std, qs, theta, radius, return_info=True)
    rp, cols, vals, nrow, ncol, _ = okr.get_sparse_kriging_matrix_data(hr, std, q, qs, theta, radius)
    assert W.shape == (nrow, ncol)
    np.testing.assert_array_equal(W.indptr, rp)
    np.testing.assert_array_equal(W.indices, cols)
    # both are float64 solves of systems with a condition number below 1e5
    assert np.linalg.norm(W.data - vals) <= 1e-10 * np.linalg.norm(vals)
    return info


@pytest.mark.parametrize("radius", [1.0, 2.3, 3.1, 4.2])  # balls of 7, 57, 147 and 341 offsets
@pytest.mark.parametrize("kind", ["full", "ellipsoid", "most", "half", "few"])
def test_weights_match_the_oracle(kind, radius):
    info = _check((14, 12, 10), kind, radius, (0.806, 0.2, 1.3))
    assert info["n_lu"] == 0


def test_indefinite_kernels_are_solved_directly():
    info = _check((10, 10, 8), "most", 2.3, (1.6, 0.05, 1.8))
    assert info["n_lu"] > 0


def test_nearly_singular_kernels_are_solved_directly():
    # 1 - tau^2 = 1e-6 bounds the diagonal of the inverse by 1e6: past the limit for the shared inverse
    from dualres_amd.kriging import kriging_build
    hr, q, std, qs = _images((10, 10, 8), _mask("most", (10, 10, 8)))
    W, info = kriging_build(hr, q, std, qs, (1.0 - 1e-6, 0.01, 1.9), 2.3, return_info=True)
    assert np.isfinite(W.data).all() and np.allclose(np.asarray(W.sum(axis=1)).ravel()[np.diff(W.indptr) > 0], 1.0)

"""W with what a CSR matrix may repeat, in the stencil layout against plain
CSR: rows with the same entries (several coarse voxels that map to one fine
voxel) and columns named twice in a row (a neighbourhood wider than the image
wraps onto itself), on both sides of the size from which W mu goes by stencil
lines."""
import numpy as np
import pytest
import scipy.sparse as sp

from helpers import rel
from test_gpu_w_lines import _gradient, _problem

pytestmark = pytest.mark.gpu

# the layouts differ in summation order alone: sums of up to 400 terms
TOL = {"fp64": 1e-13, "fp32": 1e-5}


def _compare(ijk, W, Yh, Ys, precision):
    (g0, s0), _ = _gradient(ijk, W, Yh, Ys, precision, True)
    (g1, s1), st = _gradient(ijk, W, Yh, Ys, precision, False)
    assert st["stencil_layout"] and st["interior_rows"] > 0
    assert rel(g1, g0) < TOL[precision] and abs(s1 - s0) < TOL[precision] * abs(s0)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims,step,reach,share,copies", [
    ((19, 14, 13), (2, 2, 2), (1, 2, 1), 1.0, 8),   # every row 8 times
    ((21, 15, 14), (1, 2, 2), (2, 1, 1), 0.3, 2),
    ((36, 20, 18), (5, 2, 2), (3, 2, 2), 0.3, 3),   # lattice step 5: the window table and tiles
    ((127, 61, 30), (2, 1, 2), (3, 2, 1), 0.1, 2),  # W mu by lines
])
def test_repeated_rows_match_csr(dims, step, reach, share, copies, precision):
    ijk, W, Yh, _ = _problem(dims, step, reach)
    rng = np.random.default_rng(11)
    at = np.repeat(np.arange(W.shape[0]), np.where(rng.random(W.shape[0]) < share, copies, 1))
    _compare(ijk, W[at], Yh, rng.standard_normal(len(at)), precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims,step,reach", [
    ((19, 14, 13), (2, 2, 2), (1, 2, 1)),
    ((36, 20, 18), (5, 2, 2), (3, 2, 2)),   # the window table and tiles
    ((127, 61, 30), (2, 1, 2), (3, 2, 1)),  # W mu by lines
])
def test_repeated_columns_match_csr(dims, step, reach, precision):
    """Every entry in two parts, as two entries of one column."""
    ijk, W, Yh, Ys = _problem(dims, step, reach)
    parts = np.stack([0.25 * W.data, 0.75 * W.data], axis=1).ravel()
    W2 = sp.csr_matrix((parts, np.repeat(W.indices, 2), 2 * W.indptr), shape=W.shape)
    assert W2.nnz == 2 * W.nnz
    _compare(ijk, W2, Yh, Ys, precision)

"""The interior W products by stencil lines against plain CSR: lattice steps
1 to 4 along x, lines of 1 to 4 chunks of taps, grids on both sides of the
size from which W mu takes the lines, and stencils the lines do not take."""
import numpy as np
import pytest
import scipy.sparse as sp

from helpers import rel

pytestmark = pytest.mark.gpu


def _problem(dims, step, reach, seed=4):
    """Rows on a lattice of the box with one translation-invariant stencil
    (a box of 2 reach + 1 voxels per axis, some entries missing), their own
    weights where it leaves the box."""
    rng = np.random.default_rng(seed)
    nx, ny, nz = dims
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    ijk = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1)
    r = [np.arange(-reach[a], reach[a] + 1) for a in range(3)]
    oz, oy, ox = np.meshgrid(r[2], r[1], r[0], indexing="ij")
    P = np.stack([ox.ravel(), oy.ravel(), oz.ravel()], axis=1)
    P = P[rng.random(len(P)) < 0.85]
    w = rng.standard_normal(len(P)) / len(P)
    cx, cy, cz = (np.arange(1, dims[a] - 1, step[a]) for a in range(3))
    c = np.stack([v.ravel() for v in np.meshgrid(cz, cy, cx, indexing="ij")][::-1], axis=1)
    at = c[:, None, :] + P[None]
    ok = ((at >= 0) & (at < np.array(dims))).all(axis=2)
    rows = np.broadcast_to(np.arange(len(c))[:, None], ok.shape)[ok]
    cols = (at[..., 0] + nx * (at[..., 1] + ny * at[..., 2]))[ok]
    vals = np.broadcast_to(w, ok.shape).copy()
    edge = ~ok.all(axis=1)
    vals[edge] *= 1.0 + rng.random((edge.sum(), 1))
    W = sp.csr_matrix((vals[ok], (rows, cols)), shape=(len(c), len(ijk)))
    W.sort_indices()
    return ijk, W, rng.standard_normal(len(ijk)), rng.standard_normal(len(c))


def _gradient(ijk, W, Yh, Ys, precision, csr):
    from dualres_amd import Chain
    emb = tuple(int(2 * (v + 1)) if (v + 1) % 2 == 0 else int(2 * (v + 2)) for v in ijk.max(0))
    emb = tuple(max(8, e) for e in emb)
    from dualres_amd.problem import smooth_even
    c = Chain(ijk, (0.8, 0.4, 1.0), np.diag([2.0, 2.0, 2.0, 1.0]).astype(np.float32), n_datasets=2,
              precision=precision, state_mode="real", embed=tuple(smooth_even(e) for e in emb), seed=9)
    c.w_layout(csr)
    c.set_data(Yh, Ys, W)
    c.add_data_to_mu()
    c.set_sigma_sq_inv([0.7, 3.0])
    st = c.w_stats()
    out = c.gradient().real, c.sse()[1]
    c.close()
    return out, st


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims,step,reach", [
    ((19, 14, 13), (2, 2, 2), (1, 2, 1)),
    ((21, 15, 14), (1, 2, 2), (2, 1, 1)),
    ((33, 14, 13), (3, 1, 2), (4, 2, 1)),
    ((41, 17, 12), (4, 2, 3), (7, 2, 1)),
    ((40, 13, 12), (1, 1, 2), (7, 1, 1)),
    ((36, 20, 18), (5, 2, 2), (3, 2, 2)),   # lattice step 5: the window table and tiles
    ((60, 13, 12), (2, 2, 2), (9, 1, 1)),   # 19 taps: the window table and tiles
    ((70, 42, 40), (1, 2, 2), (2, 2, 2)),   # enough items for W mu by lines
    ((127, 61, 30), (2, 1, 2), (3, 2, 1)),
])
def test_interior_products_match_csr(dims, step, reach, precision):
    p = _problem(dims, step, reach)
    (g0, s0), _ = _gradient(*p, precision, True)
    (g1, s1), st = _gradient(*p, precision, False)
    assert st["stencil_layout"] and st["interior_rows"] > 0
    # the two differ in summation order alone: sums of up to 400 terms
    tol = 1e-13 if precision == "fp64" else 1e-5
    assert rel(g1, g0) < tol and abs(s1 - s0) < tol * abs(s0)

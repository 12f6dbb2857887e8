"""The kernels that are chosen by size, each with the route it is meant to take:
the interior W products by stencil lines at every lattice step and length of
line against plain CSR, and single-resolution likelihoods by planes and by rows."""
import numpy as np
import pytest
import scipy.sparse as sp

from dualres_amd import Chain
from helpers import rel
from test_gpu_lines import LINES, TILES, TOL, _chain, _step
from test_gpu_w_lines import _problem

pytestmark = pytest.mark.gpu


def _run(ijk, W, Yh, Ys, embed, precision, csr):
    c = Chain(ijk, (0.8, 0.4, 1.0), np.diag([2.0, 2.0, 2.0, 1.0]).astype(np.float32), n_datasets=2,
              precision=precision, state_mode="real", embed=embed, seed=9)
    c.w_layout(csr)
    c.set_data(Yh, Ys, W)
    c.add_data_to_mu()
    c.set_sigma_sq_inv([0.7, 3.0])
    out = c.gradient().real, c.sse()[1], c.routes()
    c.close()
    return out


def _lattice(step, width, seed=6):
    """Rows every `step` voxels along x, 27 x 27 lines of them, with a stencil of `width` voxels along x, 3 along y and
    2 along z whose first entry is not its leftmost; rows whose stencil leaves the box keep what is inside."""
    rng = np.random.default_rng(seed)
    nx, ny, nz = 50 * step + 24, 29, 28
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    ijk = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1)
    left = (width - 1) // 2
    oz, oy, ox = np.meshgrid([0, 1], [-1, 0, 1], np.arange(-left, width - left), indexing="ij")
    P = np.stack([ox.ravel(), oy.ravel(), oz.ravel()], axis=1)
    if width > 1:
        P = P[1:]  # the first line starts one voxel further right
    w = rng.standard_normal(len(P)) / len(P)
    c = np.stack([v.ravel() for v in np.meshgrid(np.arange(27), np.arange(1, 28), np.arange(0, nx, step),
                                                 indexing="ij")][::-1], axis=1)
    at = c[:, None, :] + P[None]
    ok = ((at >= 0) & (at < np.array([nx, ny, nz]))).all(axis=2)
    W = sp.csr_matrix((np.broadcast_to(w, ok.shape)[ok], (at[..., 0] + nx * (at[..., 1] + ny * at[..., 2]))[ok],
                       np.concatenate([[0], np.cumsum(ok.sum(axis=1))])), shape=(len(c), len(ijk)))
    d = P[:, 0] - P[0, 0]  # from the first entry, a row's base
    t = -(d // step)
    return (ijk, W, rng.standard_normal(len(ijk)), rng.standard_normal(len(c))), (width - 1) // 4 + 1, \
        (t.max() - t.min()) // 4 + 1


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("step", [1, 2, 3, 4])
@pytest.mark.parametrize("width", [1, 4, 5, 8, 9, 12, 13, 16])  # remainders and whole chunks of 4 taps
def test_w_products_by_lines_match_csr(step, width, precision):
    problem, nc, mc = _lattice(step, width)
    emb = tuple({74: 160, 124: 250, 174: 350, 224: 450, 29: 60, 28: 56}[int(v) + 1] for v in problem[0].max(0))
    g0, s0, r0 = _run(*problem, emb, precision, True)
    g1, s1, r1 = _run(*problem, emb, precision, False)
    assert r0["w_mu_step"] == r0["wt_v_step"] == 0
    assert (r1["w_mu_step"], r1["w_mu_chunks"], r1["wt_v_step"], r1["wt_v_chunks"]) == (step, nc, step, mc)
    # the two differ in summation order alone: sums of up to 96 terms
    tol = 1e-13 if precision == "fp64" else 1e-5
    assert rel(g1, g0) < tol and abs(s1 - s0) < tol * abs(s0)


@pytest.mark.parametrize("dims,step,reach,mu,wt", [
    ((19, 14, 13), (2, 2, 2), (1, 2, 1), 0, 2),   # too few items for W mu by lines
    ((40, 13, 12), (1, 1, 2), (7, 1, 1), 0, 1),
    ((36, 20, 18), (5, 2, 2), (3, 2, 2), 0, 0),   # lattice step 5
    ((60, 13, 12), (2, 2, 2), (9, 1, 1), 0, 0),   # 19 taps
    ((70, 42, 40), (1, 2, 2), (2, 2, 2), 0, 1),   # 5,814 items
    ((127, 61, 30), (2, 1, 2), (3, 2, 1), 2, 2),  # 12,768
])
def test_w_routes_by_size(dims, step, reach, mu, wt):
    from dualres_amd.problem import smooth_even
    p = _problem(dims, step, reach)
    r = _run(*p, tuple(smooth_even(max(8, 2 * d)) for d in dims), "fp32", False)[2]
    assert (r["w_mu_step"], r["wt_v_step"]) == (mu, wt)


@pytest.mark.parametrize("region,embed,route", [
    ((2, 1, 3), (32, 32, 8), {"fp32": "planes", "fp64": "planes"}),
    ((17, 17, 3), (32, 32, 8), {"fp32": "planes", "fp64": "planes"}),
    ((33, 32, 2), (64, 64, 8), {"fp32": "planes", "fp64": "planes"}),
    ((16, 65, 2), (32, 128, 8), {"fp32": "planes", "fp64": "planes"}),
    ((64, 16, 2), (128, 32, 8), {"fp32": "planes", "fp64": "planes"}),
    ((47, 30, 3), (96, 64, 8), {"fp32": "planes", "fp64": "rows"}),    # M0 M1 past 4096
    ((32, 64, 3), (64, 128, 8), {"fp32": "planes", "fp64": "rows"}),
    ((47, 48, 2), (96, 96, 8), {"fp32": "rows", "fp64": "rows"}),      # past 8192
    ((20, 20, 3), (40, 40, 8), {"fp32": "rows", "fp64": "rows"}),      # no plane kernel for these lengths
    ((1, 12, 3), (32, 32, 8), {"fp32": "passes", "fp64": "passes"}),   # samples are fetched in pairs
    ((11, 5, 3), (600, 16, 8), {"fp32": "passes", "fp64": "passes"}),  # no line kernel for 600
])
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_likelihood_routes_match_tiles(region, embed, route, precision):
    got = []
    for tuning, want in ((LINES, route[precision]), (TILES, "passes")):
        c = _chain(embed, region, precision, "compat", False)
        assert c.routes()["likelihood"] is None
        got.append(_step(c, tuning))
        assert c.routes()["likelihood"] == want
        c.close()
    for a, b in zip(*got):
        assert rel(a, b) < TOL[precision], (embed, region, precision)

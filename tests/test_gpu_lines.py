"""The register line transforms of a leapfrog step (dr_lines.hpp) against the
tile kernels of dr_fft.hpp, which hand-set tile lines select, at every length
a plan exists for, on each axis, and against the oracle."""
import numpy as np
import pytest

from helpers import rel

pytestmark = pytest.mark.gpu

LENGTHS = [m for m in range(8, 513, 2) if 2 ** 20 * 3 ** 12 * 5 ** 8 * 7 ** 8 % m == 0]
TILES = [0, 0, 0, 0, 0, 0, 0, 0]  # two-line tiles in every pass
LINES = [-1, -1, -1, -1, -1, 0, 0, 0]
# a transform of N <= 512 * 80 points is off by about eps log2(N); three
# gradients and two steps multiply that by less than 10
TOL = {"fp64": 1e-12, "fp32": 1e-4}


def _chain(embed, region, precision, state, dual, seed=3):
    import scipy.sparse as sp

    from dualres_amd import Chain
    rng = np.random.default_rng(seed)
    n0, n1, n2 = region
    z, y, x = np.meshgrid(np.arange(n2), np.arange(n1), np.arange(n0), indexing="ij")
    ijk = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1)
    keep = rng.random(len(ijk)) < 0.7
    keep[0] = keep[-1] = True
    ijk = ijk[keep]
    q = np.diag([2.0, 2.0, 2.0, 1.0]).astype(np.float32)
    c = Chain(ijk, (0.8, 0.3, 1.2), q, n_datasets=2 if dual else 1, precision=precision, state_mode=state,
              embed=embed, seed=seed)
    Y = rng.standard_normal(len(ijk))
    if dual:
        W = sp.random(9, len(ijk), density=0.3, random_state=5, format="csr")
        c.set_data(Y, rng.standard_normal(9), W)
    else:
        c.set_data(Y)
    c.add_data_to_mu()
    c.set_sigma_sq_inv([1.3, 2.1][:c.n_datasets])
    return c


def _step(c, tuning, eps=0.1):
    c.set_tuning(tuning)
    r = c.update(eps, 2, 0.0)
    mu, p = c.get_state()
    return np.array([r[k] for k in ("log_prior0", "log_lik0", "log_prior1", "log_lik1", "k1", "sse_h")]), mu.real, p.real, c.mu_()


def _compare(embed, region, precision, state, dual):
    got = []
    for t in (LINES, TILES):
        c = _chain(embed, region, precision, state, dual)
        got.append(_step(c, t))
        c.close()
    for a, b in zip(*got):
        assert rel(a, b) < TOL[precision], (embed, region, precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_every_length_matches_the_tile_kernels(axis, precision):
    for i, m in enumerate(LENGTHS):
        embed, region = [10, 8, 8], [4 + i % 2, 3, 4]
        embed[axis] = m
        region[axis] = min(m // 2 + 1, (m * (3 + i % 3)) // 10 + 2)  # odd and even, short of and up to the half
        _compare(tuple(embed), tuple(region), precision, "compat" if i % 2 else "real", False)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_dual_resolution_matches_the_tile_kernels(precision):
    for embed, region in (((10, 14, 16), (2, 5, 3)), ((40, 36, 60), (17, 15, 27)), ((56, 98, 50), (28, 40, 25)),
                          ((64, 90, 126), (33, 41, 60))):
        _compare(embed, region, precision, "compat", True)


def test_one_voxel_rows_keep_the_tile_kernels():
    _compare((8, 12, 10), (1, 5, 4), "fp64", "compat", False)


def test_lengths_without_a_plan_keep_the_tile_kernels():
    _compare((540, 8, 10), (20, 3, 4), "fp64", "real", False)
    _compare((8, 4, 600), (4, 2, 100), "fp32", "real", False)

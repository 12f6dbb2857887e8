"""The pruned correlation transforms of the minimum-contrast summaries against
direct sums over voxel pairs: images shorter than the offsets' reach on some
axes (every row of the torus is then kept), odd sizes, missing voxels (0 and
NaN), and an axis past the line kernels' lengths."""
import numpy as np
import pytest

from dualres_amd import mce, problem

pytestmark = pytest.mark.gpu


def _image(dims, seed):
    rng = np.random.default_rng(seed)
    img = rng.standard_normal(dims[::-1])
    img[rng.random(img.shape) < 0.3] = 0.0
    img[rng.random(img.shape) < 0.05] = np.nan
    return img


def _direct(img, p):
    """Sums over the pairs (u, u + p) present in the image."""
    x, y, z = p
    nz, ny, nx = img.shape

    def cut(n, d):
        return slice(max(0, -d), min(n, n - d)), slice(max(0, d), min(n, n + d))
    (az, bz), (ay, by), (ax, bx) = cut(nz, z), cut(ny, y), cut(nx, x)
    if abs(x) >= nx or abs(y) >= ny or abs(z) >= nz:
        return 0.0, 0.0, 0.0, 0
    a, b = img[az, ay, ax], img[bz, by, bx]
    ok = ~(np.isnan(a) | np.isnan(b) | (a == 0) | (b == 0))
    a, b = a[ok], b[ok]
    return float(np.sum(a * b)), float(a.sum()), float(b.sum()), int(ok.sum())


@pytest.mark.parametrize("dims", [(6, 7, 5), (31, 29, 8), (30, 26, 40), (3, 50, 27), (1, 1, 9), (500, 4, 3)])
def test_summary_matches_direct_sums(dims):
    img = _image(dims, 3)
    q = problem.qform_axis(1.5, dims)
    cov, dist, npairs = mce.mce_summary(img, q)
    off = mce.mce_offsets()
    inside = (np.abs(off) < np.array(dims)).all(axis=1)
    assert (npairs[~inside] == 0).all()
    pick = np.flatnonzero(inside)
    pick = pick[np.random.default_rng(1).permutation(len(pick))[:300]]
    for i in pick:
        sxy, sx, sy, n = _direct(img, off[i])
        assert npairs[i] == n
        want = (sxy - sx * sy / n) / (n - 1) if n > 1 else 0.0
        # float64 sums of at most 1e4 terms of order 1, returned in float32
        assert abs(cov[i] - want) <= 1e-6 * max(1.0, abs(want))


@pytest.mark.parametrize("dims,maxdist", [((20, 17, 14), 9.0), ((9, 30, 5), 12.0), ((600, 3, 3), 4.0)])
def test_binned_matches_direct_sums(dims, maxdist):
    img = _image(dims, 5)
    cov, dist, n = mce.mce_binned(img, problem.qform_axis(1.0, dims), nbins=6, maxdist=maxdist)
    S = np.zeros((6, 4))
    r = int(np.ceil(maxdist))
    for z in range(0, r + 1):
        for y in range(-r, r + 1):
            for x in range(-r, r + 1):
                if z == 0 and (y < 0 or (y == 0 and x < 0)):
                    continue
                d = np.sqrt(np.float32(x * x + y * y + z * z))
                if d <= maxdist:
                    S[min(5, int(d / (maxdist / 6)))] += _direct(img, (x, y, z))
    np.testing.assert_array_equal(n, S[:, 3].astype(np.int64))
    ok = n > 1
    want = (S[ok, 0] - S[ok, 1] * S[ok, 2] / n[ok]) / (n[ok] - 1)
    np.testing.assert_allclose(cov[ok], want, rtol=0, atol=1e-11)

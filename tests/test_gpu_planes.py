"""Single-resolution likelihoods by whole planes (k_plane) against the tile kernels, which
hand-set tile lines select, at the edges of the plane kernel's range: the smallest and
largest tori, one data row, regions of half the torus and one row more, odd rows, and
lengths of three times a power of two.  Bounds as for the separate line passes."""
import pytest

from helpers import rel
from test_gpu_lines import LINES, TILES, TOL, _chain, _step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("region,embed", [
    ((2, 1, 3), (32, 32, 8)), ((16, 16, 4), (32, 32, 8)), ((17, 17, 3), (32, 32, 8)), ((13, 31, 2), (48, 64, 10)),
    ((31, 24, 3), (64, 48, 16)), ((33, 32, 2), (64, 64, 8)), ((47, 9, 3), (96, 32, 12)), ((16, 48, 3), (32, 96, 8)),
    ((16, 65, 2), (32, 128, 8)), ((64, 16, 2), (128, 32, 8)), ((32, 64, 3), (64, 128, 8)),
    ((64, 31, 2), (128, 64, 8)),
])
def test_planes_against_tiles(region, embed, precision):
    got = []
    for tuning in (LINES, TILES):
        c = _chain(embed, region, precision, "compat", False)
        got.append(_step(c, tuning))
        c.close()
    for a, b in zip(*got):
        assert rel(a, b) < TOL[precision], (embed, region, precision)

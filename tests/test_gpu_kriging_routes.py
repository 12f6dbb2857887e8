"""How the kriging systems are worked on, with the weights against the oracle."""
import numpy as np
import pytest

from test_gpu_kriging_inverse import _check

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

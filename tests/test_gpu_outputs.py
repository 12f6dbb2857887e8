"""Reading the data voxels leaves the output voxels' buffer alone."""
import numpy as np
import pytest

from test_gpu_lines import _chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_data_voxels_read_between_output_voxels(precision):
    region = (12, 10, 9)
    c = _chain((24, 20, 18), region, precision, "compat", False)
    z, y, x = np.meshgrid(*(np.arange(n) for n in region[::-1]), indexing="ij")
    every = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1)  # more outputs than data
    c.set_output_indices(every)
    c.update(0.1, 2, 0.0)
    out, data = c.mu_(), c.mu()
    assert out.size == len(every) > data.size
    c.summary_update()
    again = c.mu_()
    assert np.array_equal(out, again) and np.array_equal(data, c.mu())
    assert np.array_equal(c.summary_read()[0], out)
    at = c._ijk @ np.array([1, region[0], region[0] * region[1]])
    assert np.array_equal(out[at], data)
    c.close()

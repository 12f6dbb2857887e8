"""Chains created in memory that held NaN: the columns that pad the last block of
the spectral state stay 0, with ragged and whole last blocks."""
import numpy as np
import pytest
import torch

from test_gpu_lines import LINES, TILES, _chain, _step

pytestmark = pytest.mark.gpu


def _results(embed, precision, state, tuning):
    c = _chain(embed, tuple(e // 2 for e in embed), precision, state, False)
    out = _step(c, tuning)
    out += (c.gradient(), np.array([c.log_prior(), c.log_likelihood()]), c.lambda_())
    c.set_tau_sq_inv(1.7)
    out += (np.array([c.update(0.1, 2, 0.0)[k] for k in ("H0", "H1")]), c.mu_())
    c.close()
    return out


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("state", ["compat", "real"])
@pytest.mark.parametrize("embed", [(20, 18, 16), (30, 32, 10), (24, 16, 12)])  # 198, 512 and 208 columns
@pytest.mark.parametrize("tuning", [LINES, TILES])
def test_padding_is_zero_whatever_the_memory_held(embed, state, precision, tuning):
    clean = _results(embed, precision, state, tuning)
    blocks = [torch.full((n,), float("nan"), device="cuda") for n in 32 * [1 << 18]]
    torch.cuda.synchronize()
    del blocks
    torch.cuda.empty_cache()  # given back to the driver, where the chain's arrays come from
    for a, b in zip(clean, _results(embed, precision, state, tuning)):
        assert np.isfinite(a).all() and np.array_equal(a, b)

"""The autotuner and the register line kernels: choices timed before those
kernels were built are not taken over, and a search finds its way back to them."""
import json

import numpy as np
import pytest

from helpers import engine_chain, small_single

pytestmark = pytest.mark.gpu

THETA = (0.806, 0.132, 1.0)
EMBED = (64, 64, 32)
TILES = [0, 0, 0, 0, 0, 1, 1, 1]


def _chain():
    p = small_single(dims=(30, 28, 14))
    return engine_chain(p, THETA, precision="fp32", embed=EMBED, seed=4)


def test_entries_of_the_tile_kernels_are_not_taken(tmp_path):
    cache = tmp_path / "tune.json"
    c = _chain()
    _, hit = c.autotune(cache)
    assert not hit
    (key,) = json.loads(cache.read_text())
    # the key was device, precision, state, datasets, torus and region alone
    old = "|".join(key.split("|")[:6])
    other = tmp_path / "old.json"
    other.write_text(json.dumps({old: TILES}))
    prm, hit = c.autotune(other)
    assert not hit
    entries = json.loads(other.read_text())
    assert entries[old] == TILES and entries[key] == prm  # kept for an engine that still reads it
    c.close()


def test_a_search_from_hand_set_tiles_reaches_the_lines():
    """Two-line tiles are several times slower than the lines on this torus, so
    a search that can pick the lines does."""
    c = _chain()
    c.set_tuning(TILES)
    prm, _ = c.autotune()
    assert prm[0] == -1 and c.tuning() == prm
    c.close()

"""The tile height of float64 domains: its rule, the count it is fed with, and that both mesh builders
take it."""
import numpy as np
import pytest

import geoswe_amd.flatmesh as FM


def test_rule():
    want = {0: 1, 999: 1, 1000: 2, 6000: 2, 6001: 3, 9000: 3, 24001: 9, 27000: 9}
    assert {b: FM.sweep_rows_for64(b) for b in want} == want
    for busy in (27001, 60000, 10 ** 6, 10 ** 9):
        assert FM.sweep_rows_for64(busy) == FM.sweep_rows_for(busy)


@pytest.mark.parametrize("shape", [(9, 5), (9, 66), (30, 128), (41, 185), (12, 63), (12, 64)])
def test_window_rows(shape):
    """As many as there are (row, window) pairs with an active lane among the written ones."""
    rng = np.random.default_rng(shape[1])
    inside = np.zeros(shape, bool)
    inside[2:-2, 2:-2] = rng.random((shape[0] - 4, shape[1] - 4)) < 0.05
    want = sum(bool(inside[i, 60 * w + 2:60 * w + 62].any()) for i in range(shape[0]) for w in range(shape[1] // 60 + 1))
    assert FM.window_rows(inside) == want
    assert FM.window_rows(np.zeros(shape, bool)) == 0


@pytest.mark.parametrize("native", [True, False])
def test_both_builders(native):
    inside = np.zeros((1008, 488), bool)
    inside[4:-4, 4:-4] = True
    busy = FM.window_rows(inside)
    rows = FM.sweep_rows_for64(busy)
    assert rows == 3 and busy == 9000 and FM.sweep_rows_for(busy) == 1
    a = FM.build_flat_mesh(inside, 4, native=native, dtype=np.float64)
    b = FM.build_flat_mesh(inside, 4, native=native, sweep_rows=rows)
    assert np.array_equal(a.tile_irc, b.tile_irc) and np.array_equal(a.ent, b.ent)
    c = FM.build_flat_mesh(inside, 4, native=native, sweep_rows=1, dtype=np.float64)
    assert int(c.tile_irc[:, 1].max()) == 1

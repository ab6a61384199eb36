"""The incremental re-sort at the edges of its tiles (256 slots a block up to
65,536 slots, 512 beyond): order and cell table against the oracle's stable
sort after every step, with few and with most keys changed."""
import numpy as np
import pytest

import bdem
from bdem import scenarios as S
from helpers import make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vmax", [400.0, 2.0e5])
@pytest.mark.parametrize("n", [1, 255, 256, 257, 1025, 65536, 65537])
def test_order_and_cells_at_tile_edges(n, vmax):
    print(f"[case] n={n} vmax={vmax}", flush=True)
    deck = S.random_deck(n, seed=n % 89 + 2, L=2.0 + n ** (1.0 / 3.0), radius=0.3, vmax=vmax)
    dev, ora = make_pair(deck)
    try:
        for step in range(3):
            dev.step(1)
            ora.step(1)
            kg, ig = dev.debug_sorted()
            ko, io = ora.sorted()
            assert np.array_equal(kg, ko) and np.array_equal(ig, io), f"step {step}: order"
            dev.step(1)
            ora.step(1)
            sg, eg = dev.debug_cells()
            so, eo = ora.cells()
            assert np.array_equal(sg, so) and np.array_equal(eg, eo), f"step {step}: cells"
        assert not dev.status() & bdem.lib.WARN_SORT
    finally:
        dev.close()
        ora.close()

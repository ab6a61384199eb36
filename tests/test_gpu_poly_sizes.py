"""Polyhedra steps at the sizes where the contact list changes form (24,576
particles) and at the remainders of its blocks, against the FP32
restatement: a few steps, states within the build's 1e-5 bar (bit-equal away
from the quaternion's sine and cosine)."""
import numpy as np
import pytest

from bdem import scenarios as S
from helpers import by_pid, make_pair, oracle_positions_out, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,shape,spacing", [
    (1, "hull", 0.85), (15, "hull", 0.85), (17, "mixed", 1.1), (129, "cubes2", 1.1), (2000, "hull", 0.5),
    (24576, "hull", 0.85), (24577, "hull", 0.8), (25001, "mixed", 1.1), (26000, "hull", 0.6)])
def test_states_at_list_edges(n, shape, spacing):
    print(f"[case] n={n} {shape} spacing={spacing}", flush=True)
    L = int(np.ceil(n ** (1.0 / 3.0))) * spacing + 3.2
    deck = S.poly_deck(n, seed=n % 83 + 2, L=L, shape=shape, size=1.0, spacing=spacing, vmax=10.0, wmax=5.0)
    dev, ora = make_pair(deck)
    try:
        dev.step(2)
        ora.step(2)
        g, o = by_pid(dev.get_state()), by_pid(ora.state())
        assert np.array_equal(g["pid"], o["pid"])
        for k, ref in (("pos", oracle_positions_out(deck, o)), ("vel", o["vel"]), ("avel", o["avel"]),
                       ("quat", o["quat"])):
            scale = max(float(np.max(np.abs(ref))), 1e-30)
            assert rel_err(g[k], ref, 1e-3 * scale) <= 1e-5, k
    finally:
        dev.close()
        ora.close()

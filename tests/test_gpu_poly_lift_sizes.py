"""Polyhedra against turning lifters on both sides of the count where the
lifter kernel takes more hulls per wave (16,384), and at the remainders of
its blocks, against the FP32 restatement.  Tolerance as in the other
polyhedra tests."""
import numpy as np
import pytest

from bdem import scenarios as S
from helpers import by_pid, make_pair, oracle_positions_out, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [97, 16384, 16385, 16391])
def test_lifter_forces_at_wave_edges(n):
    print(f"[case] poly mill {n}", flush=True)
    kw = dict(R=40.0, L=40.0, lifter_w=3.0, lifter_h=3.0) if n > 1000 else {}
    deck = S.poly_mill_deck(n, **kw)
    dev, ora = make_pair(deck)
    try:
        dev.drum_rotation(True)
        ora.set_drum_rotation(True)
        dev.set_lifter_rotation(deck["rad_per_step"], deck["lifter_about"])
        dev.step(3)
        ora.run(3, deck["rad_per_step"], deck["lifter_about"])
        assert ora.lifter_contacts() > 0
        g, o = by_pid(dev.get_state()), by_pid(ora.state())
        assert np.array_equal(g["pid"], o["pid"])
        for k, ref in (("pos", oracle_positions_out(deck, o)), ("vel", o["vel"]), ("avel", o["avel"]),
                       ("quat", o["quat"])):
            scale = max(float(np.max(np.abs(ref))), 1e-30)
            assert rel_err(g[k], ref, 1e-3 * scale) <= 1e-5, k
    finally:
        dev.close()
        ora.close()

"""Polyhedra on a capped cylinder followed by an infinite plane, against the
FP32 restatement.  The plane has no method of its own for polyhedra: it acts
with the result of the wall tested before it, which for a capped cylinder is
that of its last cap, also where the body is far from the caps."""
import numpy as np
import pytest

from bdem import scenarios as S
from helpers import by_pid, make_pair, oracle_positions_out, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("top,bot", [(False, False), (True, False), (False, True), (True, True)])
def test_plane_after_a_capped_cylinder(top, bot):
    print(f"[case] caps top={top} bot={bot}", flush=True)
    R, L, n = 15.0, 10.0, 300
    deck = S.poly_mill_deck(n, R=R, L=L)
    rb = deck["pobj"][0].radius
    a = S.uniform(7, 11, n, 0.0, 2.0 * np.pi)
    r = R - rb * S.uniform(7, 12, n, 0.3, 1.1)
    z = S.uniform(7, 13, n, 0.4 * rb, L - 0.4 * rb)
    deck["pos"] = np.stack([R + r * np.cos(a), R + r * np.sin(a), z], 1).astype(np.float32)
    deck["dobj"] = None
    deck["wobj"] = [S.cylinder_wobj(R, L, (0.0, 0.0, 1.0), (0.0, 0.0, 0.0), top=top, bot=bot),
                    S.infinite_plane_wobj((R, 1.0, 0.0), (0.0, 1.0, 0.0))]
    dev, ora = make_pair(deck)
    try:
        g, o = dev.debug_forces(), ora.forces()
        assert np.array_equal(g[4], o[4])
        touching = np.abs(o[2]).max(1) > 0
        clear = (z > 1.2 * rb) & (z < L - 1.2 * rb)   # by P_ID
        assert (touching & clear[o[4]]).sum() > 30
        for q, what in ((2, "F_wall"), (3, "T_wall")):
            scale = max(float(np.max(np.abs(o[q]))), 1e-30)
            assert rel_err(g[q], o[q], 1e-3 * scale) <= 1e-5, what
        dev.step(5)
        ora.step(5)
        sg, so = by_pid(dev.get_state()), by_pid(ora.state())
        for k, ref in (("pos", oracle_positions_out(deck, so)), ("vel", so["vel"]), ("avel", so["avel"])):
            scale = max(float(np.max(np.abs(ref))), 1e-30)
            assert rel_err(sg[k], ref, 1e-3 * scale) <= 1e-5, k
    finally:
        dev.close()
        ora.close()

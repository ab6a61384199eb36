"""The sphere step's team shapes against the FP32 restatement at the sizes
where they change: one particle, blocks of 16 and 32 and their remainders,
the last size of each shape and the first of the next, and packs whose
particles have more contacts than the kernel lists (12) and more stencil
candidates than it lists at a time (64)."""
import numpy as np
import pytest

from bdem import scenarios as S
from helpers import make_pair, by_pid

pytestmark = pytest.mark.gpu


# n, law, spheres per cm^3 (1.5: about 6 contacts; 5: about 20, 135 candidates)
@pytest.mark.parametrize("n,law,density", [
    (1, "ref", 1.5), (16, "hm", 1.5), (17, "lsd", 1.5), (31, "ref", 1.5), (33, "hm", 5.0), (1000, "hm", 5.0),
    (19648, "hm", 1.5), (19649, "lsd", 1.5), (20000, "hm", 5.0), (39296, "lsd", 1.5), (39297, "ref", 1.5),
    (45001, "hm", 5.0), (131072, "hm", 1.5), (131073, "ref", 1.5)])
def test_states_equal_the_oracle_at_shape_edges(n, law, density):
    print(f"[case] n={n} law={law} density={density}", flush=True)
    L = 1.2 + max((n / density) ** (1.0 / 3.0), 0.5)
    deck = S.random_deck(n, seed=n % 97 + 3, L=L, law=law)
    dev, ora = make_pair(deck)
    try:
        # three steps: the same float operations in the same order, so the
        # states are equal to the last bit (springs carried over twice)
        dev.step(3)
        ora.step(3)
        g, o = by_pid(dev.get_state()), by_pid(ora.state())
        for k in ("pid", "pos", "vel", "avel"):
            assert np.array_equal(g[k], np.asarray(o[k], g[k].dtype)), k
    finally:
        dev.close()
        ora.close()


def test_step_contact_lists_past_the_listed_ones():
    """The contacts the step kernel used, with up to 32 listed."""
    deck = S.random_deck(2000, seed=5, L=1.2 + (2000 / 4.0) ** (1.0 / 3.0), law="lsd")
    dev, ora = make_pair(deck)
    try:
        lo, no = ora.contacts()
        assert no.max() > 12
        lg, ng = dev.debug_step_contacts()
        assert np.array_equal(ng, no)
        for i in np.nonzero(no)[0]:
            k = min(int(no[i]), 32)
            assert np.array_equal(lg[i, :k], lo[i, :k]), f"particle {i}"
    finally:
        dev.close()
        ora.close()

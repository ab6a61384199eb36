"""Polyhedra in grids whose lists are not the same from both bodies of a
contact, against the FP32 restatement, which computes every listed entry on
its own: more z than x cells (hulls whose hash passes the cell table list
their neighbours and are not listed back, and rows that end past it are
dropped), grids two or three cells thin (two rows of a stencil share cells,
and a partner is listed twice), hulls outside the grid, and packs whose lists
overflow.  Both list kernels (24,577 hulls and more take the second).  Forces
and states within the build's 1e-5 bar (bit-equal away from the quaternion's
sine and cosine)."""
import numpy as np
import pytest

import bdem
from bdem import scenarios as S
from bdem import types as T
from helpers import by_pid, make_pair, oracle_positions_out, rel_err

pytestmark = pytest.mark.gpu


def grid_deck(cells, n=None, outside=0, spacing=0.55, seed=61):
    """Hulls on a jittered lattice through a grid of exactly `cells` cells
    (edge 2 x the bounding radius), `outside` of them moved up to half a cell
    past its ends.  They overlap deeply; steps of 1e-6 s keep the speeds near
    those of the other decks (at 1e-5 s they reach 2,900 cm/s in 20 steps, and
    last-bit differences of the quaternion's sine grow with the pack's)."""
    m = np.array([max(int(c / spacing), 1) for c in cells])
    n = int(m.prod()) if n is None else n
    assert n <= m.prod()
    deck = S.poly_deck(n, seed=seed, L=3.2 + 1.1 * np.ceil(n ** (1.0 / 3.0)), shape="hull", size=1.7,
                       spacing=1.0, dt=1e-6)
    sim = deck["sim"]
    c = sim.cellSize.x
    gi = np.indices(m).reshape(3, -1).T[:n].astype(np.float64)
    pos = (gi + 0.5) * (np.array(cells) * c / m)
    pos += S.uniform(seed, 91, 3 * n, -0.05 * c, 0.05 * c).reshape(n, 3)
    rng = np.random.RandomState(seed)
    for k in range(outside):
        i, ax = rng.randint(n), rng.randint(3)
        pos[i, ax] = rng.choice([-1.0, 1.0]) * rng.uniform(0.05, 0.45) * c + rng.choice([0.0, cells[ax] * c])
    deck["pos"] = np.ascontiguousarray(pos, np.float32)
    sim.worldOrigin = T.f3(0.0, 0.0, 0.0)
    sim.num_NNCells = T.Int3(*[int(x) for x in cells])
    sim.max_size = T.f3(*[x * c for x in cells])
    deck["wobj"] = [S.box_walls(float(max(cells) * c) + 1.0)]
    return deck


def unmatched(lists, counts):
    """Entries without a counterpart in the partner's list, and repeated ones."""
    one, twice = 0, 0
    rows = [list(lists[i, :min(int(counts[i]), 32)]) for i in range(len(counts))]
    for i, r in enumerate(rows):
        for j in set(r):
            one += max(r.count(j) - rows[j].count(i), 0)
            twice += r.count(j) - 1
    return one, twice


CASES = [((4, 4, 7), None, 0), ((2, 2, 5), None, 0), ((4, 4, 2), None, 0), ((2, 4, 4), None, 0), ((3, 3, 3), None, 0),
         ((5, 2, 6), None, 0), ((6, 5, 1), None, 0), ((1, 6, 6), None, 0), ((5, 5, 5), None, 24), ((4, 4, 7), None, 24),
         ((10, 10, 42), 24576, 40), ((10, 10, 42), 24577, 40), ((70, 60, 2), 26000, 0)]
CASES = [c + (0.55,) for c in CASES] + [((6, 6, 6), None, 0, 0.45), ((4, 4, 7), None, 8, 0.45), ((13, 13, 16), None, 0, 0.45)]


@pytest.mark.parametrize("cells,n,outside,spacing", CASES)
def test_forces_and_states_equal_the_oracle(cells, n, outside, spacing):
    print(f"[case] grid {cells} n={n} outside={outside} spacing={spacing}", flush=True)
    deck = grid_deck(cells, n, outside, spacing)
    dev, ora = make_pair(deck)
    try:
        lo, no = ora.contacts()
        one, twice = unmatched(lo, no)
        assert one + twice > 0 or cells in ((3, 3, 3), (6, 5, 1))
        assert spacing > 0.5 or no.max() > 32
        lg, ng = dev.debug_contacts()
        assert np.array_equal(ng, no)
        for i in np.nonzero(no)[0]:
            k = min(int(no[i]), 32)
            assert np.array_equal(lg[i, :k], lo[i, :k]), f"particle {i}"
        g, o = dev.debug_forces(), ora.forces()
        assert np.array_equal(g[4], o[4])
        for a, b, what in zip(g[:4], o[:4], ("F_pp", "T_pp", "F_wall", "T_wall")):
            scale = max(float(np.max(np.abs(b))), 1e-30)
            assert rel_err(a, b, 1e-3 * scale) <= 1e-5, what
        steps = 20 if len(deck["pos"]) < 10000 else 3
        dev.step(steps)
        ora.step(steps)
        sg, so = by_pid(dev.get_state()), by_pid(ora.state())
        assert np.array_equal(sg["pid"], so["pid"])
        so["pos"] = oracle_positions_out(deck, so)
        for k in ("pos", "vel", "avel", "quat"):
            scale = max(float(np.max(np.abs(so[k]))), 1e-30)
            assert rel_err(sg[k], so[k], 1e-3 * scale) <= 1e-5, k
        assert not dev.status() & bdem.lib.WARN_SORT
    finally:
        dev.close()
        ora.close()

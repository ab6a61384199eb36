"""hash_is_local, the rule by which the polyhedra step takes most contacts
from one body's list only, against the restatement's contact lists: where it
holds, no partner is listed twice, and an entry that the partner's list lacks
belongs to the lower sorted slot or to a particle whose key is in the cell
table's last two or past it.  Grids of every aspect from one cell up, cells
from half to twice the particles' diameter, particles outside the grid."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from bdem import scenarios as S
from bdem import types as T
from oracle_py import Oracle

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(S.__file__))), "csrc")


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("grid")
    (d / "g.cpp").write_text('#include "bdem_grid.hpp"\n'
                             'extern "C" int local_(int x, int y, int z, float r, float cx, float cy, float cz) {\n'
                             '  return bdem::hash_is_local(x, y, z, bdem::contact_reach(r, cx, cy, cz)); }\n')
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "g.cpp"), "-o",
                    str(d / "g.so")], check=True)
    f = C.CDLL(str(d / "g.so")).local_
    f.argtypes = [C.c_int] * 3 + [C.c_float] * 4
    return lambda cells, r, cell: bool(f(*[int(x) for x in cells], r, *cell))


def _pack(rng, cells, cell, r, n):
    """n overlapping spheres through the grid and a little past its ends."""
    deck = S.random_deck(n, seed=int(rng.randint(1 << 30)), L=8.0, radius=r)
    hi = np.array(cells) * np.array(cell)
    deck["pos"] = (rng.uniform(-0.3, 1.0, (n, 3)) * 0.6 + rng.uniform(0.0, 1.0, (n, 3)) * hi).astype(np.float32)
    sim = deck["sim"]
    sim.worldOrigin = T.f3(0.0, 0.0, 0.0)
    sim.cellSize = T.f3(*[float(c) for c in cell])
    sim.num_NNCells = T.Int3(*[int(c) for c in cells])
    sim.max_size = T.f3(*hi)
    return deck


def _lists(deck):
    ora = Oracle(deck)
    try:
        keys, _ = ora.sorted()
        lists, nn = ora.contacts()
    finally:
        ora.close()
    return keys, [list(lists[i, :int(nn[i])]) for i in range(len(nn))], int(nn.max())


def test_lists_agree_where_the_hash_is_local(rule):
    rng = np.random.RandomState(5)
    held = broken = 0
    for trial in range(700):
        cells = np.exp(rng.uniform(0.0, np.log(13.0), 3)).astype(int)
        r = 0.5
        cell = rng.choice([0.5, 0.9, 1.0, 1.0, 1.0, 1.3, 2.0]) * np.ones(3) + (rng.rand(3) < 0.2) * 0.37
        vol = float(np.prod(np.array(cells) * cell))
        keys, lists, most = _lists(_pack(rng, cells, cell, r, int(min(max(3.0 * vol, 8), 700))))
        if most > 32:
            continue
        last = int(np.prod(cells)) - 2
        ok = rule(cells, r, cell)
        bad = 0
        for i, row in enumerate(lists):
            bad += len(row) - len(set(row))
            if int(keys[i]) < last:
                bad += sum(1 for j in row if j < i and i not in lists[j])
        assert not (ok and bad), (cells, cell, bad)
        held += ok
        broken += bad > 0
    assert held > 100 and broken > 50


def test_usual_grids_hold(rule):
    for cells in ((10, 10, 10), (17, 17, 19), (19, 19, 7), (4, 4, 4), (64, 8, 64), (9, 40, 100), (100, 40, 9)):
        assert rule(cells, 0.5, (1.0, 1.0, 1.0)), cells
    for cells in ((4, 4, 2), (2, 4, 4), (4, 4, 3), (3, 4, 4)):
        assert not rule(cells, 0.5, (1.0, 1.0, 1.0)), cells
    assert not rule((50, 50, 50), float("inf"), (1.0, 1.0, 1.0))
    assert not rule((50, 50, 50), 0.5, (0.01, 1.0, 1.0))

"""The forms of the sphere step that the packs at the shapes' edges do not
take, in each of its kernels, against the FP32 restatement: orientations,
dissipation tallies, lifters and recorded wall forces together, discharge,
grids with fewer and with more z than x cells, contacts past the listed
twelve, and pairs that touch to within the float's last places.  20,001
spheres are stepped by teams of eight lanes, 45,001 by teams of four, more
than 131,072 by a lane each; a batch of more than 131,072 slots on the plain
grid by the batch's own lane kernel.

States are equal to the last bit (quaternions within 1e-5: device and host
sine differ).  Tallies are float sums of some N = 4e5 positive increments in
another order: at most N 2^-25 = 1.2e-2 apart in the worst case, as a random
walk of roundings about 1e-5; 1e-3 is asked for."""
import ctypes as C

import numpy as np
import pytest

import bdem
from bdem import scenarios as S
from bdem import types as T
from helpers import by_pid, make_device, make_pair, rel_err

pytestmark = pytest.mark.gpu

TEAM8, TEAM4, LANE = 20001, 45001, 131077


def _equal(g, o, keys=("pid", "pos", "vel", "avel")):
    g, o = by_pid(g), by_pid(o)
    for k in keys:
        assert np.array_equal(g[k], np.asarray(o[k], g[k].dtype)), k


@pytest.mark.parametrize("law", ["ref", "lsd", "hm"])
@pytest.mark.parametrize("n", [TEAM8, TEAM4, LANE])
def test_mill_with_everything_on(n, law):
    print(f"[case] mill n={n} {law}", flush=True)
    R = (n / (1.1 * np.pi)) ** (1.0 / 3.0)
    deck = S.mill_deck(300, R=R, L=R, law=law, lifter_w=3.0, lifter_h=3.0)
    rng = np.random.RandomState(3)
    r, a = (R - 0.4) * np.sqrt(rng.rand(n)), rng.uniform(0.0, 2.0 * np.pi, n)
    deck["sim"].Num_Particles = n
    deck["sim"].sphere_orient = True
    deck["sim"].EnergyCalc = True
    deck["pos"] = np.stack([R + r * np.cos(a), R + r * np.sin(a), rng.uniform(0.4, R - 0.4, n)], 1).astype(np.float32)
    deck["vel"] = rng.uniform(-20.0, 20.0, (n, 3)).astype(np.float32)
    deck["avel"] = rng.uniform(-20.0, 20.0, (n, 3)).astype(np.float32)
    deck["ptype"], deck["pid"] = np.zeros(n, np.uint32), np.arange(n, dtype=np.int32)
    deck = S.place_at_lifters(deck)
    dev, ora = make_pair(deck)
    try:
        dev.drum_rotation(True)
        ora.set_drum_rotation(True)
        dev.set_lifter_rotation(deck["rad_per_step"], deck["lifter_about"])
        dev._check(dev.lib.bdem_record_wall_forces(dev.h, 1))
        for step in range(3):
            fw = ora.forces()[2]   # of the coming step: walls do not turn
            dev.step(1)
            ora.run(1, deck["rad_per_step"], deck["lifter_about"])
            wf = np.zeros((n, 3), np.float32)
            dev._check(dev.lib.bdem_get_wall_forces(dev.h, wf.ctypes.data_as(C.POINTER(T.Float3)), None))
            assert np.array_equal(-wf, np.asarray(fw, np.float32)), f"wall forces, step {step}"
        assert np.count_nonzero(ora.lifter_types()) > 8
        sg, so = dev.get_state(), ora.state()
        _equal(sg, so)
        assert rel_err(by_pid(sg)["quat"], by_pid(so)["quat"], 1e-3) <= 1e-5
        eg, (_, ex) = dev.energy().astype(np.float64), ora.energy()
        assert (ex > 0).all()
        assert np.allclose(eg, ex * 1e-4, rtol=1e-3, atol=0)
    finally:
        dev.close()
        ora.close()


@pytest.mark.parametrize("law", ["lsd", "hm"])
@pytest.mark.parametrize("n", [TEAM8, TEAM4, LANE])
def test_discharge(n, law):
    """Spheres below the kill height go at the checks, every second step."""
    print(f"[case] discharge n={n} {law}", flush=True)
    L = 1.2 + (n / 1.2) ** (1.0 / 3.0)
    deck = S.random_deck(n, seed=8, L=L, law=law, vmax=2000.0)
    deck["sim"].Kill_Particles = True
    deck["sim"].Silo_Kill_Height = 2.0
    deck["ext"].kill_check_interval = 2
    dev, ora = make_pair(deck)
    try:
        killed = 0
        for _ in range(3):
            dev.step(2)
            ora.step(2)
            so = ora.state()
            dead = int(np.count_nonzero(so["pid"] < 0))
            assert dev.kill_count() == dead >= killed
            killed = dead
            g, o = by_pid(dev.get_state()), by_pid(so)
            assert np.array_equal(g["pid"], o["pid"])
            live = o["pid"] >= 0
            for k in ("pos", "vel", "avel"):
                assert np.array_equal(g[k][live], np.asarray(o[k], np.float32)[live]), k
        assert killed > n // 100
    finally:
        dev.close()
        ora.close()


@pytest.mark.parametrize("law", ["ref", "lsd", "hm"])
@pytest.mark.parametrize("more_z", [False, True])
@pytest.mark.parametrize("n", [TEAM8, TEAM4, LANE])
def test_grids_with_unequal_sides(n, more_z, law):
    """Half as many z as x cells (spheres past the grid's end too), and twice
    as many (spheres whose hash passes the cell table)."""
    print(f"[case] grid n={n} more_z={more_z} {law}", flush=True)
    L = 1.2 + (n / 1.5) ** (1.0 / 3.0)
    deck = S.random_deck(n, seed=9, L=L, law=law, aliased=not more_z)
    if more_z:
        c = deck["sim"].num_NNCells
        deck["sim"].num_NNCells = T.Int3(c.x, c.y, 2 * c.z)
    dev, ora = make_pair(deck)
    try:
        lo, no = ora.contacts()
        lg, ng = dev.debug_step_contacts()
        assert np.array_equal(ng, no)
        used = np.arange(32)[None, :] < np.minimum(no, 32)[:, None]
        assert np.array_equal(np.where(used, lg, 0), np.where(used, lo, 0))
        dev.step(2)
        ora.step(3)
        _equal(dev.get_state(), ora.state())
    finally:
        dev.close()
        ora.close()


@pytest.mark.parametrize("law", ["ref", "lsd", "hm"])
def test_contacts_past_the_listed_by_a_lane(law):
    """About 20 contacts a sphere, 135 candidates: the tail after the twelve
    listed contacts, and rows past the stage."""
    deck = S.random_deck(LANE, seed=5, L=1.2 + (LANE / 5.0) ** (1.0 / 3.0), law=law)
    dev, ora = make_pair(deck)
    try:
        _, no = ora.contacts()
        assert no.max() > 32 and (no > 12).mean() > 0.5
        dev.step(3)
        ora.step(3)
        _equal(dev.get_state(), ora.state())
    finally:
        dev.close()
        ora.close()


@pytest.mark.parametrize("use_graph", [0, 1])
def test_large_batch_on_the_plain_grid(use_graph):
    """More than 131,072 slots: the batch's lane kernel, against lone runs,
    which teams of lanes step."""
    decks = S.batch_box_decks(count=5, seed=6, nmin=26000, nmax=45000)
    total = sum(d["sim"].Num_Particles for d in decks)
    print(f"[case] batch of {total} spheres, graphs {use_graph}", flush=True)
    assert total > 140000
    batch = bdem.Batch()
    for d in decks:
        dev = make_device(d)
        batch.add(dev)
        dev.close()
    batch.set_tuning(threads=256, waves_per_cu=0, grab=1, cell_factor=1.0, use_graph=use_graph)
    batch.finalize()
    for nsteps in (1, 2, 35):
        batch.step(nsteps)
    for k, d in enumerate(decks):
        lone = make_device(dict(d, sim=batch.instance_sim(k)))
        lone.step(38)
        _equal(batch.get_state(k), lone.get_state())
        lone.close()
    assert batch.status() == 0
    batch.close()


def touching_deck(m, cell):
    """m^3 spheres on a lattice of pitch exactly 1 with radii 0.5 (1 + k 2^-23),
    k in -45 .. 45: d^2 is 1 and (ra + rb)^2 within 90 of its last places."""
    n = m ** 3
    deck = S.random_deck(n, seed=11, L=m + 2.0, law="lsd", polydisperse=True, rmin=0.4, rmax=0.5, cell=cell,
                         vmax=0.5, wmax=0.5)
    gi = np.indices((m, m, m)).reshape(3, -1).T
    deck["pos"] = (gi + 0.75).astype(np.float32)
    k = np.random.RandomState(12).randint(-45, 46, n)
    deck["radius"] = (0.5 * (1.0 + k * 2.0 ** -23)).astype(np.float32)
    return deck


# 17 / 30 / 36 / 51 cubed: teams of 16, 8 and 4 lanes, a lane each.  Cells of
# 1 and 2.5: runs of 3 and of about 47 candidates (odd and even, past 32)
@pytest.mark.parametrize("cell", [1.0, 2.5])
@pytest.mark.parametrize("m", [17, 30, 36, 51])
def test_touching_to_the_last_places(m, cell):
    print(f"[case] touching {m}^3 cell {cell}", flush=True)
    deck = touching_deck(m, cell)
    dev, ora = make_pair(deck)
    try:
        lo, no = ora.contacts()
        assert 0.2 < no.sum() / (6.0 * m ** 3) < 0.8   # about half of the neighbours touch
        lg, ng = dev.debug_step_contacts()
        assert np.array_equal(ng, no)
        used = np.arange(32)[None, :] < np.minimum(no, 32)[:, None]
        assert np.array_equal(np.where(used, lg, 0), np.where(used, lo, 0))
    finally:
        dev.close()
        ora.close()


@pytest.mark.parametrize("m", [25, 30])
def test_touching_polyhedra_lists(m):
    """The same for the bounding spheres of both list kernels (15,625 and
    27,000 cubes): the step's listed contacts, counted."""
    deck = S.poly_deck(m ** 3, seed=13, L=m + 3.2, shape="cube", size=0.5, spacing=1.0)
    gi = np.indices((m, m, m)).reshape(3, -1).T
    deck["pos"] = (gi + 0.75).astype(np.float32)
    deck["vel"] = np.zeros_like(deck["vel"])
    base = deck["pobj"][0]
    rng = np.random.RandomState(14)
    pobj = []
    for _ in range(8):
        p = type(base).from_buffer_copy(base)
        p.radius = float(np.float32(0.5 * (1.0 + rng.randint(-45, 46) * 2.0 ** -23)))
        pobj.append(p)
    deck["pobj"] = pobj
    deck["sim"].Num_ParticleObjects = 8
    deck["ptype"] = rng.randint(0, 8, m ** 3).astype(np.uint32)
    dev, ora = make_pair(deck)
    try:
        _, no = ora.contacts()
        assert 0.15 < no.sum() / (6.0 * m ** 3) < 0.85
        dev.step(1)
        assert dev.debug_poly_queues()[0] == int(np.minimum(no, 32).sum())
    finally:
        dev.close()
        ora.close()

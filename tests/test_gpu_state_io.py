"""The state's way in and out at the edges of its staging (4 MiB halves,
copies split over threads past 512 KiB): what was set comes back bit for bit,
per-particle radii and masses stay with their slots through a reload,
arrays that are not asked for are left alone, threads may read one context or
batch at once, and a read leaves the steps around it alone."""
import ctypes as C
import threading

import numpy as np
import pytest

import bdem
from bdem import scenarios as S
from bdem import types as T
from helpers import make_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 257, 262144, 262145, 700001])
def test_state_round_trip(n):
    print(f"[case] n={n}", flush=True)
    deck = S.random_deck(n, seed=3, L=2.0 + n ** (1.0 / 3.0), law="lsd", polydisperse=True)
    dev = make_device(deck)
    try:
        for _ in range(2):   # the second load keeps the slots' radii and masses
            g = dev.get_state()
            for k in ("pos", "vel", "avel"):
                assert np.array_equal(g[k], np.asarray(deck[k], np.float32)), k
            assert np.array_equal(g["pid"], deck["pid"]) and np.array_equal(g["ptype"], deck["ptype"])
            dev.set_state(deck["pos"], deck["ptype"], deck["pid"], vel=deck["vel"], avel=deck["avel"])
        # positions alone: velocities and spins stay
        dev.set_state(deck["pos"][::-1].copy(), deck["ptype"], deck["pid"])
        g = dev.get_state()
        assert np.array_equal(g["pos"], np.asarray(deck["pos"], np.float32)[::-1])
        assert np.array_equal(g["vel"], np.asarray(deck["vel"], np.float32))
        # IDs alone
        pid = np.full(n, -7, np.int32)
        assert dev.lib.bdem_get_positions(dev.h, None, None, None, pid.ctypes.data_as(C.POINTER(C.c_int))) == 0
        assert np.array_equal(pid, deck["pid"])
    finally:
        dev.close()


def test_quaternions_and_centres_round_trip():
    deck = S.hull_box_deck(300, seed=46)
    dev = make_device(deck)
    try:
        g = dev.get_state()
        com = np.array([[s.COM.x, s.COM.y, s.COM.z] for s in deck["shapes"]], np.float32)
        assert np.array_equal(g["pos"], np.asarray(deck["pos"], np.float32) - com[deck["pid"]])
        assert np.array_equal(g["quat"], np.asarray(deck["quat"], np.float32))
        assert isinstance(deck["shapes"][0], T.PolyShape)
    finally:
        dev.close()


def _in_threads(count, work):
    errors = []

    def run(k):
        try:
            work(k)
        except BaseException as e:   # noqa: BLE001 - handed to the test
            errors.append(e)

    threads = [threading.Thread(target=run, args=(k,)) for k in range(count)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if errors:
        raise errors[0]


def test_threads_read_one_context():
    n = 50001
    deck = S.random_deck(n, seed=4, L=2.0 + n ** (1.0 / 3.0), law="lsd")
    dev = make_device(deck)
    try:
        dev.step(3)
        want = dev.get_state()

        def read(k):
            for _ in range(6):
                g = dev.get_state()
                for key in ("pos", "vel", "avel", "pid", "ptype"):
                    assert np.array_equal(g[key], want[key]), (k, key)

        _in_threads(4, read)
    finally:
        dev.close()


def test_threads_read_one_batch():
    decks = S.batch_box_decks(count=4, seed=5, nmin=1024, nmax=6000)
    devs = [make_device(d) for d in decks]
    b = bdem.Batch()
    for d in devs:
        b.add(d)
    b.finalize()
    b.step(3)
    want = [b.get_state(k) for k in range(4)]

    def read(k):
        for r in range(8):
            g = b.get_state((k + r) % 4)
            for key, v in g.items():
                assert np.array_equal(v, want[(k + r) % 4][key]), key

    _in_threads(4, read)
    b.close()
    for d in devs:
        d.close()


def test_reads_leave_the_steps_alone():
    """Steps queued one launch at a time by one thread while another reads."""
    n = 20001
    deck = S.random_deck(n, seed=6, L=2.0 + n ** (1.0 / 3.0), law="hm")
    dev, ref = make_device(deck), make_device(deck)
    try:
        dev.set_graphs(False)
        done = threading.Event()

        def work(k):
            if k == 0:
                for _ in range(60):
                    dev.step(5)
                done.set()
            else:
                while not done.is_set():
                    g = dev.get_state()
                    assert np.array_equal(np.sort(g["pid"]), np.arange(n))

        _in_threads(2, work)
        ref.step(300)
        a, b = dev.get_state(), ref.get_state()
        for key in ("pos", "vel", "avel", "pid"):
            assert np.array_equal(a[key], b[key]), key
    finally:
        dev.close()
        ref.close()

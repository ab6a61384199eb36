"""The state's way in and out at the edges of its staging (4 MiB halves,
copies split over threads past 512 KiB): what was set comes back bit for bit,
per-particle radii and masses stay with their slots through a reload, and
arrays that are not asked for are left alone."""
import ctypes as C

import numpy as np
import pytest

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

"""The contact scan's one-integer test against the reference's own expression
sqrt(d2) - s < 0 in float32: a key below 0 is a sure overlap, one above 64 a
sure miss, over all magnitudes, the floats around equality, denormals,
infinities and NaN of both signs.  This proves the arithmetic, restated here
in numpy; the device's own scans are held to the restatement's contact lists
with pairs inside the undecided band in test_gpu_step_forms.py."""
import numpy as np


def _key(d2, s):
    with np.errstate(over="ignore", invalid="ignore"):
        s2 = (s * s).astype(np.float32)
    b = d2.view(np.uint32) & np.uint32(0x7FFFFFFF)
    return (b - (s2.view(np.uint32) - np.uint32(32))).astype(np.uint32)


def _check(d2, s):
    d2, s = np.broadcast_arrays(np.asarray(d2, np.float32), np.asarray(s, np.float32))
    d2, s = np.ascontiguousarray(d2), np.ascontiguousarray(s)
    k = _key(d2, s)
    with np.errstate(invalid="ignore"):
        hit = (np.sqrt(d2) - s) < 0
    assert hit[k.view(np.int32) < 0].all()
    assert not hit[(k.view(np.int32) >= 0) & (k > 64)].any()


def test_key_never_decides_against_the_reference():
    rng = np.random.RandomState(7)
    s = np.exp(rng.uniform(np.log(1e-15), np.log(1e15), 20000)).astype(np.float32)
    s2 = (s * s).astype(np.float32)
    for off in list(range(-80, 81)) + [-(1 << 20), 1 << 20]:
        _check((s2.view(np.int32) + off).view(np.float32), s)
    # mantissas at the ends of a binade, where a float is widest and narrowest
    for m in (1.0, np.nextafter(np.float32(1), np.float32(2)), 1.41421354, 1.41421366, 1.99999988):
        e = np.float32(m) * np.float32(2.0) ** np.arange(-30, 31, dtype=np.float32)
        for off in range(-80, 81):
            _check(((e * e).astype(np.float32).view(np.int32) + off).view(np.float32), e)
    _check(np.exp(rng.uniform(-60, 60, 200000)), np.exp(rng.uniform(-30, 30, 200000)))


def test_key_on_the_edges_of_the_format():
    tiny = np.float32(1e-30)   # s * s is a denormal or zero
    _check(np.array([0.0, 1e-45, 1e-40, 1e-38, 1.0], np.float32), tiny)
    _check(np.array([0.0, 1.0, 3e38, np.inf], np.float32), np.float32(1.0))
    _check(np.array([0.0, 1.0, 3e38, np.inf], np.float32), np.float32(1e19))   # s * s near the largest float
    _check(np.array([0.0, 1.0, 3e38], np.float32), np.float32(3e19))           # s * s overflows
    nan = np.array([0x7FC00000, 0xFFC00000, 0x7F800001, 0xFF800001, 0xFFFFFFFF], np.uint32).view(np.float32)
    for s in (1e-10, 1.0, 1e10):
        k = _key(nan, np.full(5, s, np.float32))
        assert (k.view(np.int32) > 64).all()   # a miss, as the comparison with NaN gives

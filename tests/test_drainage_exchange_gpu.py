"""Fields and history between host and device: the FP64 split into two FP32
words and back, both in pieces of 2^19 cells, kept fields, and a history ring
that has wrapped."""
import ctypes as C

import numpy as np
import pytest

from soap_bubble_simulation_amd import _lib as L
from soap_bubble_simulation_amd.drainage import DrainageContext

pytestmark = pytest.mark.gpu


def _context(nt, npf, flags=0, rebase=None):
    p = L.Params()
    L.check(L.lib().sf_params_cpu_default(p))
    p.flags = flags
    if rebase:
        p.rebase_interval = rebase
    return DrainageContext(p, nt, npf, 5e-7)


@pytest.mark.parametrize("nt,npf", [(3, 1), (5, 7), (64, 128), (257, 511), (1024, 512), (1025, 512), (1499, 1399), (1500, 1401), (2048, 2048)])
def test_fields_round_trip(nt, npf):
    rng = np.random.default_rng(nt)
    h = rng.uniform(1e-7, 9e-7, (nt, npf))
    g = rng.uniform(0.0, 1.0, (nt, npf))
    hi = h.astype(np.float32)
    lo = (h - hi).astype(np.float32)
    want_h, want_g = hi.astype(np.float64) + lo, g.astype(np.float32).astype(np.float64)
    c = _context(nt, npf)
    c.set_fields(h, g)
    got = c.fields()
    assert np.array_equal(got[0], want_h) and np.array_equal(got[1], want_g)
    f32 = c.fields_f32()
    assert np.array_equal(f32[0], want_h.astype(np.float32)) and np.array_equal(f32[1], want_g.astype(np.float32))
    # one field kept, each way and in both widths
    c.set_fields(None, 1.0 - g)
    got = c.fields()
    assert np.array_equal(got[0], want_h) and np.array_equal(got[1], (1.0 - g).astype(np.float32))
    c.set_fields_f32(0.5 * hi, None)
    got = c.fields()
    assert np.array_equal(got[0], 0.5 * hi) and np.array_equal(got[1], (1.0 - g).astype(np.float32))
    c.set_fields_f32(None, g.astype(np.float32))
    c.set_fields(None, None)
    got = c.fields()
    assert np.array_equal(got[0], 0.5 * hi) and np.array_equal(got[1], want_g)


@pytest.mark.parametrize("nt,npf", [(5, 7), (64, 128), (300, 1100)])
def test_kept_field_after_odd_steps(nt, npf):
    """A field kept after an odd number of one-step launches (the current
    half of the state is the second) and the volume of fixed pole rows.  Each
    step renormalises the two words.  Reading their sum rounds it to FP64
    (2^-53 of h) and the two steps after it round the low word (|lo| <=
    2^-24 h) to 24 bits a few times each: the two states agree to 2^-45."""
    rng = np.random.default_rng(npf)
    h = rng.uniform(3e-7, 6e-7, (nt, npf))
    c = _context(nt, npf, 32 | 8, rebase=1)
    c.set_fields(h, np.full((nt, npf), 0.5))
    c.step(1, 1e-7)
    before = c.fields()[0]
    c.set_fields(None, rng.uniform(0.0, 1.0, (nt, npf)))
    assert np.array_equal(c.fields()[0], before)
    other = _context(nt, npf, 32 | 8, rebase=1)
    other.set_fields(before, c.fields()[1])
    c.step(2, 1e-7)
    other.step(2, 1e-7)
    bound = 2.0 ** -45
    assert c.history(1)[0] == pytest.approx(other.history(1)[0], rel=bound)
    assert np.all(np.abs(c.fields()[0] - other.fields()[0]) <= bound * before)


def test_history_ring_wraps():
    c = _context(5, 8, 32)
    c.step(1 << 16, 1e-9)
    first = c.history(1 << 16)
    assert len(first[0]) == 1 << 16
    c.step(100, 1e-9)
    last = c.history(1 << 16)
    assert np.array_equal(last[0][:-100], first[0][100:]) and np.array_equal(last[1][:-100], first[1][100:])
    short = c.history(130)
    assert np.array_equal(short[0], last[0][-130:]) and np.array_equal(short[1], last[1][-130:])
    assert len(c.history(0)[0]) == 0


@pytest.mark.parametrize("nt,npf,flags", [(1500, 1024, 0), (1024, 2048, 0), (4000, 256, 32 | 8)])
def test_exchange_and_steps_allocate_nothing(nt, npf, flags):
    """Device memory is taken when a context is made: exchanging its fields,
    stepping it and reading its history take none, so they cannot fail on a
    card that has filled up since."""
    hip = C.CDLL("libamdhip64.so.7")

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    warm = _context(nt, npf, flags)        # code objects and the runtime's own buffers
    for c in (warm, _context(nt, npf, flags)):
        before = free()
        h = np.full((nt, npf), 5e-7)
        c.fields()
        c.fields_f32()
        c.set_fields(h, None)
        c.set_fields_f32(h.astype(np.float32), None)
        c.step(9, 1e-9)
        c.history(4)
        after = free()
    assert after == before

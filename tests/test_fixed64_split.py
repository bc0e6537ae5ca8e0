"""The Q32.32 number of a fp32 quotient by exact fp32 steps (og_fixed64_split,
og_modes.h) restated on the CPU, against the fp64 form (uint64)(q 2^32 + 0.5)
over every exponent that takes that path: equal for every value.  A planted
mistake -- halves dropped instead of rounded up -- must be caught."""
import numpy as np


def by_split(q, half=True):
    w = np.floor(q)
    v = np.ldexp((q - w).astype(np.float32), 32).astype(np.float32)
    t = np.floor(v)
    up = ((v - t).astype(np.float32) >= np.float32(0.5)) & half
    return (w.astype(np.uint64) << np.uint64(32)) + t.astype(np.uint64) + up.astype(np.uint64)


def by_fp64(q):
    return (q.astype(np.float64) * 4294967296.0 + 0.5).astype(np.uint64)


def _values():
    rng = np.random.default_rng(3)
    out = [np.zeros(1, np.float32)]
    for e in range(0, 159):   # up to just below 2^32
        m = np.concatenate([rng.integers(0, 1 << 23, 400), [0, 1, (1 << 23) - 1, 1 << 22, (1 << 22) + 1]])
        out.append(((e << 23) | m).astype(np.uint32).view(np.float32))
    return np.concatenate(out)


def test_equal_to_the_fp64_form():
    q = _values()
    assert np.array_equal(by_split(q), by_fp64(q))


def test_a_dropped_half_is_caught():
    q = _values()
    assert not np.array_equal(by_split(q, half=False), by_fp64(q))

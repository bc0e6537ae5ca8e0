"""The wavefront sums of the binned and direct pulls (og_rowsum.h,
og_bin_wave_step) restated on the CPU: T consecutive terms per lane (36 in the
binned pull's steps, 28 in the direct one's, 12 in a short last one), each lane's run as the
moves of an even and of an odd running sum, the runs composed in lane order,
the first lane that leaves the binade added term by term.  Bar: the bits of
the sequential fp32 sum, by brute force.  Two planted mistakes -- one move per
run (a tie's parity ignored), and a binade top that is not checked -- must be
caught by the same sums."""
import numpy as np
import pytest

F, U = np.float32, np.uint32


def seq(y, x):
    y = F(y)
    for a in x:
        y = F(y + a)
    return y


def bits(y):
    return int(np.asarray(y, F).view(U))


def val(b):
    return np.asarray(b, U).view(F)[()]


def wave_sum(x, y0, T, lanes, parity=True, top=True):
    """Sum of x onto y0 in steps of lanes * T terms."""
    x = np.asarray(x, F)
    y = F(y0)
    pad = -len(x) % (lanes * T)
    for block in np.concatenate([x, np.zeros(pad, F)]).reshape(-1, lanes, T):
        p = 0
        while p < lanes:
            yb = bits(y)
            f = p
            if 2.0 ** -100 <= y < 2.0 ** 100:
                bb = yb & 0xFF800000
                s = np.empty((2, lanes), F)
                s[0], s[1] = val(bb), val(bb | 1)
                for t in range(T):
                    s = (s + block[None, :, t]).astype(F)
                d = s.view(U).astype(np.int64) - np.array([[bb], [bb | 1]])
                bad = (block < 0).any(1) | (d >= 1 << 23).any(0)
                low, move, f = yb & 0x7FFFFF, 0, lanes
                for lane in range(p, lanes):
                    step = d[((yb + move) & 1) if parity else 0, lane]
                    if bad[lane] or (top and low + move + step >= 1 << 23):
                        f = lane
                        break
                    move += int(step)
                y = val(yb + move)
                if f == lanes:
                    break
            y = seq(y, block[f])
            p = f + 1
    return y


def terms(kind, n, rng):
    if kind == "few bits":                      # many exact halves of an ulp
        return (rng.integers(1, 8, n) * F(2.0) ** -rng.integers(18, 28, n)).astype(F)
    if kind == "ranks":
        return (F(0.15) / rng.integers(1, 400, n)).astype(F)
    if kind == "power law":
        return (rng.pareto(1.1, n) * 1e-4).astype(F)
    if kind == "equal":
        return np.full(n, F(0.15) / F(7), F)
    return np.where(rng.random(n) < 0.3, 0, rng.random(n)).astype(F)   # "zeros"


KINDS = ["few bits", "ranks", "power law", "equal", "zeros"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [1, 27, 28, 29, 36, 37, 63, 64, 65, 1791, 1792, 1793, 2303, 2304, 2305, 6000])
def test_equal_to_the_sequential_sum(kind, n):
    rng = np.random.default_rng(n)
    x = terms(kind, n, rng)
    for y0 in (0.0, 0.3, 1e-5, 7.99999):
        want = seq(y0, x)
        for T, lanes in ((36, 64), (28, 64), (12, 64), (4, 8)):
            assert bits(wave_sum(x, y0, T, lanes)) == bits(want), (kind, n, y0, T)


@pytest.mark.parametrize("mistake", [dict(parity=False), dict(top=False)])
def test_planted_mistakes_are_caught(mistake):
    caught = 0
    for kind in KINDS:
        x = terms(kind, 6000, np.random.default_rng(5))
        caught += bits(wave_sum(x, 0.3, 28, 64, **mistake)) != bits(seq(0.3, x))
    assert caught


def test_terms_that_are_not_positive_and_finite():
    x = terms("ranks", 3000, np.random.default_rng(1))
    for at, a in ((700, -0.5), (1500, np.inf), (2000, np.nan), (10, -0.0)):
        y = x.copy()
        y[at] = a
        got, want = wave_sum(y, 0.0, 28, 64), seq(0.0, y)
        assert bits(got) == bits(want) or (np.isnan(got) and np.isnan(want))


def test_zeros_and_leading_zeros():
    x = np.zeros(3000, F)
    for T in (36, 28, 12):
        assert bits(wave_sum(x, 0.0, T, 64)) == 0
    x[1500:] = F(1e-3)
    for T in (36, 28, 12):
        assert bits(wave_sum(x, 0.0, T, 64)) == bits(seq(0.0, x))


@pytest.mark.parametrize("kind", KINDS)
def test_long_rows(kind):
    x = terms(kind, 40_000, np.random.default_rng(40))
    assert bits(wave_sum(x, 0.0, 36, 64)) == bits(seq(0.0, x))

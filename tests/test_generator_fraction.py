"""The generator compares a draw's scaled fraction with scaled thresholds
instead of the draw modulo 10000 with the thresholds: the same outcome for
every residue, at the ends of the draws' range and over random draws."""
import numpy as np

INV = np.uint64((2**64 - 1) // 10000 + 1)


def fraction(v):
    with np.errstate(over="ignore"):
        return (v.astype(np.uint64) * INV) >> np.uint64(32)


def limits(k):
    return np.where(k >= 10000, 2**32 - 1, (k.astype(np.uint64) << np.uint64(32)) // np.uint64(10000))


def test_fraction_orders_like_the_residue():
    residue = np.arange(10000)
    top = (2**31 - 2) // 10000
    for q in (0, 1, 2, 4295, top // 2, top - 1, top):
        v = q * 10000 + residue
        v = v[v < 2**31 - 1]
        f = fraction(v)
        r = residue[: len(v)]
        lim = limits(np.arange(10001))
        # residue r is at least k exactly for k <= r: the last limit f reaches is r's own
        assert np.array_equal(np.searchsorted(lim, f, side="right") - 1, r), q
    rng = np.random.default_rng(1)
    v = rng.integers(0, 2**31 - 1, 1 << 20)
    assert np.array_equal(np.searchsorted(limits(np.arange(10001)), fraction(v), side="right") - 1, v % 10000)

"""The square root in the device's normals (sqrt_rn_log): from a reciprocal root
r of x, g = x r, and one Goldschmidt step g + (r / 2) (x - g g), all of them
float32 with the two last operations fused.  Restated in numpy (products of
floats are exact in float64, the last sum is taken in long double) for the
range of -2 log a: with r correctly rounded the result is the correctly rounded
root; with r an ulp off, which the hardware's may be, it is never off by more
than an ulp, and hardly ever off."""
import numpy as np

F = np.float32


def _step(x, r):
    g = x * r
    e = (x.astype(np.float64) - g.astype(np.float64) ** 2).astype(F)
    h = F(0.5) * r
    return (g.astype(np.longdouble) + (e.astype(np.float64) * h.astype(np.float64)).astype(np.longdouble)).astype(F)


def test_goldschmidt_step_from_reciprocal_roots_within_an_ulp():
    rng = np.random.default_rng(5)
    bits = np.arange(0, 1 << 24, 7, dtype=np.uint32) + (np.uint32(127) << np.uint32(23))  # [1, 4)
    x = bits.view(F)
    sq = (np.arange(1, 1200, dtype=F) / F(128.0)) ** 2  # exact squares
    wide = np.exp(rng.uniform(np.log(2.0**-23), np.log(89.0), 200_000)).astype(F)
    x = np.concatenate([x, sq, np.nextafter(sq, F(0)), np.nextafter(sq, F(100)), wide, F([2.0**-23, 1.0, 2.0, 89.0])])
    root = np.sqrt(x)
    r = (1 / np.sqrt(x.astype(np.float64))).astype(F)
    np.testing.assert_array_equal(_step(x, r), root)
    for near in (np.nextafter(r, F(0)), np.nextafter(r, F(np.inf))):
        d = _step(x, near).view(np.int32).astype(np.int64) - root.view(np.int32)
        assert np.abs(d).max() <= 1 and np.count_nonzero(d) <= 10

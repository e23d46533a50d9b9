"""The merge's single-precision pair bound (k_merge_groups) rejects no pair within
the threshold: the expression restated in numpy float32 for pairs exactly on
it, their (u, v) covariances up to the correlation 1 - 1e-6 beyond which a
survivor counts as ill-conditioned, their offsets along the thin axis (where
the terms cancel) and in any direction.  The slack left has to be more than
what the rounding of this restatement's own inputs is worth."""
import numpy as np

F = np.float32


def _cov(rng, n):
    a = 10 ** rng.uniform(-6, 1, n)
    b = a * 10 ** rng.uniform(-3, 3, n)
    r = np.sqrt(1 - 10 ** rng.uniform(np.log10(2.1e-6), 0, n)) * rng.choice([-1, 1], n)
    return np.stack([a, r * np.sqrt(a * b), b])


def test_no_pair_within_the_threshold_is_rejected():
    rng = np.random.default_rng(1)
    n = 400_000
    s = _cov(rng, n)
    t = np.where(rng.random(n) < 0.5, s * 10 ** rng.uniform(-2, 2, n), _cov(rng, n))
    uu, uv, vv = s + t
    thr = 10 ** rng.uniform(-1, 2, n)
    th = rng.uniform(0, 2 * np.pi, n)
    thin = rng.random(n) < 0.5
    du = np.where(thin, 1 + 1e-3 * rng.normal(size=n), np.cos(th)) * np.sqrt(uu)
    dv = np.where(thin, -np.sign(uv) * (1 + 1e-3 * rng.normal(size=n)), np.sin(th)) * np.sqrt(vv)
    k = np.sqrt(thr * (uu * vv - uv * uv) / (vv * du * du - 2 * uv * du * dv + uu * dv * dv))
    du, dv = (k * du).astype(F), (k * dv).astype(F)
    tuu, tuv, tvv = s.astype(F) + t.astype(F)
    thrf = (1.0011 * thr).astype(F)
    x, y, w = tvv * du * du, tuu * dv * dv, tuu * tvv
    left = x + y - F(2) * tuv * du * dv - F(2e-6) * (x + y)
    right = thrf * (w - tuv * tuv + F(2e-6) * w)
    assert ((right.astype(np.float64) - left) / (thr * w)).min() > 5e-7

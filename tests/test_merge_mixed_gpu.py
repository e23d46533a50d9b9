"""Merging survivors of which some have an ill-conditioned (u, v) covariance
(clouds whose points the camera sees in a line) and some do not: pairs of one
kind and of both, the first index of either.  The candidates, from windows and
from the list of the ill-conditioned ones, must be those of every pair, and
the groups those of the reference's round loop.  Groups alike give the same
moments to the bit; the round loop adds them up in another order."""
import numpy as np
import pytest

import oracle
import workloads

pytestmark = pytest.mark.gpu


def _state(p, G, share, seed):
    """Clouds about a quarter of the image; a `share` of them lines in (u, v)."""
    rng = np.random.Generator(np.random.PCG64(seed))
    N, S = p["n_particles"], p["particles_per_feature"]
    n = N * G
    mid = np.stack([rng.uniform(150, 330, n), rng.uniform(120, 260, n)], 1)[:, None]
    line = rng.uniform(0, 1, n) < share
    a = rng.uniform(0.3, 1.2, n) + np.pi / 2 * rng.integers(0, 2, n)  # 2e-4 pixels wide: still positive definite
    along = (rng.normal(0, 3.0, (n, S, 1)) * np.stack([np.cos(a), np.sin(a)], 1)[:, None]
             + rng.normal(0, 2e-4, (n, S, 1)) * np.stack([-np.sin(a), np.cos(a)], 1)[:, None])
    uv = mid + np.where(line[:, None, None], along, rng.normal(0, 2.0, (n, S, 2)))
    z = rng.uniform(4, 6, (n, 1)) * (1 + rng.normal(0, 0.03, (n, S)))
    pos = np.stack([-(uv[..., 0] - p["u0"]) * z / p["fx"], -(uv[..., 1] - p["v0"]) * z / p["fy"], z], 2)
    smp = np.concatenate([pos, rng.normal(0, 0.05, (n, S, 3)), np.full((n, S, 1), 1.0 / S)], 2)
    states, _ = oracle.Oracle(p).parents()
    return dict(states=states, weights=np.full(N, 1.0 / N), gcount=np.full(N, G, np.int32),
                wg=rng.uniform(0.05, 0.9, n), samples=np.ascontiguousarray(smp.reshape(n * S, 7).T), n_predict=0,
                n_update=0, n_resample=0), line


@pytest.mark.parametrize("share", [0.03, 0.5, 1.0])
def test_mixed_survivors_merge_as_with_every_pair(share):
    import scphd_amd

    p, _ = workloads.workload("c0", n_particles=6, particles_per_feature=64)
    p["storage"], p["max_gaussians"], p["min_separation"] = 1, 0, 12.0
    st, line = _state(p, 120, share, 61)
    rng = np.random.Generator(np.random.PCG64(62))
    u, v = rng.uniform(150, 330, 90), rng.uniform(120, 260, 90)
    out = {}
    for name, limits in dict(windows={}, scratch=dict(merge_lds_cap=0), every=dict(merge_all_pairs=True),
                             rounds=dict(merge_force_rounds=True)).items():
        gpu = scphd_amd.Filter(p)
        gpu.set_debug_limits(**limits)
        gpu.set_state(st)
        gpu.update(u, v, True)
        P = gpu.fit_debug()[[6, 7, 7, 8]].T.reshape(-1, 2, 2)
        P = P - P @ np.linalg.solve(P + np.eye(2), P)  # of the survivors
        good = P[:, 0, 0] * P[:, 1, 1] - P[:, 0, 1] ** 2 > 2e-6 * P[:, 0, 0] * P[:, 1, 1]
        np.testing.assert_array_equal(good, ~line)
        out[name] = (gpu.update_debug(), gpu.maps())
        gpu.close()
    debug, maps = out["windows"]
    assert (debug["nsurvivors"] > 150).all()  # births and detection terms
    assert (debug["nmerged"] < 0.8 * debug["nsurvivors"]).all()  # many merge
    for name in ("scratch", "every"):
        for key in debug:
            np.testing.assert_array_equal(out[name][0][key], debug[key], err_msg=f"{name}: {key}")
        for x, y in zip(out[name][1], maps):
            np.testing.assert_array_equal(x, y, err_msg=name)
    np.testing.assert_array_equal(out["rounds"][0]["nmerged"], debug["nmerged"])
    np.testing.assert_allclose(out["rounds"][1][1], maps[1], rtol=1e-12, atol=0)

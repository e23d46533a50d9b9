"""Samples on the image's edge: whether one counts as seen is the same in the
fit's sweep, which writes the clouds of the terms it knows to be kept, and in
k_nd_fill, which writes those it knows only afterwards.  Points whose u or v
is the image's first or last to a rounding, seen by turned cameras, fall on
either side of it with the order of a sum; the weights 1 - pd_i of a cloud
must not depend on its Gaussian's weight, which decides who writes it.  Exact:
the two are the same expressions."""
import numpy as np
import pytest

import oracle
import workloads

pytestmark = pytest.mark.gpu


def _edge_state(p, G, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    N, S = p["n_particles"], p["particles_per_feature"]
    states, _ = oracle.Oracle(p).parents()
    states = np.array(states)
    states[:, 3:6] = rng.uniform(-0.3, 0.3, (N, 3))
    n = N * G * S
    u, v = rng.uniform(40, 600, n), rng.uniform(40, 440, n)
    side = rng.integers(0, 4, n)
    u = np.where(side == 0, 0.0, np.where(side == 1, 2 * p["u0"], u))
    u[np.arange(n) % 5 < 2] = -80.0  # never seen: pd_g at most 3/5 of pd, so every term is kept
    v = np.where(side == 2, 0.0, np.where(side == 3, 2 * p["v0"], v))
    d = -p["fx"] / rng.uniform(3, 9, n)
    pos = np.empty((n, 3))
    for i in range(n):
        pos[i] = oracle.disparity_to_world(p, states[i // (G * S)], [u[i], v[i], d[i], 0.0, 0.0, 0.0])[:3]
    smp = np.concatenate([pos.T, np.zeros((3, n)), np.full((1, n), 1.0 / S)])
    return dict(states=states, weights=np.full(N, 1.0 / N), gcount=np.full(N, G, np.int32), wg=None,
                samples=np.ascontiguousarray(smp), n_predict=0, n_update=0, n_resample=0)


@pytest.mark.parametrize("samples", [96, 100, 41])
def test_who_writes_a_cloud_does_not_change_it(samples):
    import scphd_amd

    p, _ = workloads.workload("c0", n_particles=8, particles_per_feature=samples)
    p["storage"], p["min_weight"] = 1, 1e-2
    G = 64
    st = _edge_state(p, G, samples)
    out = []
    for w in (0.9, 0.06):  # (1 - pd) w above the threshold: the sweep; below it: k_nd_fill
        assert (w * (1 - p["pd"]) >= p["min_weight"]) == (w == 0.9)
        gpu = scphd_amd.Filter(p)
        gpu.set_state(dict(st, wg=np.full(8 * G, w)))
        gpu.update(np.zeros(0), np.zeros(0), False)
        assert gpu.update_debug()["nnondetect"].sum() == 8 * G
        out.append(gpu.maps()[2])
        gpu.close()
    seen = out[0][6] < 0.5
    assert 0.1 < seen.mean() < 0.9  # the points are on the edge
    np.testing.assert_array_equal(out[0], out[1])

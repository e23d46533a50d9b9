"""The sample blocks and the kernels that stream them at the edges of their
layout: sample counts about the step of 16 and the noise group of 64, and
parents whose map sizes are about the four Gaussians of a wavefront (none at
all among them).  Lock-step against the FP64 oracle with the tolerances of
test_gpu_parity, and clouds through the ABI and a compaction unchanged."""
import numpy as np
import pytest

import oracle
import scene
import workloads
from test_gpu_parity import _close, compare_fit, run_lockstep

pytestmark = pytest.mark.gpu


def _params(samples, storage, n_particles=12):
    p, s = workloads.workload("c0", n_particles=n_particles, particles_per_feature=samples, n_landmarks=12, lam=4.0)
    p["storage"] = storage
    return p, s


@pytest.mark.parametrize("storage", [0, 1], ids=["fp32", "fp64"])
@pytest.mark.parametrize("samples", [15, 16, 17, 33, 63, 64, 65, 129])
def test_lockstep_samples_about_the_layout_edges(samples, storage):
    p, s = _params(samples, storage)
    run_lockstep(p, s, frames=3)


def _ragged_state(p, gcounts, seed):
    """A snapshot whose parents hold gcounts[p] clouds."""
    rng = np.random.Generator(np.random.PCG64(seed))
    G, S = int(sum(gcounts)), p["particles_per_feature"]
    center = np.stack([rng.uniform(-1, 1, G), rng.uniform(-1, 1, G), rng.uniform(3, 9, G)], 1)
    pos = center[:, None, :] * (1 + rng.normal(0, 0.02, (G, S, 1))) + rng.normal(0, 0.01, (G, S, 3))
    smp = np.concatenate([pos, rng.normal(0, 0.05, (G, S, 3)), np.full((G, S, 1), 1.0 / S)], 2)
    smp = smp.astype(np.float32).astype(np.float64).reshape(G * S, 7).T
    orc = oracle.Oracle(p)
    states, _ = orc.parents()
    n = len(gcounts)
    return dict(states=states, weights=np.full(n, 1.0 / n), gcount=np.array(gcounts, np.int32),
                wg=rng.uniform(0.05, 0.9, G), samples=np.ascontiguousarray(smp), n_predict=3, n_update=3,
                n_resample=2)


@pytest.mark.parametrize("storage", [0, 1], ids=["fp32", "fp64"])
@pytest.mark.parametrize("samples", [7, 48, 100])
def test_parents_of_every_size_about_a_wavefront(samples, storage):
    import scphd_amd

    gcounts = [0, 1, 2, 3, 4, 5, 0, 0, 7, 8, 9, 0]
    p, s = _params(samples, storage, len(gcounts))
    st = _ragged_state(p, gcounts, 11)
    sc = scene.generate(seed=3, **s)
    u, v, fixed = scene.frame_measurements(sc, 1)
    orc, gpu = oracle.Oracle(p), scphd_amd.Filter(p)
    orc.set_state(st)
    gpu.set_state(st)
    np.testing.assert_array_equal(gpu.maps()[2], st["samples"])
    gpu.compact()
    np.testing.assert_array_equal(gpu.maps()[2], st["samples"])
    for f in (orc, gpu):
        f.predict(0.5)
        f.update(u, v, fixed)
    do, dg = orc.update_debug(), gpu.update_debug()
    for key in ("nsurvivors", "nmerged", "nnondetect"):
        np.testing.assert_array_equal(dg[key], do[key], err_msg=key)
    compare_fit(gpu.fit_debug(), orc.fit_debug(int(sum(gcounts))), "ragged")
    _close(dg["eta"], do["eta"], 1e-11, 1e-11, "eta")
    for a, b, tol, what in zip(gpu.maps(), orc.maps(), (0, 1e-9, 1e-6), ("sizes", "weights", "samples")):
        _close(a, b, tol, tol and (1e-6 if what == "samples" else 1e-15), what)
    gpu.close()

"""Resampling at the edges of its cumulative sum's steps (16) and chunks (2048)
and of the draw's workgroups (256): ancestors, states and weights against the
FP64 oracle, whose left-to-right sum it keeps bit for bit."""
import numpy as np
import pytest

import oracle
import workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 255, 256, 257, 2047, 2048, 2049, 2064, 4096, 4097, 6150])
def test_ancestors_about_the_steps_and_chunks(n):
    import scphd_amd

    p, _ = workloads.workload("c0", n_particles=n, particles_per_feature=4)
    rng = np.random.Generator(np.random.PCG64(n))
    orc, gpu = oracle.Oracle(p), scphd_amd.Filter(p)
    st = orc.state()
    for k in range(3):
        w = np.exp(rng.normal(0, 3.0, n))
        if n > 1:
            w[rng.integers(0, n, n // 3)] = 0.0
        st["weights"] = w / w.sum()
        st["states"] = rng.normal(0, 1, np.shape(st["states"]))
        st["n_resample"] = k
        for f in (orc, gpu):
            f.set_state(st)
        ro, rg = orc.resample(), gpu.resample()
        assert ro == rg and (n == 1 or ro)
        if ro:
            np.testing.assert_array_equal(gpu.ancestors(), orc.ancestors()[0])
        np.testing.assert_array_equal(gpu.parents()[0], orc.parents()[0])
        np.testing.assert_array_equal(gpu.parents()[1], orc.parents()[1])
    gpu.close()

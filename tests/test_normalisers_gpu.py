"""The normalisers and the survivor lists (k_eta, k_survivors) at the edges of
their blocks: parents whose map sizes are about a word of the masks (32), a
wavefront and the masks' 2048 bits, measurement counts about a wavefront (64)
and a round (256), measurements outside the image, and maps so dense that the
kept terms outgrow their list.  One update against the FP64 oracle with the
tolerances of test_gpu_parity."""
import numpy as np
import pytest

import oracle
import workloads
from test_gpu_parity import _close
from test_clouds_gpu import _ragged_state

pytestmark = pytest.mark.gpu


def _compare(p, st, u, v, limits=None):
    import scphd_amd

    orc, gpu = oracle.Oracle(p, threads=8), scphd_amd.Filter(p)
    if limits:
        gpu.set_debug_limits(**limits)
    for f in (orc, gpu):
        f.set_state(st)
        f.predict(0.5)
        f.update(u, v, True)
    do, dg = orc.update_debug(), gpu.update_debug()
    for key in ("nsurvivors", "nmerged", "nnondetect"):
        np.testing.assert_array_equal(dg[key], do[key], err_msg=key)
    _close(dg["eta"], do["eta"], 1e-11, 1e-11, "eta")
    _close(dg["loglik"], do["loglik"], 1e-11, 1e-9, "loglik")
    for a, b, tol, what in zip(gpu.maps(), orc.maps(), (0, 1e-9, 1e-6), ("sizes", "weights", "samples")):
        _close(a, b, tol, tol and (1e-6 if what == "samples" else 1e-15), what)
    gpu.close()
    return do


def _setup(gcounts, M, seed, spread=None):
    p, _ = workloads.workload("c0", n_particles=len(gcounts), particles_per_feature=16)
    p["storage"], p["max_gaussians"] = 1, 20000
    st = _ragged_state(p, gcounts, seed)
    rng = np.random.Generator(np.random.PCG64(seed + 1))
    if spread is not None:  # every cloud about one point
        smp = st["samples"]
        smp[:2] = rng.normal(0, spread, (2, smp.shape[1]))
        smp[2] = 6 + rng.normal(0, spread, smp.shape[1])
    return p, st, rng


@pytest.mark.parametrize("limits", [None, dict(eta_heavy_cap=0), dict(eta_ncand_cap=1), dict(eta_ncand_cap=0)],
                         ids=["lists", "no-windows", "short-lists", "no-lists"])
@pytest.mark.parametrize("M", [1, 63, 64, 65, 255, 256, 257, 600])
def test_map_and_measurement_counts_about_the_blocks(M, limits):
    p, st, rng = _setup([0, 1, 2, 31, 32, 33, 63, 64, 65, 129, 0, 257], M, 21)
    # a sixth of them outside the image, some twice, some in one row
    u, v = rng.uniform(-60, 720, M), rng.uniform(-60, 540, M)
    v[::7] = v[0]
    u[::11], v[::11] = u[-1], v[-1]
    _compare(p, st, u, v, limits)


@pytest.mark.parametrize("M", [40, 300])
def test_maps_about_the_chunk_of_2048(M):
    p, st, rng = _setup([2047, 2048, 2049, 3, 4100], M, 22)
    _compare(p, st, rng.uniform(0, 640, M), rng.uniform(0, 480, M))


@pytest.mark.parametrize("M", [3, 70])
def test_more_kept_terms_than_a_list_holds(M):
    p, st, rng = _setup([0, 40, 500, 1], M, 23, spread=0.01)
    u, v = 320 + rng.normal(0, 2.0, M), 240 + rng.normal(0, 2.0, M)
    do = _compare(p, st, u, v)
    assert do["nsurvivors"].max() > 8 * M

"""The merge's groups (k_merge_groups) at the edges of its workspaces: survivor
counts about a wavefront, a workgroup, the largest bucket of the weight order
(1024 equal weights) and the LDS of two and of one workgroup a CU (2048 and
4352), more candidate pairs than the buffer holds, and every pair a candidate.
Births alone weigh the same, so ties go by index.  One update against the FP64
oracle with the tolerances of test_gpu_parity."""
import numpy as np
import pytest

from test_normalisers_gpu import _compare, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 2, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 2047, 2048, 2049, 4352, 4353])
def test_survivor_counts_about_the_workspaces(M):
    p, st, rng = _setup([0, 3, 40, 0], M, 31)
    do = _compare(p, st, rng.uniform(0, 640, M), rng.uniform(0, 480, M))
    assert do["nsurvivors"].min() == M


@pytest.mark.parametrize("limits", [None, dict(merge_lds_cap=100), dict(merge_all_pairs=True),
                                    dict(merge_lds_cap=100, merge_all_pairs=True)],
                         ids=["lds", "scratch", "all-pairs", "scratch-all-pairs"])
@pytest.mark.parametrize("M,box", [(300, 200.0), (3000, 200.0), (700, 12.0)])
def test_crowded_measurements(M, box, limits):
    """3000 in 200 x 200 pixels: about 2800 pairs within reach of each other,
    more than the buffer's 2048; 700 in 12 x 12: more neighbours than their
    lists hold, so the round loop."""
    p, st, rng = _setup([0, 30, 2], M, 32)
    u, v = 100 + rng.uniform(0, box, M), 100 + rng.uniform(0, box, M)
    u[::5] = u[0]
    do = _compare(p, st, u, v, limits)
    assert do["nmerged"].max() < do["nsurvivors"].max()

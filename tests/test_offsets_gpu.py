"""The output offsets and the lists of kept terms: parent counts about one value
a thread of the scan's workgroup (1024) and the most it takes (8192), and maps
of more than one wavefront's 64 entries.  Lock-step against the FP64 oracle
with the tolerances of test_gpu_parity."""
import pytest

import workloads
from test_gpu_parity import run_lockstep

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 1023, 1024, 1025, 2049, 8191, 8192, 8193])
def test_parent_counts_about_the_scan(n):
    p, s = workloads.workload("c0", n_particles=n, particles_per_feature=8, n_landmarks=5, lam=2.0)
    run_lockstep(p, s, frames=3)


def test_maps_of_more_than_a_wavefront():
    p, s = workloads.workload("c0", n_particles=5, particles_per_feature=16, n_landmarks=60, lam=20.0)
    rep = run_lockstep(p, s, frames=4)
    assert rep[-1][1] > 5 * 128

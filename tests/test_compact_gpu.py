"""scphd_compact of a map whose values are more than a launch's 2^32 threads:
a parent's 300 clouds of 512 samples become the map of all 4096 parents by
resampling (4.4e9 values, 17.6 GB), and compaction gives every one its own
block.  The last rig's clouds, in the last of these blocks, come back as they
were set."""
import numpy as np
import pytest

import workloads
from test_clouds_gpu import _ragged_state

pytestmark = pytest.mark.gpu


def test_map_of_more_values_than_a_launch_has_threads():
    import scphd_amd

    P, G, S = 4096, 300, 512
    rigs = [workloads.rig(r + 1, n, 12, 4.0, samples=S) for r, n in enumerate((P, 2))]
    params = [dict(p, max_gaussians=0) for p, _ in rigs]
    gcounts = [0] * P + [3, 4]
    gcounts[5] = G
    st = _ragged_state(dict(params[0], n_particles=P + 2), gcounts, 41)
    st["weights"] = np.full(P + 2, 0.0)
    st["weights"][5] = 1.0
    st["weights"][P:] = 0.5
    ens = scphd_amd.Ensemble(params)
    ens.set_state(st)
    assert ens.resample() and list(ens.rig_resample()[0]) == [True, False]
    n = ens.counts()["n_gaussians"]
    assert n == P * G + 7 and n * S * 7 > 1 << 32
    before = ens.memory()
    ens.compact()
    assert ens.memory() - before > 4 * n * S * 7 // 2
    ens.remove_rig(0)
    np.testing.assert_array_equal(ens.maps()[0], [3, 4])
    np.testing.assert_array_equal(ens.maps()[2], st["samples"][:, G * S:])
    ens.close()

"""Estimates of more rigs than one slice of their launch takes (65535): every
rig's mean, covariance and cardinality against numpy."""
import numpy as np
import pytest

import workloads
from test_clouds_gpu import _ragged_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rigs", [65535, 65536, 131071])
def test_estimates_of_many_rigs(rigs):
    import scphd_amd

    p, _ = workloads.rig(1, 2, 12, 4.0, samples=4)
    rng = np.random.Generator(np.random.PCG64(rigs))
    N = 2 * rigs
    gcounts = np.zeros(N, np.int32)
    gcounts[[0, 1, N - 3, N - 2, N - 1]] = [2, 1, 3, 1, 4]
    st = _ragged_state(dict(p, n_particles=2), gcounts, 51)
    w = rng.uniform(0.1, 0.9, rigs)
    st["states"], st["weights"] = rng.normal(0, 1, (N, 12)), np.stack([w, 1 - w], 1).reshape(N)
    ens = scphd_amd.Ensemble([scphd_amd.Params.from_dict(p)] * rigs)
    ens.set_state(st)
    mean, cov, card = ens.rig_estimates()
    ens.close()
    x, w = st["states"].reshape(rigs, 2, 12), st["weights"].reshape(rigs, 2, 1)
    mu = (w * x).sum(1)
    d = x - mu[:, None]
    # sums of two terms: a few roundings of values below 20
    np.testing.assert_allclose(mean, mu, rtol=0, atol=1e-13)
    np.testing.assert_allclose(cov, (w[..., None] * d[..., None] * d[:, :, None]).sum(1), rtol=0, atol=1e-13)
    off = np.concatenate([[0], np.cumsum(gcounts)])
    best = 2 * np.arange(rigs) + (w[:, 1, 0] > w[:, 0, 0])
    np.testing.assert_allclose(card, [st["wg"][off[b]:off[b + 1]].sum() for b in best], rtol=0, atol=1e-13)

"""Parents of more Gaussians than the normalisers' masks hold (2048), whose kept
terms k_eta_list lists: map sizes just above and far above, measurement counts
about a round (256), beside parents of small maps; lists too short for the
terms, by their room per measurement and by the room of a round (4096).  One
update against the FP64 oracle with the tolerances of test_gpu_parity."""
import numpy as np
import pytest

from test_normalisers_gpu import _compare, _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limits", [None, dict(eta_heavy_cap=0), dict(eta_ncand_cap=1), dict(eta_ncand_cap=0)],
                         ids=["lists", "no-windows", "short-lists", "no-lists"])
@pytest.mark.parametrize("M", [1, 63, 256, 257, 600])
def test_map_and_measurement_counts(M, limits):
    p, st, rng = _setup([2049, 5, 0, 2300, 6000, 2048], M, 24)
    # some outside the image, some twice, some in one row
    u, v = rng.uniform(-60, 720, M), rng.uniform(-60, 540, M)
    v[::7] = v[0]
    u[::11], v[::11] = u[-1], v[-1]
    _compare(p, st, u, v, limits)


def test_more_kept_terms_than_a_parents_list_holds():
    p, st, rng = _setup([2100, 3], 3, 23, spread=0.01)
    do = _compare(p, st, 320 + rng.normal(0, 2.0, 3), 240 + rng.normal(0, 2.0, 3))
    assert do["nsurvivors"][0] > 8 * 3


def test_more_kept_terms_than_a_round_holds():
    M = 1000
    p, st, rng = _setup([2600], M, 26)
    u, v = -200 - rng.uniform(0, 300, M), rng.uniform(0, 480, M)
    u[:256], v[:256] = 320 + rng.normal(0, 60, 256), 240 + rng.normal(0, 60, 256)
    do = _compare(p, st, u, v)
    # all but the births are the first round's
    assert 4096 + M < do["nsurvivors"][0] < 8 * M

"""A snapshot that the device has no memory for is refused and leaves the
filter as it was: the same state, and the same frames from it as a filter that
was never offered the snapshot, bit for bit.  The offers are larger than the
staging buffer of the samples (FP32), and than a generation of clouds beside
one (FP64); none of their samples is read."""
import ctypes

import numpy as np
import pytest

import scene
import workloads

pytestmark = pytest.mark.gpu


def _offer(f, n):
    import scphd_amd

    L, N = scphd_amd.lib(), f.Np
    gc = np.zeros(N, np.int32)
    gc[N // 2] = n
    wg, one = np.zeros(n), np.zeros(1)
    return L.scphd_set_state(f.h, scphd_amd._dp(np.zeros((N, 12))), scphd_amd._dp(np.full(N, 1.0 / N)),
                             scphd_amd._ip(gc), ctypes.c_int64(n), scphd_amd._dp(wg), scphd_amd._dp(one), 9, 9, 9)


@pytest.mark.parametrize("pending", [False, True], ids=["between-frames", "predicted"])
@pytest.mark.parametrize("storage,n", [(0, 12_000_000), (1, 4_600_000)], ids=["staging", "generation"])
def test_refused_snapshot_leaves_the_state(storage, n, pending):
    import scphd_amd

    p, s = workloads.workload("c0", n_particles=8, particles_per_feature=512, n_landmarks=12, lam=4.0)
    p["storage"] = storage
    sc = scene.generate(seed=5, **s)
    fs = [scphd_amd.Filter(p) for _ in range(2)]
    for k in range(6):
        u, v, fixed = scene.frame_measurements(sc, k)
        for f in fs:
            f.predict(s["dt"])
            if k == 3 and pending and f is fs[0]:
                assert _offer(f, n) == -2, "the offer was to be refused"
            f.update(u, v, fixed)
            if k == 3 and not pending and f is fs[0]:
                assert _offer(f, n) == -2, "the offer was to be refused"
            f.resample()
        a, b = (f.state() for f in fs)
        for key in a:
            np.testing.assert_array_equal(a[key], b[key], err_msg=f"frame {k}: {key}")
    for f in fs:
        f.close()

"""Performance cases of the SC-PHD calibration filter: the work that a user
has the framework do, through its public entry points.

A pass is a whole calibration run over a rig's first frames: the handle is set
back to its prior (no map) and then stepped frame by frame as the reference's
main loop does (predict, update, check, resample), the cameras alternating.
So a pass meets what a run meets, births only in the first frame, maps that
grow to their steady size over the next eight or so, merging, non-detection
clouds and resampling, and every pass does the same work.  Four forms:

  plain     one rig through scphd_amd.Filter
  ensemble  many rigs in one handle, scphd_amd.Ensemble
  batch     many rigs with queued frames, scphd_amd.Batch
  resume    an evicted rig comes back: its host snapshot is loaded, one frame
            is run, and the whole state is read back

Sizes are those of workloads.py, bench.py and the tests, and odd ones between.
"""
import math
import os
import sys

import numpy as np
import torch  # noqa: F401  (loaded before the library, as programs that use both do)

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "scphd-camera-calibration_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import scene  # noqa: E402
import scphd_amd  # noqa: E402
import serve  # noqa: E402
import workloads  # noqa: E402

FP32, FP64, FP32_ARITH = 0, 1, 2


def _case(name, form="plain", parents=256, samples=100, landmarks=30, lam=10.0, storage=FP32, slam=False, rigs=1,
          frames=8):
    return dict(name=name, form=form, parents=parents, samples=samples, landmarks=landmarks, lam=float(lam),
                storage=storage, slam=slam, rigs=rigs, frames=frames)


def listed():
    return [
        # the smallest runs: a first try on a few parents; launches and read-backs count
        _case("tiny", parents=32, samples=100, frames=6),
        # the small plain workload (c0): 256 parents, 30 landmarks
        _case("c0", parents=256, samples=100, frames=12),
        # c0's scene with FP64 clouds at odd sizes
        _case("fp64_odd", parents=300, samples=77, landmarks=50, lam=15, storage=FP64, frames=8),
        # a mid-sized rig at odd sizes, calibrated from the moving camera alone (the configuration's slam switch)
        _case("odd_slam", parents=777, samples=123, landmarks=77, lam=23, slam=True, frames=8),
        # the benchmark's workload (c1): 4096 parents, 200 samples, 200 landmarks, to its steady map size
        _case("c1", parents=4096, samples=200, landmarks=200, lam=50, frames=10),
        # c1's scene in the single-precision variant
        _case("c1_fp32_arith", parents=1024, samples=200, landmarks=200, lam=50, storage=FP32_ARITH, frames=8),
        # c1's scene with FP64 clouds
        _case("c1_fp64", parents=1024, samples=200, landmarks=200, lam=50, storage=FP64, frames=8),
        # the dense scene (c3's): 300 landmarks and clutter 100, more measurements than a workgroup has threads
        _case("dense", parents=2048, samples=100, landmarks=300, lam=100, frames=8),
        # c3's parent count on a sparse scene: much resampling, small maps
        _case("many_parents", parents=16384, samples=100, landmarks=20, lam=5, frames=6),
        # small ragged rigs stepped together by one set of launches
        _case("ensemble", form="ensemble", rigs=32, parents=384, landmarks=60, lam=22, frames=6),
        # served rigs of 256 to 2048 parents, frames queued, eight workers
        _case("served", form="batch", rigs=10, parents=724, landmarks=110, lam=32, frames=6),
        # eviction and return of a rig: host snapshot, one frame, host snapshot
        _case("resume", form="resume", parents=24, samples=100, landmarks=30, frames=1),
    ]


def _steady(c):
    return 0.9 * serve.expected_gaussians_per_parent(dict(n_landmarks=c["landmarks"], lam=c["lam"]))


def _n_meas(c):
    return 0.83 * c["landmarks"] + c["lam"]


def _gaussians(c, k):
    """Map size per parent before frame k: it grows to its steady size over about eight frames."""
    return _steady(c) * (1.0 - math.exp(-k / 2.5)) if c["form"] != "resume" else 3.0 * c["landmarks"]


def _cost(c):
    n = c["parents"] * c["rigs"] * c["frames"] * _steady(c)
    return max(n * c["samples"] * (2 if c["storage"] == FP64 else 1), 2.0 * n * _n_meas(c))


def draw(rng):
    form = rng.choice(["plain"] * 6 + ["ensemble", "batch", "resume"])
    c = _case("", form=form, parents=int(round(math.exp(rng.uniform(math.log(32), math.log(6000))))),
              samples=rng.randint(64, 200), landmarks=int(round(math.exp(rng.uniform(math.log(20), math.log(300))))),
              lam=round(rng.uniform(5.0, 100.0), 1), storage=rng.choice([FP32, FP32, FP32, FP64, FP32_ARITH]),
              slam=rng.random() < 0.2, frames=rng.randint(4, 9))
    if form in ("ensemble", "batch"):
        c.update(rigs=rng.randint(3, 24), parents=min(c["parents"], 700), landmarks=min(c["landmarks"], 150),
                 lam=min(c["lam"], 60.0), slam=False)
    if form == "resume":
        c.update(parents=rng.randint(8, 40), storage=rng.choice([FP32, FP64]), frames=1, slam=False,
                 landmarks=min(c["landmarks"], 60))
    top = 0.6 * max(_cost(x) for x in listed())
    while _cost(c) > top:
        c["parents"] = max(32, int(c["parents"] * 0.8))
    del c["name"]
    return c


def work(c):
    esz = 8 if c["storage"] == FP64 else 4
    S, M, n = c["samples"], _n_meas(c), c["parents"] * c["rigs"]
    b = fl = 0.0
    for k in range(c["frames"]):
        g0, g1 = _gaussians(c, k), _gaussians(c, k + 1)
        # the state read and written once a frame: seven values a sample, a weight a Gaussian, 104 B a parent
        b += n * ((7 * esz * S + esz) * (g0 + g1) + 2 * 104) + 16 * M
        # a sample predicted, projected and summed; a posterior sample drawn (about half of the map is new);
        # a likelihood a (Gaussian, measurement)
        fl += n * (g0 * S * 200 + 0.5 * g1 * S * 150 + g0 * M * 15)
    if c["form"] == "resume":  # the snapshot crosses in doubles, twice
        b += 2 * n * _gaussians(c, 0) * S * 56
    return {"bytes": b, "flops": fl}


def _rig(c, seed, r=0):
    """Parameters and frames of rig r of a case."""
    rng = np.random.Generator(np.random.PCG64([seed, r]))
    n, L, lam, f, bl = c["parents"], c["landmarks"], c["lam"], 500.0, 0.2
    if c["rigs"] > 1:  # ragged: sizes, focal lengths and baselines differ from rig to rig, the first one's do not
        k = 2.0 ** (((r * 7) % 8) / 3.5 - 1.0) if c["form"] == "batch" else 2.0 ** (r % 2) * 2 / 3
        n, L, lam = max(8, int(n * k)), max(8, int(L * (0.4 + 1.2 * ((r * 5) % 8) / 7))), lam * (0.4 + (r % 4) * 0.4)
        f, bl = 400.0 + 400.0 * rng.random(), 0.1 + 0.4 * rng.random()
    p, s = workloads.rig(seed=seed * 1000 + r + 1, n_particles=n, n_landmarks=L, lam=lam, f=f, baseline=bl,
                         samples=c["samples"], n_frames=c["frames"], scene_rig=r)
    p["storage"] = c["storage"]
    sc = scene.generate(seed=p["seed"], **s)
    return p, s, [_sized(*scene.frame_measurements(sc, k, slam=c["slam"]), L, lam, k, rng) for k in range(c["frames"])]


def _sized(u, v, fixed, L, lam, k, rng):
    """Frame k's set at a size that the seed does not change (about the mean,
    other frames other sizes): some of the shuffled set left out, or more
    clutter."""
    n = int((0.83 * L + lam) * (1.0 + 0.03 * ((5 * k) % 7 - 3))) + 1
    more = max(0, n - len(u))
    u, v = np.append(u, rng.uniform(0, 640, more)), np.append(v, rng.uniform(0, 480, more))
    return np.ascontiguousarray(u[:n]), np.ascontiguousarray(v[:n]), fixed


def _prior(f):
    """The state that a filter is created with: its prior's parents, equal weights, no map."""
    states, weights = f.parents()
    return dict(states=states, weights=weights, gcount=np.zeros(len(weights), np.int32), wg=np.zeros(0),
                samples=np.zeros(0), n_predict=0, n_update=0, n_resample=0)


def _room(p, s):
    return int(1.1 * p["n_particles"] * serve.expected_gaussians_per_parent(s))


def prepare(c, seed):
    st = dict(form=c["form"])
    if c["form"] == "resume":
        p, snap, frame = _snapshot(c, seed)
        f = scphd_amd.Filter(p)
        # the buffers that the rig's next snapshot goes to
        room = 4 * len(snap["wg"])
        kind = np.float64 if c["storage"] == FP64 else np.float32
        st.update(f=f, snap=snap, frame=frame, wg=np.zeros(room), samples=np.zeros((7, room * c["samples"]), kind))
    elif c["form"] == "plain":
        p, s, frames = _rig(c, seed)
        f = scphd_amd.Filter(p)
        f.reserve(_room(p, s), max(len(u) for u, _, _ in frames))
        st.update(f=f, dt=s["dt"], frames=frames, prior=_prior(f))
    elif c["form"] == "ensemble":
        rigs = [_rig(c, seed, r) for r in range(c["rigs"])]
        f = scphd_amd.Ensemble([p for p, _, _ in rigs])
        f.reserve(sum(_room(p, s) for p, s, _ in rigs), max(len(u) for _, _, fr in rigs for u, _, _ in fr))
        frames = [([fr[k][0] for _, _, fr in rigs], [fr[k][1] for _, _, fr in rigs], rigs[0][2][k][2])
                  for k in range(c["frames"])]
        st.update(f=f, dt=rigs[0][1]["dt"], frames=frames, prior=_prior(f))
    else:
        b = scphd_amd.Batch(hbm_budget_bytes=200e9, n_workers=8)
        rigs = []
        for r in range(c["rigs"]):
            p, s, frames = _rig(c, seed, r)
            rid = b.add_rig(p, int(1.5 * scphd_amd.rig_footprint(p, serve.expected_gaussians_per_parent(s))))
            f = b.filter(rid)
            rigs.append(dict(id=rid, f=f, dt=s["dt"], frames=frames, prior=_prior(f)))
        st.update(b=b, rigs=rigs)
    return st


def run(st):
    if st["form"] == "resume":
        return _run_resume(st)
    if st["form"] == "batch":
        return _run_batch(st)
    f = st["f"]
    f.set_state(st["prior"])
    resampled, counts = [], []
    for u, v, fixed in st["frames"]:
        f.predict(st["dt"])
        f.update(u, v, fixed)
        if f.check() != scphd_amd.SCPHD_OK:
            raise RuntimeError("NaN parent weight")
        resampled.append(f.resample())
        q = f.update_stats()
        counts.append([q["n_gaussians_in"], q["n_survivors"], q["n_merged"], q["n_nondetect"]])
    out = dict(resampled=np.array(resampled, np.int32), counts=np.array(counts), ancestors=f.ancestors())
    out["states"], out["weights"] = f.parents()
    if st["form"] == "ensemble":
        out["mean"], out["cov"], out["cardinality"] = f.rig_estimates()
    else:
        out["mean"], out["cov"], out["cardinality"] = f.estimate()
        out["update"] = f.update_debug()
    return out


def _run_batch(st):
    b = st["b"]
    for r in st["rigs"]:
        r["f"].set_state(r["prior"])
    for k in range(len(st["rigs"][0]["frames"])):
        for r in st["rigs"]:
            b.submit(r["id"], k, r["dt"], *r["frames"][k])
    b.step()
    res = sorted(b.collect(), key=lambda x: (x["rig"], x["frame_id"]))
    if any(x["status"] != scphd_amd.SCPHD_OK for x in res):
        raise RuntimeError("a served frame failed")
    par = [r["f"].parents() for r in st["rigs"]]
    return dict(estimates=np.array([x["estimate"] for x in res]), cardinality=np.array([x["cardinality"] for x in res]),
                counts=np.array([[x["n_pairs"], x["n_gaussians"], x["resampled"]] for x in res]),
                states=np.concatenate([x for x, _ in par]), weights=np.concatenate([w for _, w in par]))


def _run_resume(st):
    f = st["f"]
    u, v, fixed = st["frame"]
    f.set_state(st["snap"])
    f.predict(DT)
    f.update(u, v, fixed)
    out = dict(fit=f.fit_debug(), update=f.update_debug())
    out["states"], out["weights"] = f.parents()
    out["resampled"] = int(f.resample())
    after = f.state()
    st["wg"][:len(after["wg"])] = after["wg"]
    st["samples"][:, :after["samples"].shape[1]] = after["samples"]
    out.update(gcount=after["gcount"], wg=st["wg"], samples=st["samples"])
    return out


# ------------------------------------------------------------------ resume: its snapshot, and its results in 64 bits
DT = 0.5


def _snapshot(c, seed):
    """A rig between frames: parents about the true extrinsics, and for each
    about three clouds a landmark (where it was seen, and ghosts beside it),
    some of them partly or wholly out of view."""
    p, s = workloads.rig(seed=seed + 1, n_particles=c["parents"], n_landmarks=c["landmarks"], lam=c["lam"],
                         samples=c["samples"], n_frames=2)
    p["storage"] = c["storage"]
    sc = scene.generate(seed=p["seed"], **s)
    rng = np.random.Generator(np.random.PCG64([seed, 77]))
    N, S, L = c["parents"], c["samples"], c["landmarks"]
    states = sc["ext2"] + rng.normal(0, 1, (N, 12)) * np.array([0.002] * 3 + [0.001] * 3 + [0.0008] * 3 + [0.0005] * 3)
    gcount = (2 * L + (13 * np.arange(N)) % (2 * L + 1)).astype(np.int32)
    G = int(gcount.sum())
    at = sc["truth"][0][rng.integers(0, L, G)] * (1.0 + rng.normal(0, 0.02, (G, 1)))
    pos = at[:, None, :] * (1.0 + rng.normal(0, 0.03, (G, S, 1))) + rng.normal(0, 0.004, (G, S, 3))
    vel = np.array([-0.04, 0.0, 0.04]) + rng.normal(0, 0.05, (G, 1, 3)) + rng.normal(0, 0.03, (G, S, 3))
    w = np.where(rng.random((G, 1)) < 0.4, 1.0 - 0.95 * (rng.random((G, S)) < 0.9), 1.0 / S)
    smp = np.concatenate([pos, vel, w[:, :, None]], axis=2).astype(np.float32).astype(np.float64)
    snap = dict(states=states, weights=rng.dirichlet(np.full(N, 5.0)), gcount=gcount,
                wg=np.exp(rng.uniform(math.log(2e-4), 0.0, G)),
                samples=np.ascontiguousarray(smp.reshape(G * S, 7).T), n_predict=11, n_update=11, n_resample=4)
    return p, snap, _sized(*scene.frame_measurements(sc, 1), L, c["lam"], 1, rng)


def _philox(c0, c1, c2, c3, seed):
    """Philox4x32-10 on uint64 arrays of 32-bit words."""
    m = np.uint64(0xFFFFFFFF)
    c0, c1, c2, c3 = np.broadcast_arrays(*[np.asarray(x, np.uint64) for x in (c0, c1, c2, c3)])
    k0, k1 = seed & 0xFFFFFFFF, seed >> 32
    for _ in range(10):
        a, b = c0 * np.uint64(0xD2511F53), c2 * np.uint64(0xCD9E8D57)
        c0, c1, c2, c3 = ((b >> np.uint64(32)) ^ c1 ^ np.uint64(k0), b & m, (a >> np.uint64(32)) ^ c3 ^ np.uint64(k1),
                          a & m)
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return c0, c1, c2, c3


def _normals(c0, c1, c2, c3, seed):
    """Four standard normals a block (last axis): Box-Muller of its word pairs, the leading 24 bits of each word."""
    x = [v.astype(np.int64) for v in _philox(c0, c1, c2, c3, seed)]
    z = []
    for h in (0, 2):
        n = x[h] + 1
        drop = np.maximum(np.frexp(n.astype(np.float64))[1] - 24, 0)
        a = np.ldexp(((n >> drop) << drop).astype(np.float64), -32)
        r, t = np.sqrt(-2.0 * np.log(a)), 2.0 * math.pi * np.ldexp((x[h + 1] >> 8).astype(np.float64), -24)
        z += [r * np.cos(t), r * np.sin(t)]
    return np.stack(z, axis=-1)


def exact(c, seed):
    """The resumed frame in 64 bits: the refit of every cloud, the
    normalisers, the likelihoods and the parents.  The other forms are whole
    runs of a particle filter, whose later frames rest on its earlier
    decisions."""
    if c["form"] != "resume":
        return None
    p, snap, (zu, zv, fixed) = _snapshot(c, seed)
    N, S, G = c["parents"], c["samples"], int(snap["gcount"].sum())
    step, key = snap["n_predict"], p["seed"]
    # parents: constant velocity with N(0, std^2) accelerations
    e = snap["states"].copy()
    par = np.arange(N)[:, None]
    a = _normals(np.arange(2), 0, par, (step << 4) | 1, key).reshape(N, 8)[:, :6] * np.array(p["cam_accel_std"])
    for o, q in ((0, a[:, :3]), (6, a[:, 3:])):
        e[:, o:o + 3] += e[:, o + 3:o + 6] * DT + 0.5 * q * DT * DT
        e[:, o + 3:o + 6] += q * DT
    # landmark samples: the same, three normals a sample, four samples to three blocks
    gp = np.repeat(np.arange(N), snap["gcount"])
    first = np.cumsum(snap["gcount"]) - snap["gcount"]
    gk = np.arange(G) - first[gp]
    s = np.arange(S)
    elem, i = ((s >> 6) << 4) | (s & 15), (s >> 4) & 3
    n12 = _normals((elem[:, None] << 2) | np.arange(3), gk[:, None, None], gp[:, None, None], (step << 4) | 2,
                   key).reshape(G, S, 12)
    n = np.take_along_axis(n12, np.broadcast_to(3 * i[:, None] + np.arange(3), (G, S, 3)), axis=2)
    q = snap["samples"].reshape(7, G, S)
    acc = n * np.array(p["feat_accel_std"])
    x = np.stack(q[:3], -1) + np.stack(q[3:6], -1) * DT + 0.5 * acc * DT * DT
    vel = np.stack(q[3:6], -1) + acc * DT
    # the moving camera's disparity space
    R = np.stack([scene.rotation(*r) for r in e[:, 6:9]])[gp]
    pc, vc = np.einsum("gsi,gij->gsj", x - e[gp, None, :3], R), np.einsum("gsi,gij->gsj", vel, R)
    fx, fy, z = p["fx"], p["fy"], pc[..., 2]
    d = np.stack([p["u0"] - fx * pc[..., 0] / z, p["v0"] - fy * pc[..., 1] / z, -fx / z,
                  -fx * (vc[..., 0] * z - vc[..., 2] * pc[..., 0]) / z ** 2,
                  -fy * (vc[..., 1] * z - vc[..., 2] * pc[..., 1]) / z ** 2, fx * vc[..., 2] / z ** 2], -1)
    seen = ((d[..., 0] >= 0) & (d[..., 0] <= 2 * p["u0"]) & (d[..., 1] >= 0) & (d[..., 1] <= 2 * p["v0"])
            & (d[..., 2] >= 0))
    pd = p["pd"] * seen
    pdg = pd.sum(1) / S
    w = q[6] * pd
    W = w.sum(1)
    some = W > 0
    w = w / np.where(some, W, 1.0)[:, None]
    mu = np.where(some[:, None], (w[..., None] * d).sum(1), d[:, 0])
    dv = d - mu[:, None, :]
    P = np.einsum("gs,gsi,gsj->gij", w, dv, dv) * (1.0 + (w * w).sum(1))[:, None, None]
    low = [(r, k) for r in range(6) for k in range(r + 1)]
    fit = np.concatenate([mu.T, np.stack([P[:, r, k] for r, k in low]), pdg[None]])
    # detection terms: innovation, gain, Joseph covariance and its test
    var = np.diag([p["std_u"] ** 2, p["std_v"] ** 2])
    Sg = P[:, :2, :2] + var
    Si, det = np.linalg.inv(Sg), np.linalg.det(Sg)
    K = P[:, :, :2] @ Si
    A = np.eye(6) - np.concatenate([K, np.zeros((G, 6, 4))], axis=2)
    Pn = A @ P @ A.transpose(0, 2, 1) + K @ var @ K.transpose(0, 2, 1)
    ok, Lc = np.ones(G, bool), np.zeros((G, 6, 6))
    with np.errstate(invalid="ignore", divide="ignore"):
        for r, k in low:
            t = Pn[:, r, k] - (Lc[:, r, :k] * Lc[:, k, :k]).sum(1)
            ok &= (t > 1e-9 * Pn[:, r, r]) if r == k else True
            Lc[:, r, k] = np.sqrt(t) if r == k else t / Lc[:, k, k]
        wg = snap["wg"] * p["ps"]
        base = np.where(ok & (pdg > 0), np.log(pdg) + np.log(wg) - math.log(2 * math.pi) - 0.5 * np.log(det), -np.inf)
    bpc = math.log(len(zu) * p["birth_w0"] + p["lambda"] / (2 * p["v0"]) ** 2)
    eta, ll = np.empty((N, len(zu))), np.empty(N)
    for j in range(N):
        g = slice(first[j], first[j] + snap["gcount"][j])
        nu = np.stack([zu[None, :] - mu[g, 0, None], zv[None, :] - mu[g, 1, None]], -1)
        lw = base[g, None] - 0.5 * np.einsum("gmi,gij,gmj->gm", nu, Si[g], nu)
        top = np.maximum(lw.max(0), bpc)
        eta[j] = top + np.log(np.exp(lw - top).sum(0) + np.exp(bpc - top))
        ll[j] = eta[j].sum() + wg[g].sum()
    lp = np.log(snap["weights"]) + ll
    wn = np.exp(lp - lp.max())
    return dict(fit=fit, update=dict(eta=eta, loglik=ll, nmerged=None, nnondetect=None, nsurvivors=None), states=e,
                weights=wn / wn.sum(), resampled=None, gcount=None, wg=None, samples=None)

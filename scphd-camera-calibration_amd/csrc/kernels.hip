/*
 * kernels.hip -- gfx950 kernels of the SC-PHD camera calibration step.
 *
 * Reference: cheesinglee/scphd-camera-calibration.  Each kernel names the
 * reference code whose semantics it implements; none is a translation of it:
 * the reference launches ~40 thrust/CUDA kernels per step over dense
 * N_g x M intermediates, this file fuses them into per-Gaussian wavefront
 * kernels and per-parent workgroup kernels that never materialise the
 * dense (Gaussian, measurement) array.
 */
#include "kernels.h"

#include <float.h>

#include <algorithm>

#include <type_traits>

namespace scphd {

static constexpr int NT = 256; /* threads per workgroup for per-parent kernels */
static constexpr int WPB = 4;  /* wavefronts (Gaussians) per workgroup for per-Gaussian kernels */

/* ------------------------------------------------------------ reductions */
/* DPP lane moves on the two 32-bit halves of a double (full EXEC assumed). */
template <int CTRL>
__device__ inline double dpp_f64(double x) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

template <int CTRL>
__device__ inline float dpp_f32(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xF, 0xF, false));
}

__device__ inline double readlane_f64(double x, int l) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(x), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(x), l);
    return __hiloint2double(hi, lo);
}

/* Sum over a full wavefront: four DPP steps inside each 16-lane row (swap
 * neighbours, swap pairs, half-row mirror, row mirror) leave every lane
 * with its row's sum; the four row sums are read into scalar registers and
 * added.  Every lane gets the result.  All 64 lanes must be active. */
__device__ inline double wave_sum_dpp(double x) {
    x += dpp_f64<0xB1>(x);  /* quad_perm [1,0,3,2] */
    x += dpp_f64<0x4E>(x);  /* quad_perm [2,3,0,1] */
    x += dpp_f64<0x141>(x); /* row_half_mirror */
    x += dpp_f64<0x140>(x); /* row_mirror */
    return (readlane_f64(x, 0) + readlane_f64(x, 16)) + (readlane_f64(x, 32) + readlane_f64(x, 48));
}

__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ inline double wave_max(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

/* Sum over a workgroup of NT threads; every thread gets the result. */
__device__ inline double block_sum(double v, double* sh) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) sh[w] = v;
    __syncthreads();
    double r = 0.0;
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) r += sh[i];
    return r;
}

__device__ inline double block_max(double v, double* sh) {
    v = wave_max(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) sh[w] = v;
    __syncthreads();
    double r = -INFINITY;
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) r = fmax(r, sh[i]);
    return r;
}

/* Exclusive scan over a workgroup of NT threads; *total gets the sum. */
__device__ inline int block_exscan(int v, int* sh, int* total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    __syncthreads();
    if (lane == 63) sh[w] = x;
    __syncthreads();
    int base = 0, tot = 0;
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) {
        if (i < w) base += sh[i];
        tot += sh[i];
    }
    *total = tot;
    return base + x - v;
}

__device__ inline int upper_parent(const int32_t* off, int n, int64_t x) {
    /* largest p in [0, n) with off[p] <= x, for nondecreasing off[0..n] with off[n] > x */
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if ((int64_t)off[mid] <= x)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

/* ------------------------------------------------------------ prediction */
struct Bounds12 {
    double a[12], b[12];
};

/* Uniform prior over [a, b] per extrinsic component, weights 1/N
 * (src/scphdcameracalibration.cu:835-980). */
__global__ void k_prior(double* ext, double* pw, int Np, Bounds12 ab, NoiseKey key) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= Np) return;
    for (int c = 0; c < 12; ++c) {
        uint32_t x[4];
        noise_block(key, NS_PRIOR, 0, (uint32_t)p, 0, 0, (uint32_t)(c / 2), x);
        const double r = (c % 2 == 0) ? uniform_co(x[0], x[1]) : uniform_co(x[2], x[3]);
        ext[(int64_t)p * 12 + c] = r * (ab.b[c] - ab.a[c]) + ab.a[c];
    }
    pw[p] = 1.0 / Np;
}

/* Parent extrinsics through OrientedLinearCVMotionModel3D::computeNoisyMotion
 * with N(0, std^2) accelerations (predict_camera functor,
 * src/scphdcameracalibration.cu:129-152, :1062-1100). */
__global__ void k_parent_predict(double* ext, int Np, OrientedLinearCVMotionModel3D cam, double dt, RigKeys rk,
                                 uint64_t step) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= Np) return;
    double a[6];
    if (!rk.keys) { /* one rig: the key stays in scalar registers */
        normals<6>(rk.key, NS_CAMERA, step, (uint32_t)p, 0, 0, a);
    } else {
        int pl;
        const LaneKey key = rk.of(p, pl);
        normals<6>(key, NS_CAMERA, step, (uint32_t)pl, 0, 0, a);
    }
    double* e = ext + (int64_t)p * 12;
    EuclideanPoint c{e[0], e[1], e[2], e[3], e[4], e[5]};
    EuclideanPoint g{e[6], e[7], e[8], e[9], e[10], e[11]};
    cam.computeNoisyMotion(c, g, dt, a[0] * cam.std_ax_cartesian(), a[1] * cam.std_ay_cartesian(),
                           a[2] * cam.std_az_cartesian(), a[3] * cam.std_ax_angular(), a[4] * cam.std_ay_angular(),
                           a[5] * cam.std_az_angular());
    e[0] = c.x; e[1] = c.y; e[2] = c.z; e[3] = c.vx; e[4] = c.vy; e[5] = c.vz;
    e[6] = g.x; e[7] = g.y; e[8] = g.z; e[9] = g.vx; e[10] = g.vy; e[11] = g.vz;
}

__global__ void k_scale(double* x, int64_t n, double a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] *= a;
}

/* One wavefront's share of writing the table that gives the streaming kernels
 * their parents: table entries off[p] .. off[p + 1] - 1 are parent p's, four
 * to a wavefront (a 16-lane row each), and wavefront w of the kernel takes
 * those from off[p] + 4 (w - first_wave(off, p)) on for p = wave_parent[w].
 * Wavefronts never straddle parents, so that a parent's camera, model and
 * noise key are scalar; one that has no entry of its parent holds -1 (at most
 * one a parent). */
__device__ inline int first_wave(int off_p, int p) { return off_p / 4 + p; }

__device__ inline void write_wave_parents(int off0, int off1, int p, int lane, int32_t* wave_parent) {
    const int w0 = first_wave(off0, p), n = first_wave(off1, p + 1) - w0, used = (off1 - off0 + 3) / 4;
    for (int i = lane; i < n; i += 64) wave_parent[w0 + i] = i < used ? p : -1;
}

/* Camera used by an update: the parent's extrinsics, or all-zero extrinsics
 * for the fixed camera (src/scphdcameracalibration.cu:1167-1176); and the map
 * table's wave_parent; and the update's counters zeroed.  One wavefront per
 * parent. */
__global__ __launch_bounds__(256) void k_pose(const double* ext, double* pose, int Np, int fixed, const int32_t* prig,
                                              const int32_t* rfixed, const int32_t* goff, int32_t* wave_parent,
                                              int32_t* counters) {
    const int p = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (blockIdx.x == 0 && threadIdx.x < UC_COUNT) counters[threadIdx.x] = 0;
    if (p >= Np) return;
    write_wave_parents(goff[p], goff[p + 1], p, lane, wave_parent);
    if (lane != 0) return;
    if (rfixed) fixed = rfixed[prig[p]];
    CameraPose c;
    if (fixed) {
        c = CameraPose::identity();
    } else {
        const double* e = ext + (int64_t)p * 12;
        Extrinsics x{{e[0], e[1], e[2], e[3], e[4], e[5]}, {e[6], e[7], e[8], e[9], e[10], e[11]}};
        c = CameraPose::fromExtrinsics(x);
    }
    double* o = pose + (int64_t)p * 12;
    for (int i = 0; i < 9; ++i) o[i] = c.R[i];
    for (int i = 0; i < 3; ++i) o[9 + i] = c.t[i];
}

__device__ inline CameraPose load_pose(const double* pose, int p) {
    CameraPose c;
    const double* o = pose + (int64_t)p * 12;
#pragma unroll
    for (int i = 0; i < 9; ++i) c.R[i] = o[i];
#pragma unroll
    for (int i = 0; i < 3; ++i) c.t[i] = o[9 + i];
    return c;
}

/* Landmark sample prediction (predict_features functor,
 * src/scphdcameracalibration.cu:154-178): the constant-velocity step with
 * acceleration draws a[i] * std_i (LinearCVMotionModel3D::computeNoisyMotion),
 * x + v dt + a std dt^2 / 2 and v + a std dt. */
__device__ inline EuclideanPoint noisy_motion(EuclideanPoint x, const NoisyMotion& m, const double a[3]) {
    x.x = fma(a[0], m.sh[0], fma(x.vx, m.dt, x.x));
    x.y = fma(a[1], m.sh[1], fma(x.vy, m.dt, x.y));
    x.z = fma(a[2], m.sh[2], fma(x.vz, m.dt, x.z));
    x.vx = fma(a[0], m.sd[0], x.vx);
    x.vy = fma(a[1], m.sd[1], x.vy);
    x.vz = fma(a[2], m.sd[2], x.vz);
    return x;
}

/* the prediction of the sample (p, k, s) */
template <typename Key>
__device__ inline EuclideanPoint predict_sample(EuclideanPoint x, const NoisyMotion& m, Key key, uint64_t step, uint32_t p, uint32_t k, uint32_t s) {
    double a[3];
    feature_normals(key, step, p, k, s, a);
    return noisy_motion(x, m, a);
}

/* the same for the members of a noise group in order (phase = member) */
template <typename Key>
__device__ inline EuclideanPoint predict_sample_seq(EuclideanPoint x, const NoisyMotion& m, Key key, uint64_t step, uint32_t p, uint32_t k, uint32_t s,
                                                    uint32_t phase, FeatureCarry& c) {
    double a[3];
    feature_normals_seq(key, step, p, k, s, phase, c, a);
    return noisy_motion(x, m, a);
}

/* the seven values of sample s of a block of S samples */
template <typename T>
__device__ inline void load_sample(const T* block, int S, int s, T r[7]) {
#pragma unroll
    for (int c = 0; c < 7; ++c) r[c] = block[cloud_at(S, s, c)];
}

template <typename T>
__global__ __launch_bounds__(256) void k_materialize(Clouds<T> src, Clouds<T> dst, const int32_t* gblock,
                                                     const int32_t* gparent, const int32_t* goff, int64_t Ng, int S,
                                                     LinearCVMotionModel3D feat, double dt, RigKeys rk, uint64_t step,
                                                     int arith32) {
    /* a grid stride: a map may have more samples than a launch threads */
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < Ng * S; i += (int64_t)gridDim.x * 256) {
        const int64_t g = i / S;
        const int s = (int)(i - g * S);
        const int p = gparent[g];
        const int k = (int)(g - goff[p]);
        T r[7];
        load_sample<T>(src.block(gblock[g]), S, s, r);
        T* const db = dst.block(g);
        auto put = [&](int c, T v) { db[cloud_at(S, s, c)] = v; };
        if (arith32) { /* the single-precision prediction of the FP32-arithmetic variant */
            float x[6], n[3];
#pragma unroll
            for (int c = 0; c < 6; ++c) x[c] = (float)r[c];
            if (!rk.keys) {
                feature_normals(rk.key, step, (uint32_t)p, (uint32_t)k, (uint32_t)s, n);
            } else {
                int pl;
                const LaneKey key = rk.of(p, pl);
                feature_normals(key, step, (uint32_t)pl, (uint32_t)k, (uint32_t)s, n);
            }
            predict_f(x, motion_f(feat, dt), n);
#pragma unroll
            for (int c = 0; c < 6; ++c) put(c, (T)x[c]);
            put(6, r[6]);
            continue;
        }
        EuclideanPoint x{(double)r[0], (double)r[1], (double)r[2], (double)r[3], (double)r[4], (double)r[5]};
        if (!rk.keys) { /* one rig: the key stays in scalar registers */
            x = predict_sample(x, NoisyMotion(feat, dt), rk.key, step, (uint32_t)p, (uint32_t)k, (uint32_t)s);
        } else {
            int pl;
            const LaneKey key = rk.of(p, pl);
            x = predict_sample(x, NoisyMotion(feat, dt), key, step, (uint32_t)pl, (uint32_t)k, (uint32_t)s);
        }
        put(0, (T)x.x);
        put(1, (T)x.y);
        put(2, (T)x.z);
        put(3, (T)x.vx);
        put(4, (T)x.vy);
        put(5, (T)x.vz);
        put(6, r[6]);
    }
}

/* ------------------------------------------------------- reproject + fit */
/* Sum over the 16 lanes of a row (four DPP steps: swap neighbours, swap
 * pairs, half-row mirror, row mirror); every lane of the row gets the sum.
 * The row must be fully active; rows are independent. */
__device__ inline double row_sum16(double x) {
    x += dpp_f64<0xB1>(x);
    x += dpp_f64<0x4E>(x);
    x += dpp_f64<0x141>(x);
    x += dpp_f64<0x140>(x);
    return x;
}
__device__ inline float row_sum16(float x) {
    x += dpp_f32<0xB1>(x);
    x += dpp_f32<0x4E>(x);
    x += dpp_f32<0x141>(x);
    x += dpp_f32<0x140>(x);
    return x;
}

/* The lane's sample of one step of a cloud, from the step's place `p` in its
 * block, w samples wide: 16 or more, fewer in the last step, whose lanes
 * without a sample read its last one, or none after it (nothing is read). */
template <typename T>
__device__ inline void load_full_step(const T* p, int lane, T r[7]) {
#pragma unroll
    for (int c = 0; c < 7; ++c) r[c] = p[c * 16 + lane];
}

template <typename T>
__device__ inline void load_step(const T* p, int w, int lane, T r[7]) {
    if (w >= 16) {
        load_full_step(p, lane, r);
    } else if (w > 0) {
        int l = min(lane, w - 1);
        asm volatile("" : "+v"(l)); /* this branch's addresses are formed in it */
#pragma unroll
        for (int c = 0; c < 7; ++c) r[c] = p[c * w + l];
    }
}

/* The order of the sums of the samples s0 .. s0 + 15 of a cloud
 * (world_to_camera): x, y, z in the second step of each triple of whole
 * steps, whose end is whole_triples(S), y, x, z in the others.  Every kernel
 * that judges whether the camera sees a sample goes by it, so that one on
 * the image's edge is judged alike. */
__device__ inline int whole_triples(int S) { return S - S % 48; }
__device__ inline bool sums_xy(int s0, int triples) { return (uint32_t)s0 / 16 % 3 == 1 && s0 < triples; }

/* One sample of a Gaussian's cloud: the deferred prediction applied, its
 * disparity-space point, its field-of-view flag and stored weight. */
template <typename T, typename Key>
__device__ inline void eval_sample(const FitArgs& a, const DisparityMeasurementModel& meas, const T r[7], Key kk,
                                   int pl, int k, int s, const CameraPose& pose, bool xy, EuclideanPoint& x,
                                   DisparityPoint& d, bool& in, double& w, FeatureCarry* fc = nullptr,
                                   uint32_t phase = 0) {
    x = EuclideanPoint{(double)r[0], (double)r[1], (double)r[2], (double)r[3], (double)r[4], (double)r[5]};
    w = (double)r[6];
    if (a.pending) {
        if (fc)
            x = predict_sample_seq(x, a.motion, kk, a.pstep, (uint32_t)pl, (uint32_t)k, (uint32_t)s, phase, *fc);
        else
            x = predict_sample(x, a.motion, kk, a.pstep, (uint32_t)pl, (uint32_t)k, (uint32_t)s);
    }
    d = disparity_fast(meas, pose, x, xy);
    in = meas.inRange(d);
}

/* The FP32-arithmetic form of eval_sample: the sample's world point x (after
 * the deferred prediction), its disparity-space point q and field-of-view
 * flag, and its stored weight, all in single precision. */
struct SampleCtxF {
    MeasF m;
    PoseF pose;
    MotionF mo;
};

template <typename T, typename Key>
__device__ inline void eval_sample_f(const FitArgs& a, const SampleCtxF& cx, const T r[7], Key kk, int pl, int k,
                                     int s, float x[6], float q[6], bool& in, float& w, FeatureCarry* fc = nullptr,
                                     uint32_t phase = 0) {
#pragma unroll
    for (int c = 0; c < 6; ++c) x[c] = (float)r[c];
    w = (float)r[6];
    if (a.pending) {
        float n[3];
        if (fc)
            feature_normals_seq(kk, a.pstep, (uint32_t)pl, (uint32_t)k, (uint32_t)s, phase, *fc, n);
        else
            feature_normals(kk, a.pstep, (uint32_t)pl, (uint32_t)k, (uint32_t)s, n);
        predict_f(x, cx.mo, n);
    }
    disparity_f(cx.m, cx.pose, x, q);
    in = in_range_f(cx.m, q);
}

__device__ inline void write_fit(const FitArgs& a, int64_t g, int lane, const double* mu, const double* P, double pdg) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int q = lane + 16 * h;
        double v = 0.0;
#pragma unroll
        for (int c = 0; c < 6; ++c)
            if (q == FP_MU + c) v = mu[c];
#pragma unroll
        for (int e = 0; e < 21; ++e)
            if (q == FP_P + e) v = P[e];
        if (q == FP_PD) v = pdg;
        if (q < FP_COUNT) a.fit[(int64_t)q * a.Ng + g] = v;
    }
}

/* The noise key of parent p and p's index in its rig: the kernel argument
 * (in scalar registers) for one rig, the rig's key per lane in an ensemble. */
template <bool RG>
__device__ inline std::conditional_t<RG, LaneKey, NoiseKey> row_key(const RigKeys& rk, int p, int& pl) {
    if constexpr (RG) {
        return rk.of(p, pl);
    } else {
        pl = p;
        return rk.key;
    }
}

/* The measurement model of parent p's rig, `m`: the kernel argument itself
 * for one rig (RG false, the model stays in scalar registers), else a copy
 * of the rig's entry of per_rig. */
template <bool RG>
struct RowMeas;
template <>
struct RowMeas<false> {
    const DisparityMeasurementModel& m;
    __device__ RowMeas(const DisparityMeasurementModel& one, const DisparityMeasurementModel*, const RigKeys&, int)
        : m(one) {}
};
template <>
struct RowMeas<true> {
    DisparityMeasurementModel m;
    __device__ RowMeas(const DisparityMeasurementModel&, const DisparityMeasurementModel* per_rig, const RigKeys& rk,
                       int p)
        : m(per_rig[rk.prig[p]]) {}
};

/* Per-parent data read through the constant address space: with a parent
 * that is the same in every active lane, the loads are scalar and the values
 * stay in scalar registers, where FP64 instructions take them as operands. */
typedef __attribute__((address_space(4))) const double cdouble_t;
typedef __attribute__((address_space(4))) const int32_t cint_t;
typedef __attribute__((address_space(4))) const uint32_t cuint_t;

__device__ inline CameraPose scalar_pose(const double* pose, int p) {
    cdouble_t* o = (cdouble_t*)(pose + (int64_t)p * 12);
    CameraPose c;
#pragma unroll
    for (int i = 0; i < 9; ++i) c.R[i] = o[i];
#pragma unroll
    for (int i = 0; i < 3; ++i) c.t[i] = o[9 + i];
    return c;
}

/* What a wavefront needs of one parent: its camera, its rig's measurement
 * model, noise key and step counter, and its index in the rig. */
struct ParentCtx {
    CameraPose pose;
    DisparityMeasurementModel meas;
    NoiseKey key;
    uint64_t step;
    int pl;
    __device__ ParentCtx(const double* poses, const DisparityMeasurementModel& one,
                         const DisparityMeasurementModel* per_rig, const RigKeys& rk, uint64_t handle_step, int p)
        : pose(scalar_pose(poses, p)), meas(one), key(rk.key), step(handle_step), pl(p) {
        if (!rk.keys) return;
        const int r = ((cint_t*)rk.prig)[p];
        pl = p - ((cint_t*)rk.poff)[r];
        cuint_t* k = (cuint_t*)(rk.keys + r);
        key.k0 = k[0];
        key.k1 = k[1];
        /* the counter a filter of the rig's own would use */
        if (rk.sbase) step = (uint32_t)handle_step - ((cuint_t*)rk.sbase)[SC_COUNT * r + rk.which];
        constexpr int ND = sizeof(DisparityMeasurementModel) / sizeof(double);
        static_assert(sizeof(NoiseKey) == 2 * sizeof(uint32_t) && ND * sizeof(double) == sizeof(meas));
        double v[ND];
#pragma unroll
        for (int i = 0; i < ND; ++i) v[i] = ((cdouble_t*)(per_rig + r))[i];
        __builtin_memcpy(&meas, v, sizeof(meas));
    }
};

/* waves per SIMD the fit kernel is compiled for (register budget 512 / n).
 * Bound: VALU issue (0.87 ms of 491,572 Gaussians x 200 samples without any
 * memory access at 3 waves, 0.98 at 2) and memory (0.90 ms without the
 * normals), which overlap only in part.  At 4096 parents, 200 landmarks: 7.6
 * ms a frame with seven planes, the camera in vector registers and 2 waves;
 * 7.1 with clouds in blocks and the camera scalar; 6.2 with 3 waves, which
 * wavefronts of one parent leave the registers for. */
#ifndef SCPHD_FIT_WAVES
#define SCPHD_FIT_WAVES 3
#endif

/* LDS accesses of one wavefront's lanes before and after it, in that order */
__device__ inline void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

/* the kernel's first argument, read here and not before: pointers that only
 * a kernel's end needs are not held in scalar registers over its sweep */
template <typename S>
__device__ inline const S& kernarg_late() {
    typedef __attribute__((address_space(4))) const char* cptr_t;
    cptr_t k = (cptr_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(k));
    return *(const S*)k;
}

/* k_fit's and k_sample's arguments */
template <typename T>
struct FitKernArgs {
    FitArgs a;
    Clouds<T> src, dst;
};
template <typename T>
struct SampleKernArgs {
    SampleArgs a;
    Clouds<T> dst;
};

/* one row's share of k_fit's LDS; 17: lanes a value apart use other banks */
template <typename A>
struct FitShared {
    A part[16 * 17];
    double tot[32], K[6];
};

/* Sixteen row sums: lane l of the row gets the sum over its lanes of v[l],
 * added up as row_sum16 does (neighbours, pairs of them, halves, the row). */
template <typename A>
__device__ inline double row_total(A* part, const A (&v)[16], int lane) {
    wave_lds_fence();
#pragma unroll
    for (int e = 0; e < 16; ++e) part[e * 17 + lane] = v[e];
    wave_lds_fence();
    A x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = part[lane * 17 + i];
#pragma unroll
    for (int w = 1; w < 16; w *= 2)
#pragma unroll
        for (int i = 0; i < 16; i += 2 * w) x[i] += x[i + w];
    return (double)x[0];
}

/* Sixteen lanes (one row of a wavefront) per Gaussian, four Gaussians per
 * wavefront: deferred prediction, world -> disparity with the parent's
 * camera and the field-of-view Pd (worldToDisparityKernel,
 * src/kernels.cu:6-47), per-Gaussian Pd (computePdKernel :82-99), sample
 * reweighting by pd and normalisation (src/scphdcameracalibration.cu:1602-1608,
 * normalizeWeightsKernel src/kernels.cu:996-1018), and the weighted moment
 * fit (fitGaussiansKernel :102-438, covariance normaliser (W^2 + sum w^2) / W).
 *
 * Samples stream through once: each lane accumulates, with weights
 * w' = w pd, the sums of w', w'^2, w' (q - K) and w' (q - K)(q - K)^T about
 * a shift K, from which the normalised mean and centred covariance follow;
 * 30 row sums through LDS.  K is the first sample with w' > 0 (the first
 * sample when there is none).
 *
 * The non-detection cloud (kept when w_g (1 - pd_g) >= min_weight,
 * computeNonDetections src/scphdcameracalibration.cu:1290-1420; sample
 * weights 1 - pd_i; the samples themselves are the predicted cloud, which
 * the reference's world -> disparity -> world round trip reproduces to
 * rounding) is written during the sweep when the term is kept for certain,
 * w_g (1 - Pd) >= min_weight (pd_g <= Pd).  A term that may go either way
 * is decided after the sweep and, when kept, listed for k_nd_fill, which
 * writes its cloud; most such terms are dropped, and their clouds are never
 * written.  A cloud whose weights are all zero, which the reference
 * normalises to weight 1 per sample, is listed in redo[] and refitted by
 * k_fit_fix when pd_g > 0; with pd_g = 0 its fit cannot reach any output and
 * is the first sample with zero covariance.
 *
 * One row of k_fit, its Gaussian g of parent p (the same for every row of
 * the wavefront).
 * A, the arithmetic type of the per-sample work: double, or float for the
 * FP32-arithmetic variant (FP32 storage), whose moment sums are single
 * precision up to the row sums and whose in-view count is an integer. */
template <typename T, typename A>
__device__ inline void fit_row(const FitArgs& a, const ParentCtx& pc, int64_t g, int k, const T* from, T* to,
                               FitShared<A>& sh) {
    constexpr bool F32 = std::is_same_v<A, float>;
    static_assert(!F32 || std::is_same_v<T, float>, "single-precision arithmetic needs FP32 storage");
    const int lane = threadIdx.x & 15;
    const DisparityMeasurementModel& meas = pc.meas;
    const CameraPose& pose = pc.pose;
    const int S = a.S;
    const double wg = a.gw[g];
    const double Pd = meas.pd();
    const bool nd_sure = wg * (1.0 - Pd) >= a.min_weight; /* kept for certain */
    /* the cloud is written in the sweep when the term is kept for certain, or
     * when it would be kept at the pd_g of its source term at the last update
     * (a non-detection term's cloud moves little in one step): a guess that
     * costs only the write of a cloud nothing references if it proves wrong */
    const bool nd_write = nd_sure || (a.gpd && wg * (1.0 - (double)a.gpd[g]) >= a.min_weight);
    SampleCtxF cx;
    if constexpr (F32) cx = SampleCtxF{meas_f(meas), pose_f(pose), motion_f(a.feat, a.dt)};
    const A PdA = (A)Pd;

    [[maybe_unused]] double spd = 0.0; /* sum of pd_i (double arithmetic) */
    [[maybe_unused]] float nin = 0.0f; /* in-view samples (single-precision arithmetic) */
    A sw = 0, sw2 = 0, m1[6], m2[21], K[6];
    bool kw = false; /* K is a weighted sample (uniform along the row) */
    FeatureCarry fc; /* prediction normals carried between the steps of a noise group */
#pragma unroll
    for (int c = 0; c < 6; ++c) m1[c] = 0.0;
#pragma unroll
    for (int e = 0; e < 21; ++e) m2[e] = 0.0;
    /* two sample buffers, used in place: a step takes its samples out of one
     * and at once loads the step two ahead into it.  Steps go in groups of
     * four, the noise group, so that a step's place in it (which normals it
     * draws and which it carries) is fixed. */
    [[maybe_unused]] const int triples = whole_triples(S);
    T buf[2][7];
    load_step(from, S, lane, buf[0]);
    load_step(from + 112, S - 16, lane, buf[1]);
    /* one step of 16 samples, s0 .. s0 + 15, member J of its noise group;
     * FULL: all of them exist */
    auto step = [&](auto full, auto member, int s0) {
        constexpr bool FULL = decltype(full)::value;
        constexpr int J = decltype(member)::value;
        T(&b)[7] = buf[J & 1];
        const int s = s0 + lane;
        const bool valid = FULL || s < S;
        const int width = FULL ? 16 : min(S - s0, 16);
        T* const o = to + 7 * s0 + lane;
        float n[3] = {0.0f, 0.0f, 0.0f};
        NoiseKey key = pc.key; /* its round keys are formed anew, not held over the sweep */
        asm volatile("" : "+s"(key.k0), "+s"(key.k1));
        if (a.pending && valid)
            feature_normals_seq(key, pc.step, (uint32_t)pc.pl, (uint32_t)k, (uint32_t)s, (uint32_t)J, fc, n);
        A x[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) x[c] = (A)b[c];
        A w = (A)b[6];
        /* out of the buffer before the loads into it */
        asm volatile("" : "+v"(w));
#pragma unroll
        for (int c = 0; c < 6; ++c) asm volatile("" : "+v"(x[c]));
        if (FULL && J < 2) /* in the same group, which is whole */
            load_full_step(from + 7 * (s0 + 32), lane, b);
        else
            load_step(from + 7 * (s0 + 32), S - s0 - 32, lane, b);
        if (a.pending && valid) {
            if constexpr (F32) {
                predict_f(x, cx.mo, n);
            } else {
                const double an[3] = {(double)n[0], (double)n[1], (double)n[2]};
                const EuclideanPoint e =
                    noisy_motion(EuclideanPoint{x[0], x[1], x[2], x[3], x[4], x[5]}, a.motion, an);
                x[0] = e.x; x[1] = e.y; x[2] = e.z; x[3] = e.vx; x[4] = e.vy; x[5] = e.vz;
            }
        }
        if (nd_write && valid) {
#pragma unroll
            for (int c = 0; c < 6; ++c) o[c * width] = (T)x[c];
        }
        A q[6] = {0, 0, 0, 0, 0, 0};
        bool in = false;
        if (valid) {
            if constexpr (F32) {
                disparity_f(cx.m, cx.pose, x, q);
                in = in_range_f(cx.m, q);
            } else {
                const DisparityPoint d = disparity_fast(
                    meas, pose, EuclideanPoint{x[0], x[1], x[2], x[3], x[4], x[5]}, sums_xy(s0, triples));
                in = meas.inRange(d);
                q[0] = d.u; q[1] = d.v; q[2] = d.d; q[3] = d.vu; q[4] = d.vv; q[5] = d.vd;
            }
        }
        if (nd_write && valid) o[6 * width] = (T)(1.0 - (in ? Pd : 0.0));
        const A pd = in ? PdA : (A)0;
        const A wp = valid ? w * pd : (A)0;
        if (J == 0 && s0 == 0) {
            /* shift: the Gaussian's first sample, broadcast along the row
             * (the fit of a cloud with no weighted sample) */
#pragma unroll
            for (int c = 0; c < 6; ++c) K[c] = __shfl(q[c], 0, 16);
        }
        if (__ballot(!kw)) {
            /* rows still without a weighted sample take the first one
             * that appears as the shift: every sum is exactly zero until
             * then, and a shift inside the weighted cloud keeps the
             * one-pass moments exact to rounding (a single weighted
             * sample gives zero covariance exactly) */
            const uint32_t rb = (uint32_t)(__ballot(wp > (A)0) >> (threadIdx.x & 48)) & 0xFFFFu;
            if (!kw && rb != 0) {
                const int l = __builtin_ctz(rb);
#pragma unroll
                for (int c = 0; c < 6; ++c) K[c] = __shfl(q[c], l, 16);
                kw = true;
            }
        }
        if constexpr (F32)
            nin += in ? 1.0f : 0.0f;
        else
            spd += pd;
        sw += wp;
        sw2 += wp * wp;
        A dv[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) dv[c] = valid ? q[c] - K[c] : (A)0;
#pragma unroll
        for (int c = 0; c < 6; ++c) m1[c] += wp * dv[c];
#pragma unroll
        for (int r = 0; r < 6; ++r)
#pragma unroll
            for (int c = 0; c <= r; ++c) m2[pidx(r, c)] += wp * dv[r] * dv[c];
        /* the sums stay in this step: left alone, the compiler moves all four
         * steps' to the group's end, and their points wait in registers */
        asm volatile("" : "+v"(sw), "+v"(sw2));
        if constexpr (F32)
            asm volatile("" : "+v"(nin));
        else
            asm volatile("" : "+v"(spd));
#pragma unroll
        for (int c = 0; c < 6; ++c) asm volatile("" : "+v"(m1[c]));
#pragma unroll
        for (int e = 0; e < 21; ++e) asm volatile("" : "+v"(m2[e]));
    };
    const std::integral_constant<bool, true> full;
    const std::integral_constant<bool, false> part;
    const std::integral_constant<int, 0> j0;
    const std::integral_constant<int, 1> j1;
    const std::integral_constant<int, 2> j2;
    const std::integral_constant<int, 3> j3;
    int s0 = 0;
    for (; s0 + 64 <= S; s0 += 64) {
        step(full, j0, s0);
        step(full, j1, s0 + 16);
        step(full, j2, s0 + 32);
        step(full, j3, s0 + 48);
    }
    if (s0 < S) { /* the last group: fewer steps, the last of them partial */
        step(part, j0, s0);
        if (s0 + 16 < S) step(part, j1, s0 + 16);
        if (s0 + 32 < S) step(part, j2, s0 + 32);
        if (s0 + 48 < S) step(part, j3, s0 + 48);
    }
    /* The row sums: sixteen values at a time, every lane's part of them
     * through LDS, each lane adding up the value of its own number -- m1 and
     * m2 at their fit planes, then sum pd_i (or the in-view count), sw, sw2.
     * The rest of the fit goes on a value a lane.  (Row sums by DPP with the
     * rest in every lane took 600 instructions a Gaussian, a seventh of the
     * kernel at S = 200 and a quarter at S = 100; this takes about 170.) */
    A v0[16], v1[16];
#pragma unroll
    for (int c = 0; c < 6; ++c) v0[c] = m1[c];
#pragma unroll
    for (int e = 0; e < 10; ++e) v0[6 + e] = m2[e];
#pragma unroll
    for (int e = 10; e < 21; ++e) v1[e - 10] = m2[e];
    if constexpr (F32)
        v1[11] = nin;
    else
        v1[11] = spd;
    v1[12] = sw;
    v1[13] = sw2;
    v1[14] = v1[15] = 0;
    const FitArgs& o = kernarg_late<FitArgs>();
    const double t0 = row_total(sh.part, v0, lane), t1 = row_total(sh.part, v1, lane);
    sh.tot[lane] = t0;
    sh.tot[16 + lane] = t1;
    if (lane == 0) {
#pragma unroll
        for (int c = 0; c < 6; ++c) sh.K[c] = (double)K[c];
    }
    wave_lds_fence();
    const double sum_pd = F32 ? sh.tot[FP_PD] * Pd : sh.tot[FP_PD], sw_r = sh.tot[28], sw2_r = sh.tot[29];
    const double pdg = sum_pd / S;

    /* normalised weights w'_i / sum w': mean K + sum w (q - K); centred
     * covariance sum w (q - K)(q - K)^T - (2 - W) dm dm^T with W = sum w */
    const double r = sw_r > 0 ? 1.0 / sw_r : 0.0;
    const double W = sw_r * r, W2 = sw2_r * r * r;
    /* W = 0: with pd_g = 0 the fit is the first sample with zero covariance
     * (its detection terms have weight 0); with pd_g > 0 (possible only when
     * Pd = 1) k_fit_fix refits it with unit weights, as the reference does */
    const double scale = W > 0 ? (W * W + W2) / W : 0.0;
    auto cov = [&](int e, double t) { /* packed entry e of the covariance */
        const int i = (e >= 1) + (e >= 3) + (e >= 6) + (e >= 10) + (e >= 15), j = e - i * (i + 1) / 2;
        const double di = sh.tot[i] * r, dj = sh.tot[j] * r;
        return (t * r - (2.0 - W) * di * dj) * scale;
    };
    const double f0 = lane < 6 ? sh.K[lane < 6 ? lane : 0] + t0 * r : cov(max(lane - 6, 0), t0);
    const double f1 = lane < 11 ? cov(min(lane + 10, 20), t1) : pdg;
    o.fit[(int64_t)lane * o.Ng + g] = f0;
    if (lane < 12) o.fit[(int64_t)(lane + 16) * o.Ng + g] = f1;
    const bool keep = wg * (1 - pdg) >= o.min_weight;
    if (lane == 0) {
        o.keep[g] = keep ? 1 : 0;
        if (sw_r == 0 && sum_pd != 0.0) o.redo[atomicAdd(o.redo_n, 1)] = (int32_t)g;
        if (keep && !nd_write) o.ndfill[atomicAdd(o.ndfill_n, 1)] = (int32_t)g;
    }
}

template <typename T, typename A = double>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(SCPHD_FIT_WAVES, SCPHD_FIT_WAVES))) void k_fit(
    FitKernArgs<T> ka) {
    __shared__ FitShared<A> sh[16];
    const int w = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (w >= ka.a.n_waves) return;
    const int p = ((cint_t*)ka.a.wave_parent)[w];
    if (p < 0) return;
    cint_t* off = (cint_t*)ka.a.goff + p;
    const int k = 4 * (w - first_wave(off[0], p)) + ((threadIdx.x & 63) >> 4);
    if (k >= off[1] - off[0]) return; /* whole rows; rows never exchange data */
    const int64_t g = off[0] + k;
    const T* const from = ka.src.block(ka.a.gblock[g]);
    T* const to = ka.dst.block(ka.a.nd_base + g);
    const FitArgs& a = kernarg_late<FitArgs>();
    const ParentCtx pc(a.pose, a.meas, a.rig_meas, a.key, a.pstep, p);
    fit_row<T, A>(a, pc, g, k, from, to, sh[threadIdx.x >> 4]);
}

/* The non-detection clouds of the terms k_fit decided only after its sweep
 * and kept, listed in ndfill[0, *ndfill_n): the predicted samples and the
 * weights 1 - pd_i, the same bits as in the sweep.  One 16-lane
 * row per listed term; workgroups stride over the list (its length is read
 * on the device). */
template <typename T, bool RG, typename A = double>
__global__ __launch_bounds__(256) void k_nd_fill(FitArgs a, Clouds<T> src, Clouds<T> dst) {
    constexpr bool F32 = std::is_same_v<A, float>;
    const int lane = threadIdx.x & 15;
    const int n = *a.ndfill_n;
    const int stride = gridDim.x * 16;
    for (int i = blockIdx.x * 16 + (threadIdx.x >> 4); i < n; i += stride) {
        const int64_t g = a.ndfill[i];
        const int p = a.gparent[g];
        const int k = (int)(g - a.goff[p]);
        int pl;
        const auto kk = row_key<RG>(a.key, p, pl);
        const RowMeas<RG> rm(a.meas, a.rig_meas, a.key, p);
        const DisparityMeasurementModel& meas = rm.m;
        const T* from = src.block(a.gblock[g]);
        T* to = dst.block(a.nd_base + g);
        const CameraPose pose = load_pose(a.pose, p);
        SampleCtxF cx;
        if constexpr (F32) cx = SampleCtxF{meas_f(meas), pose_f(pose), motion_f(a.feat, a.dt)};
        /* four steps' loads issued before their arithmetic; the four steps
         * are one noise group (phase j) */
        FeatureCarry fc;
        for (int s0 = 0; s0 < a.S; s0 += 64) {
            T r[4][7];
#pragma unroll
            for (int j = 0; j < 4; ++j) load_step(from + 7 * (s0 + 16 * j), a.S - s0 - 16 * j, lane, r[j]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int s = s0 + 16 * j + lane;
                if (s < a.S) {
                    T* const o = to + 7 * (s - lane) + lane;
                    const int w = min(a.S - s0 - 16 * j, 16);
                    bool in;
                    if constexpr (F32) {
                        float x[6], q[6], sw;
                        eval_sample_f(a, cx, r[j], kk, pl, k, s, x, q, in, sw, &fc, (uint32_t)j);
#pragma unroll
                        for (int c = 0; c < 6; ++c) o[c * w] = (T)x[c];
                    } else {
                        EuclideanPoint x;
                        DisparityPoint d;
                        double sw;
                        eval_sample(a, meas, r[j], kk, pl, k, s, pose, sums_xy(s0 + 16 * j, whole_triples(a.S)), x, d,
                                    in, sw, &fc, (uint32_t)j);
                        const double xs[6] = {x.x, x.y, x.z, x.vx, x.vy, x.vz};
#pragma unroll
                        for (int c = 0; c < 6; ++c) o[c * w] = (T)xs[c];
                    }
                    o[6 * w] = (T)(1.0 - (in ? meas.pd() : 0.0));
                }
            }
        }
    }
}

/* The rare case of k_fit, one row per listed Gaussian (redo[0, *redo_n)):
 * every weight zero.  Refitted by two sweeps with unit weights (mean = sum
 * of the samples, as the reference's normalisation of an all-zero cloud
 * gives).  Workgroups stride over the list (its length is read on the
 * device). */
template <typename T, bool RG, typename A = double>
__global__ __launch_bounds__(256) void k_fit_fix(FitArgs a, Clouds<T> src, Clouds<T> dst) {
    constexpr bool F32 = std::is_same_v<A, float>;
    const int lane = threadIdx.x & 15;
    const int nredo = *a.redo_n;
    const int S = a.S;
    for (int i = blockIdx.x * 16 + (threadIdx.x >> 4); i < nredo; i += gridDim.x * 16) {
        const int64_t g = a.redo[i];
        const int p = a.gparent[g];
        const int k = (int)(g - a.goff[p]);
        int pl;
        const auto kk = row_key<RG>(a.key, p, pl);
        const RowMeas<RG> rm(a.meas, a.rig_meas, a.key, p);
        const DisparityMeasurementModel& meas = rm.m;
        const T* from = src.block(a.gblock[g]);
        const CameraPose pose = load_pose(a.pose, p);
        SampleCtxF cx;
        if constexpr (F32) cx = SampleCtxF{meas_f(meas), pose_f(pose), motion_f(a.feat, a.dt)};
        /* the sample's disparity-space point in the arithmetic type */
        auto point = [&](int s, A q[6]) {
            T r[7];
            load_sample<T>(from, S, s, r);
            if constexpr (F32) {
                float x[6], w;
                bool in;
                eval_sample_f(a, cx, r, kk, pl, k, s, x, q, in, w);
            } else {
                EuclideanPoint x;
                DisparityPoint d;
                bool in;
                double w;
                eval_sample(a, meas, r, kk, pl, k, s, pose, false, x, d, in, w); /* a fit of its own: one order */
                q[0] = d.u; q[1] = d.v; q[2] = d.d; q[3] = d.vu; q[4] = d.vv; q[5] = d.vd;
            }
        };
        A sq[6] = {0, 0, 0, 0, 0, 0};
        for (int s0 = 0; s0 < S; s0 += 16) {
            const int s = s0 + lane;
            if (s < S) {
                A q[6];
                point(s, q);
#pragma unroll
                for (int c = 0; c < 6; ++c) sq[c] += q[c];
            }
        }
        A muA[6], cc[21];
        double mu[6], P[21];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            muA[c] = row_sum16(sq[c]);
            mu[c] = (double)muA[c];
        }
#pragma unroll
        for (int e = 0; e < 21; ++e) cc[e] = 0;
        for (int s0 = 0; s0 < S; s0 += 16) {
            const int s = s0 + lane;
            if (s < S) {
                A q[6], dv[6];
                point(s, q);
#pragma unroll
                for (int c = 0; c < 6; ++c) dv[c] = q[c] - muA[c];
#pragma unroll
                for (int r = 0; r < 6; ++r)
#pragma unroll
                    for (int c = 0; c <= r; ++c) cc[pidx(r, c)] += dv[r] * dv[c];
            }
        }
        const double W = (double)S, W2 = (double)S;
        const double scale = (W * W + W2) / W;
#pragma unroll
        for (int e = 0; e < 21; ++e) P[e] = (double)row_sum16(cc[e]) * scale;
        const double pdg = a.fit[(int64_t)FP_PD * a.Ng + g];
        write_fit(a, g, lane, mu, P, pdg);
    }
}

/* Measurement-independent detection terms of each fitted Gaussian
 * (computeDetectionsKernel, src/kernels.cu:492-598): innovation covariance,
 * gain, Joseph covariance and its PD test, log(pd) + log(w), log det. */
__global__ __launch_bounds__(128) void k_precompute(const double* fit, const double* gw, int64_t Ng, double var_u,
                                                    double var_v,
                             double* pre, double* lik) {
    /* each Gaussian's records are formed by its thread, then written by the
     * workgroup through LDS as one contiguous stretch (records of
     * consecutive Gaussians are adjacent), so that the stores coalesce */
    __shared__ double stage[128 * 21];
    const int t = threadIdx.x;
    const int64_t g0 = (int64_t)blockIdx.x * 128;
    const int64_t g = g0 + t;
    const int nb = (int)min((int64_t)128, Ng - g0);
    const bool act = g < Ng;
    DetectionTerms r;
    bool ok = false;
    double pdg = 0.0, mu[6];
    if (act) {
        double P[21];
#pragma unroll
        for (int e = 0; e < 21; ++e) P[e] = fit[(FP_P + e) * Ng + g];
        detection_terms(P, var_u, var_v, r);
        ok = is_pd6(r.Pn);
        pdg = fit[FP_PD * Ng + g];
#pragma unroll
        for (int c = 0; c < 6; ++c) mu[c] = fit[(FP_MU + c) * Ng + g];
    }
    /* out[g0 L ..) <- the block's L-double records */
    auto put = [&](double* out, int L) {
        __syncthreads();
        for (int e = t; e < nb * L; e += 128) out[g0 * L + e] = stage[e];
    };
    if (act) {
        double* rec = stage + t * LK_COUNT;
        rec[LK_MUU] = mu[0];
        rec[LK_MUV] = mu[1];
        rec[LK_S0] = r.s0;
        rec[LK_S12] = r.s1 + r.s2;
        rec[LK_S3] = r.s3;
        rec[LK_C] = safe_log(pdg) + safe_log(gw[g]);
        rec[LK_H] = 0.5 * safe_log(r.det);
        rec[LK_OK] = ok ? 1.0 : 0.0;
    }
    put(lik, LK_COUNT);
    __syncthreads();
    if (act) {
        double* mk = stage + t * PP_MK_LEN;
#pragma unroll
        for (int c = 0; c < 6; ++c) mk[c] = mu[c];
#pragma unroll
        for (int k = 0; k < 12; ++k) mk[6 + k] = r.K[k];
    }
    put(pre + PP_MK * Ng, PP_MK_LEN);
    __syncthreads();
    if (act) {
#pragma unroll
        for (int e = 0; e < 21; ++e) stage[t * 21 + e] = r.Pn[e];
    }
    put(pre + PP_PN * Ng, 21);
}

/* ------------------------------------------- normalisers and survivors */
/* Likelihood records read through the constant address space: their
 * address is the same in every lane (one Gaussian, all measurements), so
 * the reads are scalar loads into SGPRs, with no LDS staging and no
 * per-lane copies.  Scalar loads return out of order, so every use waits
 * for all of them: records come four at a time, one wait per four (the
 * record buffer holds three records of padding past the last Gaussian). */
typedef __attribute__((address_space(4))) const double lik_t;

struct Lik4 {
    double v[4][LK_COUNT];
};

__device__ inline Lik4 load_lik4(const double* lik, int64_t g) {
    lik_t* r = (lik_t*)(lik + g * LK_COUNT);
    Lik4 x;
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int q = 0; q < LK_COUNT; ++q) x.v[k][q] = r[k * LK_COUNT + q];
    return x;
}

/* log weight of the detection term of Gaussian record r and measurement
 * (zu, zv): log pd + log w - dist/2 - log 2 pi - log det / 2
 * (src/kernels.cu:527-539); log(0) when the updated covariance is not PD
 * (:597-598).  The fused multiply-adds are written out, so that every place
 * that evaluates a term gets the same bits. */
static constexpr double LOG_2PI = 1.8378770664093453;
__device__ inline double det_lw(const double* r, double zu, double zv) {
    const double i0 = zu - r[LK_MUU], i1 = zv - r[LK_MUV];
    /* one order of the three products in every kernel: a weight that is the
     * same to the last bit sorts the same */
    const double dist = fma(i1 * i1, r[LK_S3], fma(i0 * i0, r[LK_S0], i0 * i1 * r[LK_S12]));
    const double lw = fma(-0.5, dist, r[LK_C]) - LOG_2PI - r[LK_H];
    return r[LK_OK] != 0.0 ? lw : SCPHD_LOG0;
}

/* e^x for -746 < x <= 0, the normaliser's terms (within 1 ulp of a
 * correctly rounded exp): x = k ln2 + r with |r| <= ln2/2 by Cody and
 * Waite's two-part reduction (ln2 split so that k ln2_hi is exact), e^r by
 * its Taylor polynomial to degree 13 (truncation below 5e-18 relative) in
 * Horner form, scaled by 2^k (gradual underflow below 2^-1022).  Cheaper
 * than the general exp, which also handles overflow and special values. */
__device__ inline double exp_nonpos(double x) {
    const double k = rint(x * 1.4426950408889634);
    const double r = fma(k, -1.90821492927058770002e-10, fma(k, -6.93147180369123816490e-01, x));
    double p = 1.6059043836821613e-10; /* 1/13! */
    p = fma(p, r, 2.08767569878681e-09);
    p = fma(p, r, 2.505210838544172e-08);
    p = fma(p, r, 2.755731922398589e-07);
    p = fma(p, r, 2.7557319223985893e-06);
    p = fma(p, r, 2.48015873015873e-05);
    p = fma(p, r, 0.0001984126984126984);
    p = fma(p, r, 0.001388888888888889);
    p = fma(p, r, 0.008333333333333333);
    p = fma(p, r, 0.041666666666666664);
    p = fma(p, r, 0.16666666666666666);
    p = fma(p, r, 0.5);
    p = fma(p, r, 1.0);
    p = fma(p, r, 1.0);
    return ldexp(p, (int)k);
}

/* order-preserving map of a double to unsigned (for LDS atomic maxima) */
__device__ inline unsigned long long max_key(double x) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    return b >> 63 ? ~b : b | (1ull << 63);
}
__device__ inline double max_val(unsigned long long k) {
    return __longlong_as_double((long long)(k >> 63 ? k & ~(1ull << 63) : ~k));
}

/* A round's measurements by bin of v: the places of bin b are off[b] ..
 * off[b + 1] - 1. */
static constexpr int ETA_BINS = 128, ETA_CHUNK = 2048;
struct EtaBins {
    double scale;
    int* off; /* ETA_BINS + 1, LDS */
    int* cur; /* ETA_BINS, LDS */
    __device__ EtaBins(const EtaArgs& a, int rig, int* o, int* c)
        : scale(ETA_BINS / fabs(a.rig_meas ? a.rig_meas[rig].img_height() : a.img_height)), off(o), cur(c) {}
    /* monotone in v, a NaN's the first */
    __device__ int of(double v) const { return (int)fmin(fmax(v * scale, 0.0), (double)(ETA_BINS - 1)); }
    /* fills the bins; returns the place of this thread's measurement (at v,
     * when `valid`).  Begins with a barrier; off is whole after it. */
    __device__ int fill(bool valid, double v) const {
        const int t = threadIdx.x, b = of(v);
        __syncthreads();
        if (t < ETA_BINS) cur[t] = 0;
        __syncthreads();
        if (valid) atomicAdd(&cur[b], 1);
        __syncthreads();
        if (t < 64) { /* exclusive offsets, two bins a lane */
            const int c0 = cur[2 * t], c1 = cur[2 * t + 1];
            int x = c0 + c1;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(x, o, 64);
                if (t >= o) x += y;
            }
            off[2 * t] = cur[2 * t] = x - c0 - c1;
            off[2 * t + 1] = cur[2 * t + 1] = x - c1;
            if (t == 63) off[ETA_BINS] = x;
        }
        __syncthreads();
        return valid ? atomicAdd(&cur[b], 1) : 0;
    }
    /* the places [q0, q1) of the measurements that Gaussian record r may give
     * l > L, or with `all` every one it may give any; the margins cover the
     * rounding of l and of the window */
    __device__ void window(const double* r, double L, bool all, int& q0, int& q1) const {
        q0 = q1 = 0;
        if (r[LK_OK] == 0.0) return;
        const double ub = r[LK_C] - LOG_2PI - r[LK_H], over = ub - L + 1e-6 * (1.0 + fabs(ub));
        if (!(over > 0.0)) return;
        const double c = 0.5 * r[LK_S12], det = r[LK_S0] * r[LK_S3] - c * c;
        const double hw = sqrt(2.000002 * over * (r[LK_S0] / det)) * 1.000001 + 1e-12 * fabs(r[LK_MUV]);
        if (all || !(det > 1e-9 * r[LK_S0] * r[LK_S3]) || !(hw < 1e300) || r[LK_MUV] != r[LK_MUV]) {
            q1 = off[ETA_BINS]; /* near singular: every measurement */
        } else {
            q0 = off[of(r[LK_MUV] - hw)];
            q1 = off[of(r[LK_MUV] + hw) + 1];
        }
    }
};

/* the record of entry j of the map from g0 on */
__device__ inline void load_rec(const EtaArgs& a, int64_t g0, int j, double* r) {
    const double* rec = a.lik + (g0 + j) * LK_COUNT;
#pragma unroll
    for (int q = 0; q < LK_COUNT; ++q) r[q] = rec[q];
}

/* Per parent: eta_{p,m} = log( sum_g exp(lw_{g,m}) + M w0 + kappa ) for
 * every measurement (normaliser reduce_by_key + log_sum_exp,
 * src/scphdcameracalibration.cu:1729-1768, exact per-parent segments), the
 * single-cluster log-likelihood sum_m eta + sum_g w_g (:1813-1849), and the
 * detection terms whose normalised weight reaches min_weight, listed in pack
 * order and counted with the birth terms that reach it (updateKernel's prune
 * flag, src/kernels.cu:608-659).
 *
 * One workgroup per parent; 256 measurements a round.  A term matters to a
 * measurement only within a few standard deviations of it: with
 * l <= C - log 2 pi - H - dist/2 and dist >= dv^2 / S_vv (the marginal of
 * the quadratic form), l > L needs dv^2 <= 2 (C - log 2 pi - H - L) S_vv.
 * So the round's measurements are put in bins of v (a measurement's place is
 * its rank by bin), and a Gaussian meets those of the bins its window covers:
 *   1. l > bpc (L = bpc; no other term can move the maximum off bpc): few
 *      Gaussians and few measurements each, a Gaussian a lane, an atomic
 *      maximum per measurement;
 *   2. l > max - 60 (L = bpc - 60; all terms below exp(-60) of the largest
 *      add up to 1.8e-23 at most, for 2048 of them: less than a quarter of an
 *      ulp of eta where |eta| > 4e-7, and nearer to 0 far below the rounding
 *      of max itself, a sum of terms about 1 to 10): about 30 measurements a
 *      Gaussian, but all of them for a few, so a wavefront takes a Gaussian
 *      at a time against its measurements in blocks of 64, held in registers,
 *      and collects a word of the measurements' masks, 32 Gaussians, in
 *      registers too;
 *   3. the masks' terms (about 20 a measurement, up to 130) are listed by
 *      measurement and then map index, evaluated a lane each, and summed per
 *      measurement in that order, ascending in g: the oracle's.  Terms that
 *      can no longer be kept leave the mask;
 *   4. the rest are listed, evaluated against eta, and those kept written
 *      in list order, which is the pack order.
 * Gaussians go in chunks of the mask's 2048 bits in 2 and 3; the list (4) of
 * a map of more than one chunk is k_eta_list's.
 *
 * Bound: latency (LDS and the records' gathers), which is why the lists
 * spread the uneven terms over all lanes.  Ten frames of 4096 parents, 200
 * landmarks: 18.0 ms when every pair was evaluated twice and measurements
 * with more than eight candidate terms (one in seven) swept the map again,
 * 9.6 so. */
static constexpr double ETA_DROP = 60.0;

__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(3))) void k_eta(EtaArgs a) {
    constexpr int REC = 6; /* of a record, what step 2 needs */
    __shared__ double red[16];
    __shared__ int sh[8];
    __shared__ double s_zu[NT], s_zv[NT];    /* the round's measurements by place */
    __shared__ uint16_t s_m[NT];             /* the measurement at a place */
    __shared__ unsigned long long s_max[NT]; /* per measurement: its maximum's key; then eta's bits */
    __shared__ unsigned long long s_any[NT]; /* per place: its mask's non-zero words */
    __shared__ int s_cnt[NT];                /* per measurement: terms kept */
    __shared__ int s_off[ETA_BINS + 1], s_cur[ETA_BINS];
    /* a.list terms of a list: place << 16 | map index in the chunk, and in the
     * same place then exp(l - max); in step 2 the wavefronts' records of a
     * word of Gaussians.  Then per place a.mask_stride words of its mask. */
    extern __shared__ double s_dyn[];
    double* const s_e = s_dyn;
    uint32_t* const s_pair = (uint32_t*)s_dyn;
    uint32_t* const s_mask = (uint32_t*)(s_dyn + a.list);
    const int p = blockIdx.x;
    const int t = threadIdx.x, lane = t & 63;
    const int64_t g0 = a.goff[p];
    const int G = a.goff[p + 1] - a.goff[p];
    const bool lists = !a.no_lists && G <= ETA_CHUNK;
    double eta_sum = 0.0;
    int cnt = 0, kept = 0;
    /* this parent's measurement set: its rig's in an ensemble */
    const int rig = a.moff ? a.prig[p] : 0;
    const int M = a.moff ? a.moff[rig + 1] - a.moff[rig] : a.M;
    const int64_t zb = a.moff ? a.moff[rig] : 0;
    const double bpc = a.bpcs ? a.bpcs[rig] : a.bpc;
    const double logw0 = a.births[rig].logw0;
    const bool birth_ok = a.births[rig].pd_ok != 0;
    const int rounds = (M + NT - 1) / NT;
    const EtaBins bins(a, rig, s_off, s_cur);
    /* candidates: terms with l - max above the gate (less 1e-6), the only
     * ones that can pass it against eta >= max */
    const double cgate = a.lw_gate - 1e-6;
    const double drop = fmax(ETA_DROP, -cgate); /* no candidate is dropped */
    for (int r = 0; r < rounds; ++r) {
        const int m = r * NT + t;
        const bool valid = m < M;
        const double zu = valid ? a.zu[zb + m] : 0.0, zv = valid ? a.zv[zb + m] : 0.0;
        const int64_t pm = (int64_t)p * a.M + m;
        const int place = bins.fill(valid, zv);
        s_max[t] = max_key(bpc);
        s_cnt[t] = 0;
        if (valid) {
            s_zu[place] = zu;
            s_zv[place] = zv;
            s_m[place] = (uint16_t)t;
        }
        __syncthreads();
        /* 1. maxima */
        for (int j = t; j < G; j += NT) {
            double rec[LK_COUNT];
            load_rec(a, g0, j, rec);
            int q, q1;
            for (bins.window(rec, bpc, a.sweep != 0, q, q1); q < q1; ++q) {
                const double l = det_lw(rec, s_zu[q], s_zv[q]);
                if (l > bpc) atomicMax(&s_max[s_m[q]], max_key(l));
            }
        }
        __syncthreads();
        /* eta = mx + log1p(sum of the other terms' exp(l - mx)), mx the
         * first maximum of (bpc, l_0, ...), terms summed g ascending then
         * bpc: the normaliser definition the oracle uses bit for bit */
        const double mx = max_val(s_max[t]);
        bool met = !(mx > bpc); /* the maximum's own term (1, not summed) */
        double T = 0.0;
        const int nq = s_off[ETA_BINS];
        /* the terms in this thread's row of the masks from (words, bits) on,
         * ascending: fills the list's places up to `end` from `pos` on */
        unsigned long long words_left = 0;
        uint32_t bits_left = 0;
        int word = 0;
        auto row_begin = [&]() { /* and their number */
            words_left = valid ? s_any[place] : 0;
            bits_left = 0;
            int n = 0;
            for (unsigned long long w = words_left; w; w &= w - 1)
                n += __popc(s_mask[place * a.mask_stride + __builtin_ctzll(w)]);
            return n;
        };
        auto row_list = [&](int& pos, int end) {
            while (pos < end) {
                if (!bits_left) {
                    if (!words_left) return;
                    word = __builtin_ctzll(words_left);
                    words_left &= words_left - 1;
                    bits_left = s_mask[place * a.mask_stride + word];
                    continue;
                }
                s_pair[2 * (pos & (a.list - 1))] =
                    (uint32_t)place << 16 | (uint32_t)(32 * word + __builtin_ctz(bits_left));
                bits_left &= bits_left - 1;
                ++pos;
            }
        };
        for (int c0 = 0; c0 < G; c0 += ETA_CHUNK) {
            const int cn = min(ETA_CHUNK, G - c0), words = (cn + 31) / 32;
            s_any[t] = 0;
            /* 2. block k: the measurements at places 64 k + lane; a pair hits
             * when 2 ub - dist > lim (never at a place without one) */
            double bu[4], bv[4], lim[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int q = 64 * k + lane;
                bu[k] = bv[k] = 0.0;
                lim[k] = INFINITY;
                if (q < nq) {
                    bu[k] = s_zu[q];
                    bv[k] = s_zv[q];
                    lim[k] = 2.0 * (max_val(s_max[s_m[q]]) - drop);
                }
            }
            __syncthreads();
            for (int w = __builtin_amdgcn_readfirstlane(t >> 6); w < words; w += NT / 64) {
                const int jw = c0 + 32 * w, n = min(32, c0 + cn - jw);
                double* const wr = s_dyn + (t >> 6) * (32 * REC);
                /* the word's windows, a Gaussian a lane: blocks met */
                int blocks = 0;
                if (lane < n) {
                    double rec[LK_COUNT];
                    load_rec(a, g0, jw + lane, rec);
                    int q0, q1;
                    bins.window(rec, bpc - drop, a.sweep != 0, q0, q1);
                    if (q0 < q1) blocks = (2 << ((q1 - 1) >> 6)) - (1 << (q0 >> 6));
                    const double ub = rec[LK_C] - LOG_2PI - rec[LK_H];
                    wr[lane * REC] = rec[LK_MUU];
                    wr[lane * REC + 1] = rec[LK_MUV];
                    wr[lane * REC + 2] = rec[LK_S0];
                    wr[lane * REC + 3] = rec[LK_S12];
                    wr[lane * REC + 4] = rec[LK_S3];
                    wr[lane * REC + 5] = 2.0 * ub + 2e-6 * (1.0 + fabs(ub));
                }
                wave_lds_fence();
                uint32_t bits[4] = {0, 0, 0, 0};
#pragma unroll 4
                for (int b = 0; b < n; ++b) {
                    const int met_blocks = __builtin_amdgcn_readlane(blocks, b);
                    double rec[REC];
#pragma unroll
                    for (int q = 0; q < REC; ++q) rec[q] = wr[b * REC + q];
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (met_blocks >> k & 1) {
                            const double i0 = bu[k] - rec[0], i1 = bv[k] - rec[1];
                            const double dist = fma(i1 * i1, rec[4], fma(i0 * i1, rec[3], i0 * i0 * rec[2]));
                            if (rec[5] - dist > lim[k]) bits[k] |= 1u << b;
                        }
                }
                wave_lds_fence();
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int q = 64 * k + lane;
                    if (q < nq) {
                        s_mask[q * a.mask_stride + w] = bits[k];
                        if (bits[k]) atomicOr(&s_any[q], 1ull << w);
                    }
                }
            }
            __syncthreads();
            /* 3. the terms' values, and their sum */
            int total, n = row_begin();
            const int first = block_exscan(n, sh, &total);
            int pos = first;
            for (int l0 = 0; l0 < total; l0 += a.list) {
                row_list(pos, l0 + a.list);
                __syncthreads();
                const int ln = min(a.list, total - l0);
                for (int q = t; q < ln; q += NT) {
                    const uint32_t pr = s_pair[2 * q];
                    const int pl = (int)(pr >> 16), j = (int)(pr & 0xFFFFu);
                    double rec[LK_COUNT];
                    load_rec(a, g0, c0 + j, rec);
                    const double x = det_lw(rec, s_zu[pl], s_zv[pl]) - max_val(s_max[s_m[pl]]);
                    s_e[q] = x > -746.0 ? exp_nonpos(x) : 0.0;
                    if (!(x > cgate)) atomicAnd(&s_mask[pl * a.mask_stride + (j >> 5)], ~(1u << (j & 31)));
                }
                __syncthreads();
                const int q1 = min(first + n - l0, ln);
                for (int q = max(first - l0, 0); q < q1; ++q) {
                    const double e = s_e[q];
                    if (!met && e == 1.0)
                        met = true;
                    else
                        T += e;
                }
                __syncthreads();
            }
        }
        if (mx > bpc) T += exp(bpc - mx);
        const double eta = mx + log1p(T);
        s_max[t] = (unsigned long long)__double_as_longlong(eta);
        if (valid) {
            a.eta[pm] = eta;
            eta_sum += eta;
            const double w = exp(logw0 - eta);
            cnt += (w >= a.min_weight && birth_ok) ? 1 : 0;
        }
        /* 4. the kept terms */
        if (lists && G > 0) {
            int total, n = row_begin();
            int pos = block_exscan(n, sh, &total);
            for (int l0 = 0; l0 < total; l0 += a.list) {
                row_list(pos, l0 + a.list);
                __syncthreads();
                constexpr int E = 4; /* consecutive terms of a thread */
                for (int b0 = 0; b0 < min(a.list, total - l0); b0 += E * NT) {
                    double w[E];
                    uint32_t pr[E];
                    int mine = 0;
#pragma unroll
                    for (int i = 0; i < E; ++i) {
                        const int q = b0 + E * t + i;
                        w[i] = -1.0; /* not kept */
                        pr[i] = 0;
                        if (l0 + q >= total) continue;
                        pr[i] = s_pair[2 * q];
                        const int pl = (int)(pr[i] >> 16), sl = s_m[pl];
                        double rec[LK_COUNT];
                        load_rec(a, g0, (int)(pr[i] & 0xFFFFu), rec);
                        const double x = det_lw(rec, s_zu[pl], s_zv[pl]) - __longlong_as_double((long long)s_max[sl]);
                        if (!(x > a.lw_gate)) continue;
                        const double wx = exp(x);
                        if (!(wx >= a.min_weight)) continue;
                        w[i] = wx;
                        ++mine;
                        atomicAdd(&s_cnt[sl], 1);
                    }
                    int kn;
                    int k = kept + block_exscan(mine, sh, &kn);
#pragma unroll
                    for (int i = 0; i < E; ++i)
                        if (w[i] >= 0.0) {
                            if (k < a.kcap) {
                                a.kw[p * a.kcap + k] = w[i];
                                *(int2*)(a.kjm + 2 * (p * a.kcap + k)) =
                                    int2{(int)(pr[i] & 0xFFFFu), r * NT + s_m[pr[i] >> 16]};
                            }
                            ++k;
                        }
                    kept += kn;
                }
                __syncthreads();
            }
            __syncthreads();
            if (valid) {
                a.mcnt[pm] = s_cnt[t];
                cnt += s_cnt[t];
            }
        } else if (valid && (a.no_lists || G == 0)) { /* no list: sweep the map */
            int mcnt = 0;
            for (int j0 = 0; j0 < G; j0 += 4) {
                const Lik4 R = load_lik4(a.lik, g0 + j0);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const double x = det_lw(R.v[q], zu, zv) - eta;
                    if (j0 + q < G && x > a.lw_gate && R.v[q][LK_OK] != 0.0) mcnt += exp(x) >= a.min_weight ? 1 : 0;
                }
            }
            a.mcnt[pm] = mcnt;
            cnt += mcnt;
        }
    }
    double swg = 0.0;
    int nd = 0;
    for (int j = t; j < G; j += NT) {
        swg += a.gw[g0 + j];
        nd += a.keep[g0 + j];
    }
    const double se = block_sum(eta_sum, red);
    const double sg = block_sum(swg, red);
    const double sc = block_sum((double)cnt, red);
    const double sn = block_sum((double)nd, red);
    if (t == 0) {
        a.loglik[p] = se + sg;
        a.nsurv[p] = (int32_t)sc;
        a.nkeep[p] = (int32_t)sn;
        a.knum[p] = lists && kept <= a.kcap ? kept : -1;
    }
}

/* The kept detection terms of the parents with more Gaussians than k_eta's
 * masks take (it has left their normalisers and birth terms), listed and
 * counted as it does.  One workgroup per parent, 256 measurements a round: a
 * Gaussian a lane meets the measurements that its window for the smallest
 * weight covers, and the terms kept go into LDS as they are found; then they
 * are put in pack order, by measurement (counts and offsets) and within one by
 * their rank in map index.  A round of more than LATE_LIST terms makes no
 * list, and k_survivors sweeps the map.
 *
 * Bound: latency of the few terms a lane meets.  Why a kernel of its own: the
 * terms wait for eta, by when k_eta's masks hold the last chunk only.
 * Normalisers and survivors of 256 parents, 2100 Gaussians and 200
 * measurements: 0.96 ms when k_eta's count and k_survivors each evaluated
 * every pair, 0.21 so; 64 parents, 8000 and 400: 5.9 and 1.1 ms. */
static constexpr int LATE_LIST = 4096;
struct LateList {
    double w[LATE_LIST];
    int32_t j[LATE_LIST];
    uint16_t slot[LATE_LIST]; /* measurement in the round */
    uint16_t by_m[LATE_LIST]; /* the terms, measurements ascending */
};

__global__ __launch_bounds__(NT) void k_eta_list(EtaArgs a) {
    __shared__ int sh[8];
    __shared__ double s_zu[NT], s_zv[NT], s_eta[NT]; /* by place */
    __shared__ uint16_t s_m[NT];
    __shared__ int s_cnt[NT], s_base[NT], s_fill[NT]; /* per measurement: terms kept, their offsets */
    __shared__ int s_off[ETA_BINS + 1], s_cur[ETA_BINS], s_n;
    extern __shared__ double s_dyn[];
    LateList& l = *(LateList*)s_dyn;
    const int p = blockIdx.x, t = threadIdx.x;
    const int64_t g0 = a.goff[p];
    const int G = a.goff[p + 1] - a.goff[p];
    if (G <= ETA_CHUNK) return;
    const int rig = a.moff ? a.prig[p] : 0;
    const int M = a.moff ? a.moff[rig + 1] - a.moff[rig] : a.M;
    const int64_t zb = a.moff ? a.moff[rig] : 0;
    const double bpc = a.bpcs ? a.bpcs[rig] : a.bpc;
    const EtaBins bins(a, rig, s_off, s_cur);
    const double L = bpc + a.lw_gate - 1e-6; /* eta >= bpc */
    int kept = 0;
    bool listed = true;
    for (int r = 0; r < (M + NT - 1) / NT; ++r) {
        const int m = r * NT + t;
        const bool valid = m < M;
        const int64_t pm = (int64_t)p * a.M + m;
        const double zv = valid ? a.zv[zb + m] : 0.0;
        const int place = bins.fill(valid, zv);
        s_cnt[t] = 0;
        if (t == 0) s_n = 0;
        if (valid) {
            s_zu[place] = a.zu[zb + m];
            s_zv[place] = zv;
            s_eta[place] = a.eta[pm];
            s_m[place] = (uint16_t)t;
        }
        __syncthreads();
        for (int j = t; j < G; j += NT) {
            double rec[LK_COUNT];
            load_rec(a, g0, j, rec);
            int q, q1;
            for (bins.window(rec, L, a.sweep != 0, q, q1); q < q1; ++q) {
                const double x = det_lw(rec, s_zu[q], s_zv[q]) - s_eta[q];
                if (!(x > a.lw_gate)) continue;
                const double w = exp(x);
                if (!(w >= a.min_weight)) continue;
                const int sl = s_m[q], i = atomicAdd(&s_n, 1);
                atomicAdd(&s_cnt[sl], 1);
                if (i < LATE_LIST) {
                    l.w[i] = w;
                    l.j[i] = j;
                    l.slot[i] = (uint16_t)sl;
                }
            }
        }
        __syncthreads();
        const int n = s_n;
        int tot;
        s_base[t] = s_fill[t] = block_exscan(s_cnt[t], sh, &tot);
        if (valid) a.mcnt[pm] = s_cnt[t];
        listed = listed && n <= LATE_LIST && kept + n <= a.kcap;
        if (listed) { /* uniform */
            __syncthreads();
            for (int i = t; i < n; i += NT) l.by_m[atomicAdd(&s_fill[l.slot[i]], 1)] = (uint16_t)i;
            __syncthreads();
            for (int i = t; i < n; i += NT) {
                const int sl = l.slot[i], j = l.j[i], e0 = s_base[sl], e1 = e0 + s_cnt[sl];
                int k = e0;
                for (int e = e0; e < e1; ++e) k += l.j[l.by_m[e]] < j ? 1 : 0;
                const int64_t o = p * a.kcap + kept + k;
                a.kw[o] = l.w[i];
                *(int2*)(a.kjm + 2 * o) = int2{j, r * NT + sl};
            }
        }
        kept += n;
    }
    if (t == 0) {
        a.nsurv[p] += kept;
        a.knum[p] = listed ? kept : -1;
    }
}

/* Writes the surviving detection terms (Kalman-updated mean, weight
 * exp(lw - eta)) and birth terms of every parent, compacted in the
 * reference's pack order (updateKernel, src/kernels.cu:608-659: detection
 * terms measurement-major, then births).  The detection terms come from
 * k_eta's list, one a thread, so that the gathers of their records are in
 * flight together, and the means go through LDS to be stored as one stretch.
 * Ten frames of 4096 parents, 200 landmarks: 11.9 ms when a thread found and
 * wrote its measurement's terms one after the other, 4.4 from the list with
 * each thread storing its 48 bytes, 1.9 so.  A parent without a list has its
 * map swept. */
__global__ __launch_bounds__(NT) void k_survivors(SurvArgs a) {
    __shared__ int sh[8];
    __shared__ double s_mu[6 * NT]; /* means, stored as one stretch */
    const EtaArgs& e = a.e;
    const int p = blockIdx.x;
    const int t = threadIdx.x;
    const int64_t g0 = e.goff[p];
    const int G = e.goff[p + 1] - e.goff[p];
    const int64_t base = a.survoff[p];
    const int cap = a.survoff[p + 1] - a.survoff[p];
    int run = 0;
    const int rig = e.moff ? e.prig[p] : 0;
    const BirthModel& birth = e.births[rig];
    const int M = e.moff ? e.moff[rig + 1] - e.moff[rig] : e.M;
    const int64_t zb = e.moff ? e.moff[rig] : 0;
    const int rounds = (M + NT - 1) / NT;
    /* survivor i: map entry j and measurement m (at zu, zv) with weight w */
    auto put = [&](int i, int j, int m, double zu, double zv, double w) {
        if (i >= cap) return;
        const int64_t so = base + i, gi = g0 + j;
        const double* mk = e.pre + PP_MK * e.Ng + gi * PP_MK_LEN;
        const double i0 = zu - mk[0], i1 = zv - mk[1];
        a.sw[so] = w;
        a.sg[so] = (int32_t)gi;
        a.sm[so] = m;
#pragma unroll
        for (int c = 0; c < 6; ++c) a.smu[so * 6 + c] = mk[c] + i0 * mk[6 + c] + i1 * mk[12 + c];
    };
    const int kn = e.knum[p];
    if (kn >= 0) {
        for (int i0 = 0; i0 < kn; i0 += NT) {
            const int i = i0 + t, n = min(min(NT, kn - i0), cap - i0);
            if (t < n) {
                const int2 jm = *(const int2*)(e.kjm + 2 * (p * e.kcap + i));
                const int64_t gi = g0 + jm.x;
                const double* mk = e.pre + PP_MK * e.Ng + gi * PP_MK_LEN;
                const double i0u = e.zu[zb + jm.y] - mk[0], i1v = e.zv[zb + jm.y] - mk[1];
                a.sw[base + i] = e.kw[p * e.kcap + i];
                a.sg[base + i] = (int32_t)gi;
                a.sm[base + i] = jm.y;
#pragma unroll
                for (int c = 0; c < 6; ++c) s_mu[6 * t + c] = mk[c] + i0u * mk[6 + c] + i1v * mk[12 + c];
            }
            __syncthreads();
            for (int q = t; q < 6 * n; q += NT) a.smu[(base + i0) * 6 + q] = s_mu[q];
            __syncthreads();
        }
        run = kn;
    } else {
        for (int r = 0; r < rounds; ++r) {
            const int m = r * NT + t;
            const bool valid = m < M;
            const double zu = valid ? e.zu[zb + m] : 0.0, zv = valid ? e.zv[zb + m] : 0.0;
            const double eta = valid ? e.eta[(int64_t)p * e.M + m] : 0.0;
            const int cnt = valid ? e.mcnt[(int64_t)p * e.M + m] : 0; /* detection terms kept, from k_eta */
            int tot;
            int o = run + block_exscan(cnt, sh, &tot);
            if (valid && cnt > 0)
                for (int j0 = 0; j0 < G; j0 += 4) {
                    const Lik4 R = load_lik4(e.lik, g0 + j0);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        /* kept when its normalised weight reaches min_weight
                         * (the gate first: exp(x) < min_weight below it) */
                        const double x = det_lw(R.v[q], zu, zv) - eta;
                        if (j0 + q >= G || !(x > e.lw_gate && R.v[q][LK_OK] != 0.0)) continue;
                        const double w = exp(x);
                        if (w >= e.min_weight) put(o++, j0 + q, m, zu, zv, w);
                    }
                }
            run += tot;
        }
    }
    for (int r = 0; r < rounds; ++r) {
        const int m = r * NT + t;
        const bool valid = m < M;
        const double eta = valid ? e.eta[(int64_t)p * e.M + m] : 0.0;
        const double w = valid ? exp(birth.logw0 - eta) : 0.0;
        const bool ok = valid && w >= e.min_weight && birth.pd_ok;
        int tot;
        const int o = run + block_exscan(ok ? 1 : 0, sh, &tot);
        if (ok && o < cap) {
            const int64_t so = base + o;
            a.sw[so] = w;
            a.sg[so] = -1 - rig;
            a.sm[so] = m;
            a.smu[(so) * 6 + 0] = e.zu[zb + m];
            a.smu[(so) * 6 + 1] = e.zv[zb + m];
#pragma unroll
            for (int c = 2; c < 6; ++c) a.smu[(so) * 6 + c] = birth.mean[c];
        }
        run += tot;
    }
    if (t == 0 && run != cap) *a.err = 1;
}

/* -------------------------------------------------------------- merging */
/* Workspace of one parent's round loop, U survivor slots (Up = next power of two):
 *   key_w double[Up]  sort keys;            ord   int[Up]   (weight desc, index asc) order
 *   bu, bv double[U]  mean u, v;            bs    double[3U] (u,v) covariance block uu uv vv
 *   flag  uint8[U]    merged;               selfm uint8[U]  member of its own group
 *   mem   int[U]      group members;        memb  uint8[U]  round membership */
__host__ __device__ inline int next_pow2(int x) {
    int v = 1;
    while (v < x) v <<= 1;
    return v;
}

struct MergeLayout {
    int64_t ord, bu, bv, bs, flag, selfm, mem, memb, bytes;
    __host__ __device__ explicit MergeLayout(int U) {
        const int64_t Up = next_pow2(U > 0 ? U : 1);
        ord = Up * 8;
        bu = (ord + Up * 4 + 7) & ~(int64_t)7;
        bv = bu + (int64_t)U * 8;
        bs = bv + (int64_t)U * 8;
        flag = bs + (int64_t)U * 24;
        selfm = flag + U;
        mem = (selfm + U + 7) & ~(int64_t)7;
        memb = mem + (int64_t)U * 4;
        bytes = (memb + U + 7) & ~(int64_t)7;
    }
};

/* global scratch for parents that do not fit in LDS: MergeLayout(U).bytes
 * <= 71 U + 32 since Up < 2 U, GroupsLayout's and the pairs 49 U + 344 */
static constexpr int MERGE_WS_PER_SLOT = 72, MERGE_WS_PER_PARENT = 512;

/* k_merge_groups' workspace of one parent, U survivor slots, in LDS or (BIG)
 * in global scratch.  The survivors in bins of u, while the candidates are
 * enumerated:
 *   u, v  double[U]  mean;  s  float[3U]  (u, v) covariance uu uv vv (uu < 0:
 *   ill-conditioned);  id  uint16[U]  survivor;  ill  uint16[U]  those ones
 * and in the same place, from the weight sort on:
 *   key   double[U]  weights; then nbr  uint16[ecap]  neighbour lists, ranks
 *   nbo   int[U+1]   list offsets;      cnt  int[U]  fill cursors, then groups
 *   ord   uint16[U]  survivor of a rank
 *   own   uint16[U]  rank of a survivor; then rank of a rank's leader
 *   st    uint8[U]   undecided, leader or member
 * and over both self uint8[U] (member of its own group).  The neighbour pairs
 * i << 16 | j, up to ecap / 2, go to global scratch. */
struct GroupsLayout {
    int64_t v, s, id, ill, bnbo, cnt, ord, own, st, self, bytes;
    __host__ __device__ explicit GroupsLayout(int U) {
        const int64_t n = U;
        v = 8 * n;
        s = 16 * n;
        id = 28 * n;
        ill = 30 * n;
        bnbo = 2 * (8 * n + 64);
        cnt = bnbo + 4 * (n + 1);
        ord = cnt + 4 * n; /* the bitonic sort's 12 next_pow2(U) < 24 U bytes end before it */
        own = ord + 2 * n;
        st = own + 2 * n;
        const int64_t b = st + n;
        self = 32 * n > b ? 32 * n : b;
        bytes = (self + n + 7) & ~(int64_t)7;
    }
};
static constexpr int GROUPS_PAIRS_PER_SLOT = 16, GROUPS_PAIRS_PER_PARENT = 128;

/* k_merge_groups' dynamic LDS for parents of up to U survivors, and the
 * largest U of which two workgroups fit a CU and of which one does (160 KB,
 * of which the kernel's own arrays take 13 each) */
int groups_lds_bytes(int U) { return (int)GroupsLayout(std::max(U, 0)).bytes; }
static constexpr int GROUPS_CAP2 = 2048, GROUPS_CAP1 = 4352;

int merge_lds_bytes(int cap) { return (int)MergeLayout(cap).bytes; }

int64_t merge_scratch_bytes(int64_t Stot, int Np, MergeArgs* a, bool big) {
    const int slot = big ? MERGE_WS_PER_SLOT : GROUPS_PAIRS_PER_SLOT;
    const int parent = big ? MERGE_WS_PER_PARENT : GROUPS_PAIRS_PER_PARENT;
    if (a) {
        a->ws_slot = slot;
        a->ws_parent = parent;
    }
    return Stot * slot + (int64_t)Np * parent + 256;
}

/* Packed covariance entry e of a survivor's term: the updated covariance of
 * table entry g, or (g = -1 - r < 0) the birth covariance of rig r.  Both
 * live in global memory, so the choice is one global load from a chosen
 * address. */
__device__ inline double term_P(const MergeArgs& a, int g, int e) {
    return g >= 0 ? a.pre[(int64_t)PP_PN * a.Ng + (int64_t)g * 21 + e] : a.births[-1 - g].P[e];
}

/* all of them (a pointer chosen once: 16-byte loads) */
__device__ inline const double* term_P_all(const MergeArgs& a, int g) {
    return g >= 0 ? a.pre + (int64_t)PP_PN * a.Ng + (int64_t)g * 21 : a.births[-1 - g].P;
}

__device__ inline void survivor_P(const MergeArgs& a, int64_t si, double* P) {
    const double* o = term_P_all(a, a.sg[si]);
#pragma unroll
    for (int e = 0; e < 21; ++e) P[e] = o[e];
}

__device__ inline void survivor_mu(const MergeArgs& a, int64_t si, double* mu) {
#pragma unroll
    for (int c = 0; c < 6; ++c) mu[c] = a.smu[(si) * 6 + c];
}

/* Workspace pointers of one parent's round loop. */
struct MergeWs {
    double* key_w;
    int* ord;
    double* bu;
    double* bv;
    double* bs;
    uint8_t* flag;
    uint8_t* selfm;
    int* mem;
    uint8_t* memb;
    __device__ MergeWs(char* ws, int U) {
        const MergeLayout ly(U);
        key_w = (double*)ws;
        ord = (int*)(ws + ly.ord);
        bu = (double*)(ws + ly.bu);
        bv = (double*)(ws + ly.bv);
        bs = (double*)(ws + ly.bs);
        flag = (uint8_t*)(ws + ly.flag);
        selfm = (uint8_t*)(ws + ly.selfm);
        mem = (int*)(ws + ly.mem);
        memb = (uint8_t*)(ws + ly.memb);
    }
};

/* Can survivors i and j be merge partners?  The (u, v) marginal of the
 * squared Mahalanobis distance with Sigma = P_i + P_j is a lower bound of
 * the full 6-D distance for positive-definite Sigma (and a non-PD Sigma
 * never merges), so a pair is rejected when the marginal exceeds the
 * threshold by 0.1 %; an ill-conditioned (u, v) block is never rejected. */
__device__ inline bool merge_bound(const MergeWs& w, int i, int j, double thr) {
    const double du = w.bu[j] - w.bu[i], dv = w.bv[j] - w.bv[i];
    const double suu = w.bs[3 * i] + w.bs[3 * j];
    const double suv = w.bs[3 * i + 1] + w.bs[3 * j + 1];
    const double svv = w.bs[3 * i + 2] + w.bs[3 * j + 2];
    const double det = suu * svv - suv * suv;
    if (!(det > 1e-6 * suu * svv)) return true;
    const double q = svv * du * du - 2.0 * suv * du * dv + suu * dv * dv;
    return !(q > 1.001 * thr * det);
}

/* Merge membership of survivors i and j: squared Mahalanobis distance with
 * Sigma = P_i + P_j below min_separation (computeMahalDist,
 * src/device_math.cu:374-453).  The computed value is symmetric in i and j
 * to the last bit (the sum P_i + P_j commutes and negating the difference
 * negates every forward-substitution term). */
__device__ inline bool merge_full(const MergeArgs& a, int64_t sbase, int i, int j, double thr) {
    double mi[6], mj[6], Pi[21], Pj[21];
    survivor_mu(a, sbase + i, mi);
    survivor_mu(a, sbase + j, mj);
    survivor_P(a, sbase + i, Pi);
    survivor_P(a, sbase + j, Pj);
    return mahal6(mi, Pi, mj, Pj) < thr;
}

__device__ inline bool merge_pair(const MergeArgs& a, int64_t sbase, const MergeWs& w, int i, int j, double thr) {
    return merge_bound(w, i, j, thr) && merge_full(a, sbase, i, j, thr);
}

/* Bitonic sort of ord[0, Up) by descending key with ascending index on
 * ties.  Padding slots carry keys that sort last.  Ends with a barrier. */
__device__ inline void merge_bitonic(double* key, int* ord, int Up) {
    const int t = threadIdx.x;
    __syncthreads();
    for (int k = 2; k <= Up; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = t; i < Up; i += NT) {
                const int l = i ^ j;
                if (l > i) {
                    const double wi = key[i], wl = key[l];
                    const int ii = ord[i], il = ord[l];
                    const bool l_before_i = (wl > wi) || (wl == wi && il < ii);
                    const bool asc = (i & k) == 0;
                    if (asc == l_before_i) {
                        key[i] = wl;
                        key[l] = wi;
                        ord[i] = il;
                        ord[l] = ii;
                    }
                }
            }
            __syncthreads();
        }
    }
}

/* Sort one parent's survivors by (weight desc, index asc) into ord, the
 * order in which the reference's argmax loop picks leaders (ties: lowest
 * pack index). */
__device__ inline void merge_sort_w(const MergeArgs& a, int64_t sbase, int U, double* key, int* ord) {
    const int t = threadIdx.x;
    const int Up = next_pow2(U);
    __syncthreads();
    for (int i = t; i < Up; i += NT) {
        key[i] = i < U ? a.sw[sbase + i] : -INFINITY;
        ord[i] = i < U ? i : 0x7fffffff;
    }
    merge_bitonic(key, ord, Up);
}

/* The round loop's start: the (u, v) marginals, no survivor merged, and the
 * order by weight. */
__device__ inline void merge_load_sort(const MergeArgs& a, int64_t sbase, int U, MergeWs& w) {
    for (int i = threadIdx.x; i < U; i += NT) {
        w.bu[i] = a.smu[(sbase + i) * 6 + 0];
        w.bv[i] = a.smu[(sbase + i) * 6 + 1];
        const int g = a.sg[sbase + i];
        w.bs[3 * i] = term_P(a, g, pidx(0, 0));
        w.bs[3 * i + 1] = term_P(a, g, pidx(1, 0));
        w.bs[3 * i + 2] = term_P(a, g, pidx(1, 1));
        w.flag[i] = 0;
    }
    merge_sort_w(a, sbase, U, w.key_w, w.ord);
}

__device__ inline bool merge_self(const MergeArgs& a, int64_t si, double thr) {
    double m[6], P[21];
    survivor_mu(a, si, m);
    survivor_P(a, si, P);
    return mahal6(m, P, m, P) < thr;
}

/* A pair's marginal bound from the stored means and covariances (merge_bound
 * for the pairs of an ill-conditioned survivor). */
__device__ inline bool merge_bound_at(const MergeArgs& a, int64_t si, int64_t sj, double thr) {
    const double du = a.smu[sj * 6] - a.smu[si * 6], dv = a.smu[sj * 6 + 1] - a.smu[si * 6 + 1];
    const int gi = a.sg[si], gj = a.sg[sj];
    const double suu = term_P(a, gi, pidx(0, 0)) + term_P(a, gj, pidx(0, 0));
    const double suv = term_P(a, gi, pidx(1, 0)) + term_P(a, gj, pidx(1, 0));
    const double svv = term_P(a, gi, pidx(1, 1)) + term_P(a, gj, pidx(1, 1));
    const double det = suu * svv - suv * suv;
    if (!(det > 1e-6 * suu * svv)) return true;
    const double q = svv * du * du - 2.0 * suv * du * dv + suu * dv * dv;
    return !(q > 1.001 * thr * det);
}

/* Greedy Gaussian-mixture merge (phdUpdateMergeKernel, src/kernels.cu:662-874):
 * repeatedly take the heaviest unmerged term (ties: lowest pack index),
 * merge every unmerged term within squared Mahalanobis distance
 * min_separation of it by moment matching, emit the merge if PD else the
 * leader, stop when nothing is left or a group's weight is zero.
 *
 * Evaluated in phases instead of the reference's barrier-bound rounds.
 * k_merge_groups (one workgroup per parent):
 *   1. the survivors in bins of u;
 *   2. candidate pairs from each survivor's window of bins, those that pass
 *      the (u, v) marginal's bound (single precision, with its rounding
 *      errors on the safe side: it only chooses what is tested) into a
 *      buffer; whenever it is full, the full 6x6 test, one lane per pair (and
 *      per self pair), so that lanes stay busy however sparse the candidates
 *      are;
 *   3. ranks by (weight desc, index asc): buckets of the weight's leading
 *      bits, then the order within a bucket (bitonic, should one hold more
 *      than MERGE_BUCKET);
 *   4. neighbour lists, by rank;
 *   5. the greedy walk's outcome without the walk: membership depends only on
 *      the pair, so a survivor leads a group when no heavier neighbour does,
 *      and else belongs to the heaviest neighbour that does.  Decided in
 *      rounds, each survivor as soon as its heavier neighbours are;
 *   6. groups in rank order by two scans, members ascending by index.  A
 *      leader that is not its own member ends the walk.
 * k_merge_moments (one thread per group): moments with members summed in
 * ascending index order.  k_merge_rounds: the round loop, for parents whose
 * neighbour lists overflow the workspace.
 *
 * Bound: latency of short phases; three workgroups of 1200 survivors share a
 * CU.  Ten frames of 4096 parents, 200 landmarks (1000 survivors and 4800
 * candidates a parent): 27.6 ms with two bitonic sorts, the lists and a walk
 * per connected component in global scratch; 12.0 so. */
static constexpr int MERGE_BINS = 512, MERGE_CAND = 2048, MERGE_BUCKET = 1024;

template <bool BIG>
__global__ __launch_bounds__(NT) void k_merge_groups(MergeArgs a, int lo, int hi) {
    extern __shared__ char lds[];
    __shared__ int s_n, s_np, s_nill, s_stop;
    __shared__ int sh[8];
    __shared__ double s_red[8];
    __shared__ int s_off[MERGE_BINS + 1], s_cur[MERGE_BINS];
    __shared__ uint32_t s_cand[MERGE_CAND];
    const int p = blockIdx.x;
    const int t = threadIdx.x;
    const int64_t sbase = a.survoff[p];
    const int U = a.survoff[p + 1] - a.survoff[p];
    if (U <= lo || U > hi) return; /* another launch handles this parent (uniform) */
    if (U == 0) {
        if (t == 0) {
            a.ngroups[p] = 0;
            a.nmerged[p] = 0;
        }
        return;
    }
    if (U >= 65536 || a.force_rounds) { /* pairs pack two 16-bit indices: the round loop takes it */
        if (t == 0) {
            a.ngroups[p] = -1;
            a.nmerged[p] = 0;
        }
        return;
    }
    char* const scratch = a.scratch + sbase * a.ws_slot + (int64_t)p * a.ws_parent;
    uint32_t* const pairs = (uint32_t*)scratch;
    const int pcap = 4 * U + 32;
    /* a compile-time choice of workspace, so that the LDS instantiation
     * addresses it with ds_* instructions rather than flat ones */
    char* const ws = BIG ? scratch + (int64_t)U * GROUPS_PAIRS_PER_SLOT + GROUPS_PAIRS_PER_PARENT : lds;
    const GroupsLayout ly(U);
    const double thr = a.min_separation;
    uint8_t* const self = (uint8_t*)(ws + ly.self);

    /* s_cur[0, MERGE_BINS) to exclusive offsets s_off and cursors */
    auto offsets = [&]() {
        constexpr int E = MERGE_BINS / NT;
        int c[E], mine = 0;
#pragma unroll
        for (int e = 0; e < E; ++e) mine += c[e] = s_cur[E * t + e];
        int tot;
        int o = block_exscan(mine, sh, &tot);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            s_off[E * t + e] = s_cur[E * t + e] = o;
            o += c[e];
        }
        if (t == 0) s_off[MERGE_BINS] = tot;
        __syncthreads();
    };
    auto clear = [&]() {
        for (int b = t; b < MERGE_BINS; b += NT) s_cur[b] = 0;
        __syncthreads();
    };

    /* 1. bins of u, monotone in u (a NaN's the first) */
    const double bin_scale =
        MERGE_BINS / fabs(a.rig_meas ? a.rig_meas[a.prig[p]].img_width() : a.img_width);
    auto bin = [&](double u) { return (int)fmin(fmax(u * bin_scale, 0.0), (double)(MERGE_BINS - 1)); };
    if (t == 0) s_n = s_np = s_nill = 0;
    clear();
    /* a survivor's (u, v) marginal; the first few of a thread are held in
     * registers over the barriers, so that their loads wait once */
    struct Marginal {
        double u, v, suu, suv, svv;
        int bin;
    };
    constexpr int HELD = 4;
    auto load_mean = [&](int i, Marginal& m) {
        m.u = a.smu[(sbase + i) * 6];
        m.v = a.smu[(sbase + i) * 6 + 1];
    };
    auto load_cov = [&](int g, Marginal& m) {
        const double* P = term_P_all(a, g);
        m.suu = P[pidx(0, 0)];
        m.suv = P[pidx(1, 0)];
        m.svv = P[pidx(1, 1)];
    };
    Marginal held[HELD];
    {
        int g[HELD];
#pragma unroll
        for (int e = 0; e < HELD; ++e) {
            const int i = min(t + e * NT, U - 1);
            load_mean(i, held[e]);
            g[e] = a.sg[sbase + i];
        }
#pragma unroll
        for (int e = 0; e < HELD; ++e) load_cov(g[e], held[e]);
    }
#pragma unroll
    for (int e = 0; e < HELD; ++e) {
        held[e].bin = bin(held[e].u);
        if (t + e * NT < U) atomicAdd(&s_cur[held[e].bin], 1);
    }
    for (int i = t + HELD * NT; i < U; i += NT) atomicAdd(&s_cur[bin(a.smu[(sbase + i) * 6])], 1);
    __syncthreads();
    offsets();
    {
        double* const bu = (double*)ws;
        double* const bv = (double*)(ws + ly.v);
        float* const bs = (float*)(ws + ly.s);
        uint16_t* const id = (uint16_t*)(ws + ly.id);
        uint16_t* const ill = (uint16_t*)(ws + ly.ill);
        double smax = 0.0, smax_v = 0.0;
        auto good = [&](const Marginal& m) {
            return !a.all_pairs && isfinite(m.u) && isfinite(m.v) && isfinite(m.suu) && isfinite(m.suv) &&
                   isfinite(m.svv) && m.suu > 0.0 && m.svv > 0.0 &&
                   m.suu * m.svv - m.suv * m.suv > 2e-6 * m.suu * m.svv;
        };
        auto place = [&](int i, const Marginal& m) {
            const int q = atomicAdd(&s_cur[m.bin], 1);
            const bool ok = good(m);
            bu[q] = m.u;
            bv[q] = m.v;
            bs[3 * q] = ok ? (float)m.suu : -1.0f;
            bs[3 * q + 1] = (float)m.suv;
            bs[3 * q + 2] = (float)m.svv;
            id[q] = (uint16_t)i;
            if (ok) {
                smax = fmax(smax, m.suu);
                smax_v = fmax(smax_v, m.svv);
            } else {
                ill[atomicAdd(&s_nill, 1)] = (uint16_t)i;
            }
        };
#pragma unroll
        for (int e = 0; e < HELD; ++e)
            if (t + e * NT < U) place(t + e * NT, held[e]);
        for (int i = t + HELD * NT; i < U; i += NT) {
            Marginal m;
            load_mean(i, m);
            load_cov(a.sg[sbase + i], m);
            m.bin = bin(m.u);
            place(i, m);
        }
        smax = block_max(smax, s_red);
        smax_v = block_max(smax_v, s_red);
        __syncthreads();
        /* 2. candidates.
         *   A survivor is ill-conditioned when its (u, v) block is not PD with
         *   det > 2e-6 puu pvv (or holds a non-finite value).  For two that are
         *   not, the block of their sum has det > 1e-6 suu svv (the correlation
         *   of a sum of PSD 2x2 blocks is at most the larger of theirs:
         *   |auv + buv| <= r (sqrt(auu avv) + sqrt(buu bvv)) <= r sqrt(suu svv)
         *   by Cauchy-Schwarz), so the marginal's bound on the distance is
         *   q / det with q = svv du^2 - 2 suv du dv + suu dv^2, and
         *   q suu - du^2 det = (suv du - suu dv)^2 >= 0 makes q <= thr det
         *   imply du^2 <= thr suu.  Such pairs lie within
         *   du^2 <= 1.002 thr (puu_i + max puu) of each other in u: each
         *   survivor meets those after it up to the bin that window ends in,
         *   eight at a time for their v, which must lie within the same of it.
         *   (Every survivor of this filter has puu <= std_u^2: a Kalman update
         *   with H = [I2 0] never raises the measured variance above R, and
         *   births carry R; the windows span a few pixels.)  q is rejected
         *   when it exceeds thr det by 0.1 % and by the single-precision
         *   errors of both.  Those add up to at most 17 roundings of 2^-24 of
         *   svv du^2 + suu dv^2 and 12 of suu svv (1.02e-6 and 0.72e-6; |suv|
         *   of a sum is at most sqrt(suu svv), by Cauchy-Schwarz), so 2e-6 of
         *   each covers them.
         *   Pairs with an ill-conditioned survivor are tested against all
         *   others. */
        const float thrf = (float)(1.0011 * thr);
        int q = t, q2 = 0, qend = 0; /* survivor q, the next block of others */
        uint32_t near = 0;           /* those of the last block near in v */
        float suu = 0, suv = 0, svv = 0;
        double u = 0, v = 0, vlim = 0;
        auto open = [&]() { /* survivor q's window */
            if (q >= U) return;
            u = bu[q];
            v = bv[q];
            suu = bs[3 * q];
            suv = bs[3 * q + 1];
            svv = bs[3 * q + 2];
            q2 = q + 1;
            const double hw = sqrt(1.002 * thr * (1.000001 * (double)suu + smax)) * 1.000001 + 1e-12 * fabs(u);
            vlim = 1.002 * thr * (1.000001 * (double)svv + smax_v);
            qend = suu < 0.0f ? 0 : s_off[bin(u + hw) + 1];
        };
        open();
        const int64_t nx = (int64_t)s_nill * U;
        int64_t e = t; /* of the ill-conditioned survivors' pairs */
        int selfs = U; /* self tests, with the first buffer */
        for (;;) {
            /* `pair` to the buffer; false when it is full */
            auto push = [&](int i, int j) {
                const int c = atomicAdd(&s_n, 1);
                if (c >= MERGE_CAND) return false;
                s_cand[c] = (uint32_t)min(i, j) << 16 | (uint32_t)max(i, j);
                return true;
            };
            bool room = true;
            while (room && q < U) {
                if (!near) {
                    if (q2 >= qend) {
                        q += NT;
                        open();
                        continue;
                    }
                    double d[8];
#pragma unroll
                    for (int k = 0; k < 8; ++k) d[k] = bv[min(q2 + k, U - 1)] - v;
#pragma unroll
                    for (int k = 0; k < 8; ++k) near |= d[k] * d[k] <= vlim ? 1u << k : 0u;
                    near &= (1u << min(qend - q2, 8)) - 1u;
                    q2 += 8;
                    continue;
                }
                const int q1 = q2 - 8 + __builtin_ctz(near);
                const float auu = bs[3 * q1];
                const float du = (float)(bu[q1] - u), dv = (float)(bv[q1] - v);
                const float tuu = suu + auu, tuv = suv + bs[3 * q1 + 1], tvv = svv + bs[3 * q1 + 2];
                const float x = tvv * du * du, y = tuu * dv * dv, w = tuu * tvv;
                const bool far = x + y - 2.0f * tuv * du * dv - 2e-6f * (x + y) > thrf * (w - tuv * tuv + 2e-6f * w);
                if (auu < 0.0f || far || (room = push(id[q], id[q1]))) near &= near - 1u;
            }
            while (room && e < nx) {
                const int i = ill[e / U], j = (int)(e % U);
                /* two ill survivors: once */
                const bool other = j != i && (j > i || !a.all_pairs);
                bool skip = !other;
                if (other && j < i) { /* is j ill too? */
                    Marginal m;
                    load_mean(j, m);
                    load_cov(a.sg[sbase + j], m);
                    skip = !good(m);
                }
                if (skip || !merge_bound_at(a, sbase + min(i, j), sbase + max(i, j), thr) || (room = push(i, j))) e += NT;
            }
            __syncthreads();
            const int nc = min(s_n, MERGE_CAND);
            for (int c = t; c < nc + selfs; c += NT) {
                const uint32_t pr = c < nc ? s_cand[c] : (uint32_t)(c - nc) * 0x10001u;
                const bool in = merge_full(a, sbase, (int)(pr >> 16), (int)(pr & 0xFFFFu), thr);
                if (c >= nc) {
                    self[c - nc] = in ? 1 : 0;
                } else if (in) {
                    const int k = atomicAdd(&s_np, 1);
                    if (k < pcap) pairs[k] = pr;
                }
            }
            selfs = 0;
            const int more = __syncthreads_or(!room);
            if (!more) break;
            if (t == 0) s_n = 0;
            __syncthreads();
        }
    }
    const int np = s_np;
    if (np > pcap) {
        if (t == 0) {
            a.ngroups[p] = -1;
            a.nmerged[p] = 0;
        }
        return;
    }
    /* 3. ranks */
    uint16_t* const ord = (uint16_t*)(ws + ly.ord);
    uint16_t* const own = (uint16_t*)(ws + ly.own);
    {
        double* const key = (double*)ws;
        uint16_t* const tmp = (uint16_t*)(ws + 8 * (int64_t)U);
        /* five bits of the mantissa; weights below 2^-15 share a bucket */
        auto bucket = [&](double w) {
            return min(max((1024 << 5) - 1 - (__double2hiint(w) >> 15), 0), MERGE_BINS - 1);
        };
        clear();
        for (int i = t; i < U; i += NT) {
            const double w = a.sw[sbase + i];
            key[i] = w;
            atomicAdd(&s_cur[bucket(w)], 1);
        }
        __syncthreads();
        int most = 0;
        for (int b = t; b < MERGE_BINS; b += NT) most = max(most, s_cur[b]);
        if (!__syncthreads_or(most > MERGE_BUCKET)) {
            offsets();
            for (int i = t; i < U; i += NT) tmp[atomicAdd(&s_cur[bucket(key[i])], 1)] = (uint16_t)i;
            __syncthreads();
            for (int x = t; x < U; x += NT) {
                const int i = tmp[x];
                const double w = key[i];
                const int b = bucket(w), y0 = s_off[b], y1 = s_off[b + 1];
                int r = y0;
                for (int y = y0; y < y1; y += 4) { /* four reads wait together */
                    int j[4];
                    double o[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) j[k] = tmp[min(y + k, y1 - 1)];
#pragma unroll
                    for (int k = 0; k < 4; ++k) o[k] = key[j[k]];
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        r += y + k < y1 && (o[k] > w || (o[k] == w && j[k] < i)) ? 1 : 0;
                }
                ord[r] = (uint16_t)i;
                own[i] = (uint16_t)r;
            }
        } else {
            int* const o = (int*)(ws + 8 * (int64_t)next_pow2(U));
            merge_sort_w(a, sbase, U, key, o);
            for (int r = t; r < U; r += NT) {
                ord[r] = (uint16_t)o[r];
                own[o[r]] = (uint16_t)r;
            }
        }
        __syncthreads();
    }
    /* 4. neighbour lists: offsets (rows [r0, r1) per thread), fill */
    uint16_t* const nbr = (uint16_t*)ws;
    int* const nbo = (int*)(ws + ly.bnbo);
    int* const cnt = (int*)(ws + ly.cnt);
    uint8_t* const st = (uint8_t*)(ws + ly.st);
    const int rc = (U + NT - 1) / NT;
    const int r0 = min(U, t * rc), r1 = min(U, r0 + rc);
    for (int i = t; i < U; i += NT) {
        cnt[i] = 0;
        st[i] = 0;
    }
    __syncthreads();
    for (int c = t; c < np; c += NT) {
        const uint32_t pr = pairs[c];
        atomicAdd(&cnt[own[pr >> 16]], 1);
        atomicAdd(&cnt[own[pr & 0xFFFFu]], 1);
    }
    __syncthreads();
    {
        int mine = 0;
        for (int r = r0; r < r1; ++r) mine += cnt[r];
        int tot;
        int base = block_exscan(mine, sh, &tot);
        for (int r = r0; r < r1; ++r) {
            nbo[r] = base;
            base += cnt[r];
            cnt[r] = nbo[r];
        }
        if (t == 0) {
            nbo[U] = tot;
            s_stop = U;
        }
    }
    __syncthreads();
    for (int c = t; c < np; c += NT) {
        const uint32_t pr = pairs[c];
        const int x = own[pr >> 16], y = own[pr & 0xFFFFu];
        nbr[atomicAdd(&cnt[x], 1)] = (uint16_t)y;
        nbr[atomicAdd(&cnt[y], 1)] = (uint16_t)x;
    }
    __syncthreads();
    /* 5. leaders (1) and members (2).  A neighbour's state may change while
     * it is read, to what it stays. */
    for (;;) {
        int left = 0;
        for (int r = t; r < U; r += NT) {
            if (st[r]) continue;
            int s = 1;
            const int e1 = nbo[r + 1];
            for (int e = nbo[r]; e < e1 && s != 2; e += 4) { /* four reads wait together */
                int x[4], sx[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) x[k] = nbr[min(e + k, e1 - 1)];
#pragma unroll
                for (int k = 0; k < 4; ++k) sx[k] = *(volatile uint8_t*)(st + x[k]);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (x[k] < r && sx[k] != 2) s = sx[k] == 1 || s == 2 ? 2 : 0;
            }
            *(volatile uint8_t*)(st + r) = (uint8_t)s;
            left |= s == 0;
        }
        if (!__syncthreads_or(left)) break;
    }
    /* each rank's leader; sizes; the first leader that is not its own
     * member, after which no group forms */
    for (int r = t; r < U; r += NT) cnt[r] = 0;
    __syncthreads();
    for (int r = t; r < U; r += NT) {
        int L = r;
        bool counts = true;
        if (st[r] == 2) {
            for (int e = nbo[r]; e < nbo[r + 1]; ++e) {
                const int x = nbr[e];
                if (x < L && st[x] == 1) L = x;
            }
        } else if (!self[ord[r]]) {
            atomicMin(&s_stop, r);
            counts = false;
        }
        own[r] = (uint16_t)L;
        if (counts) atomicAdd(&cnt[L], 1);
    }
    __syncthreads();
    /* 6. groups in rank order */
    {
        const int re = min(r1, s_stop + 1);
        int mg = 0, mm = 0;
        for (int r = r0; r < re; ++r) {
            if (st[r] != 1) continue;
            mg += cnt[r] > 0;
            mm += cnt[r];
        }
        int ng, mtot;
        int gi = block_exscan(mg, sh, &ng);
        int mp = block_exscan(mm, sh, &mtot);
        for (int r = r0; r < r1; ++r) {
            if (st[r] != 1) continue;
            const int n = cnt[r];
            if (r >= re) {
                cnt[r] = -1; /* forms no group */
                continue;
            }
            cnt[r] = mp;
            if (n == 0) continue;
            a.glead[sbase + gi] = ord[r];
            a.gsta[sbase + gi] = mp;
            a.gend[sbase + gi] = mp + n;
            ++gi;
            mp += n;
        }
        if (t == 0) {
            a.ngroups[p] = ng;
            a.nmerged[p] = ng;
        }
    }
    __syncthreads();
    for (int r = t; r < U; r += NT) {
        const int L = own[r], st0 = cnt[L], i = ord[r];
        if (st0 < 0 || (L == r && !self[i])) continue;
        int k = L != r && self[ord[L]] && ord[L] < i ? 1 : 0;
        for (int e = nbo[L]; e < nbo[L + 1]; ++e) {
            const int x = nbr[e];
            k += own[x] == L && x != L && ord[x] < i ? 1 : 0;
        }
        a.gmem[sbase + st0 + k] = i;
    }
}

__global__ __launch_bounds__(128) void k_merge_moments(MergeArgs a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.Stot) return;
    const int p = upper_parent(a.survoff, a.Np, i);
    const int64_t sbase = a.survoff[p];
    const int gi = (int)(i - sbase);
    if (gi >= a.ngroups[p]) return; /* also every slot of a parent left to the round loop */
    const int st = a.gsta[sbase + gi], en = a.gend[sbase + gi];
    double W = 0.0;
    for (int e = st; e < en; ++e) W += a.sw[sbase + a.gmem[sbase + e]];
    if (W == 0) atomicMin(&a.nmerged[p], gi);
    double mu[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) mu[c] = 0.0;
    for (int e = st; e < en; ++e) {
        const int64_t si = sbase + a.gmem[sbase + e];
        const double w = a.sw[si];
#pragma unroll
        for (int c = 0; c < 6; ++c) mu[c] += w * a.smu[(si) * 6 + c];
    }
#pragma unroll
    for (int c = 0; c < 6; ++c) mu[c] = mu[c] / W;
    double P[21];
#pragma unroll
    for (int q = 0; q < 21; ++q) P[q] = 0.0;
    for (int e = st; e < en; ++e) {
        const int64_t si = sbase + a.gmem[sbase + e];
        const double w = a.sw[si];
        const double* Pt = term_P_all(a, a.sg[si]);
        double dl[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) dl[c] = mu[c] - a.smu[(si) * 6 + c];
#pragma unroll
        for (int r = 0; r < 6; ++r)
#pragma unroll
            for (int c = 0; c <= r; ++c) {
                P[pidx(r, c)] += w * (Pt[pidx(r, c)] + dl[c] * dl[r]);
            }
    }
#pragma unroll
    for (int q = 0; q < 21; ++q) P[q] = P[q] / W;
    const int64_t o = i;
    if (is_pd6(P)) {
        a.mw[o] = W;
#pragma unroll
        for (int c = 0; c < 6; ++c) a.mmu[c * a.scap + o] = mu[c];
#pragma unroll
        for (int q = 0; q < 21; ++q) a.mP[q * a.scap + o] = P[q];
    } else {
        const int64_t li = sbase + a.glead[sbase + gi];
        const int g = a.sg[li];
        a.mw[o] = a.sw[li];
#pragma unroll
        for (int c = 0; c < 6; ++c) a.mmu[c * a.scap + o] = a.smu[(li) * 6 + c];
#pragma unroll
        for (int q = 0; q < 21; ++q)
            a.mP[q * a.scap + o] = term_P(a, g, q);
    }
}

template <bool BIG>
__global__ __launch_bounds__(NT) void k_merge_rounds(MergeArgs a) {
    extern __shared__ char lds[];
    __shared__ int s_lead, s_pos, s_nm;
    __shared__ double s_W, s_lw, s_lmu[6], s_lP[21], s_mu[6], s_P[21];
    const int p = blockIdx.x;
    const int t = threadIdx.x;
    if (a.ngroups[p] != -1) return; /* uniform */
    const int64_t sbase = a.survoff[p];
    const int U = a.survoff[p + 1] - a.survoff[p];
    if (BIG != (U > a.rounds_cap)) return;
    char* ws = BIG ? (a.scratch + sbase * a.ws_slot + (int64_t)p * a.ws_parent) : lds;
    MergeWs w(ws, U);
    const double thr = a.min_separation;
    merge_load_sort(a, sbase, U, w);
    for (int i = t; i < U; i += NT) w.selfm[i] = merge_self(a, sbase + i, thr) ? 1 : 0;
    if (t == 0) s_pos = 0;
    __syncthreads();
    const int lane = t & 63, wave = t >> 6;
    const int64_t mbase = sbase;
    int K = 0;
    uint8_t* memb = w.memb; /* round membership */
    for (;;) {
        if (wave == 0) {
            int found = -1;
            for (int r0w = s_pos; r0w < U; r0w += 64) {
                const int r = r0w + lane;
                const bool c = r < U && !w.flag[w.ord[r]];
                const uint64_t b = __ballot(c);
                if (b) {
                    found = r0w + __ffsll((unsigned long long)b) - 1;
                    break;
                }
            }
            if (lane == 0) {
                /* restart at the leader's rank: a leader outside its own
                 * group stays selectable and the next round stops */
                s_lead = found >= 0 ? w.ord[found] : -1;
                s_pos = found >= 0 ? found : U;
            }
        }
        __syncthreads();
        const int lead = s_lead;
        if (lead < 0) break;
        if (t < 6) s_lmu[t] = a.smu[(sbase + lead) * 6 + t];
        if (t == 0) s_lw = a.sw[sbase + lead];
        if (t < 21) {
            const int g = a.sg[sbase + lead];
            s_lP[t] = term_P(a, g, t);
        }
        __syncthreads();
        for (int i = t; i < U; i += NT) {
            uint8_t mb = 0;
            if (!w.flag[i])
                mb = (i == lead ? w.selfm[i] != 0 : merge_pair(a, sbase, w, lead, i, thr)) ? 1 : 0;
            memb[i] = mb;
        }
        __syncthreads();
        if (wave == 0) {
            int nm = 0;
            for (int r0w = 0; r0w < U; r0w += 64) {
                const int i = r0w + lane;
                const bool mbit = i < U && memb[i];
                const uint64_t b = __ballot(mbit);
                if (mbit) w.mem[nm + __popcll(b & ((1ull << lane) - 1ull))] = i;
                nm += __popcll(b);
            }
            if (lane == 0) s_nm = nm;
        }
        __syncthreads();
        const int nm = s_nm;
        if (t == 0) {
            double W = 0.0;
            for (int j = 0; j < nm; ++j) W += a.sw[sbase + w.mem[j]];
            s_W = W;
        }
        __syncthreads();
        const double W = s_W;
        if (W == 0) break;
        if (t < 6) {
            double acc = 0.0;
            for (int j = 0; j < nm; ++j) {
                const int64_t si = sbase + w.mem[j];
                acc += a.sw[si] * a.smu[(si) * 6 + t];
            }
            s_mu[t] = acc / W;
        }
        __syncthreads();
        if (t < 21) {
            int r = 0;
            while ((r + 1) * (r + 2) / 2 <= t) ++r;
            const int c = t - r * (r + 1) / 2;
            double acc = 0.0;
            for (int j = 0; j < nm; ++j) {
                const int64_t si = sbase + w.mem[j];
                const int g = a.sg[si];
                const double Pe = term_P(a, g, t);
                const double dc = s_mu[c] - a.smu[(si) * 6 + c];
                const double dr = s_mu[r] - a.smu[(si) * 6 + r];
                acc += a.sw[si] * (Pe + dc * dr);
            }
            s_P[t] = acc / W;
        }
        __syncthreads();
        if (t == 0) {
            const bool ok = is_pd6(s_P);
            const int64_t o = mbase + K;
            a.mw[o] = ok ? W : s_lw;
            for (int c = 0; c < 6; ++c) a.mmu[c * a.scap + o] = ok ? s_mu[c] : s_lmu[c];
            for (int e = 0; e < 21; ++e) a.mP[e * a.scap + o] = ok ? s_P[e] : s_lP[e];
        }
        for (int j = t; j < nm; j += NT) w.flag[w.mem[j]] = 1;
        ++K;
        __syncthreads();
    }
    if (t == 0) a.nmerged[p] = K;
}

/* ------------------------------------------------------ parent weights */
/* w_p <- w_p exp(loglik_p), normalised, in the log domain with a max shift
 * (src/scphdcameracalibration.cu:1851-1875 multiplies in the linear
 * domain).  One workgroup. */
__global__ __launch_bounds__(1024) void k_parent_weights(double* pw, const double* loglik, int Np,
                                                         const int32_t* poff, const int32_t* rfixed) {
    __shared__ double red[16];
    if (rfixed && rfixed[blockIdx.x]) return; /* this rig's frame used the fixed camera */
    if (poff) { /* one workgroup per rig */
        pw += poff[blockIdx.x];
        loglik += poff[blockIdx.x];
        Np = poff[blockIdx.x + 1] - poff[blockIdx.x];
    }
    /* the first few values of a thread are held over the passes (three
     * logarithms and two exponentials a parent otherwise: 4096 parents 19 us,
     * 10 held; sixteen held cost registers that a busy CU does not have) */
    constexpr int HELD = 4;
    double v[HELD];
    double mx = -INFINITY;
    const int p1 = threadIdx.x + HELD * blockDim.x;
#pragma unroll
    for (int k = 0; k < HELD; ++k) {
        const int p = threadIdx.x + k * blockDim.x;
        v[k] = p < Np ? safe_log(pw[p]) + loglik[p] : -INFINITY;
        mx = fmax(mx, v[k]);
    }
    for (int p = p1; p < Np; p += blockDim.x) mx = fmax(mx, safe_log(pw[p]) + loglik[p]);
    mx = block_max(mx, red);
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < HELD; ++k) {
        const int p = threadIdx.x + k * blockDim.x;
        if (p >= Np) break;
        v[k] = exp(v[k] - mx);
        s += v[k];
    }
    for (int p = p1; p < Np; p += blockDim.x) s += exp(safe_log(pw[p]) + loglik[p] - mx);
    s = block_sum(s, red);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < HELD; ++k) {
        const int p = threadIdx.x + k * blockDim.x;
        if (p < Np) pw[p] = v[k] / s;
    }
    for (int p = p1; p < Np; p += blockDim.x) pw[p] = exp(safe_log(pw[p]) + loglik[p] - mx) / s;
}

/* ------------------------------------------------------ noise check */
/* Six normals per element elem = 0..n-1 of one counter stream, exactly as
 * the filter kernels draw them, for comparison with the CPU restatement. */
__global__ void k_debug_normals(NoiseKey key, uint32_t stream, uint64_t step, uint32_t parent, uint32_t gauss, int n,
                                double* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double z[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (stream == NS_FEATURE)
        feature_normals(key, step, parent, gauss, (uint32_t)i, z);
    else if (stream == NS_POSTERIOR)
        posterior_normals(key, step, parent, gauss, (uint32_t)i, z);
    else
        normals<6>(key, stream, step, parent, gauss, (uint32_t)i, z);
#pragma unroll
    for (int c = 0; c < 6; ++c) out[(int64_t)i * 6 + c] = z[c];
}

/* --------------------------------------------------------- estimate */
/* Sum each of N per-thread values over a 256-thread block; every thread
 * receives the totals (fixed order: wave sums, then waves ascending). */
template <int N>
__device__ inline void block_sum_n(double (&v)[N], double* sh) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const double t = wave_sum(v[i]);
        if (lane == 0) sh[w * N + i] = t;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = ((sh[i] + sh[N + i]) + sh[2 * N + i]) + sh[3 * N + i];
    __syncthreads();
}

/* Twelve 256-thread workgroups per rig of Np parents: weighted mean and
 * covariance of the parent extrinsics and the summed Gaussian weight of the
 * first highest-weight parent's map (exp_traj, cov_traj and cardinality of
 * load_disparity_results.m:27-34).  out per rig: mean[12], cov[144]
 * row-major, cardinality (EST_DOUBLES).
 *
 * Bound: latency, of one pass over the parents for the mean and one for a row
 * of the covariance and of their reductions, so each workgroup forms the mean
 * and then a row of its own (one workgroup a rig, row after row: 47 us for 256
 * parents, 11 so; 16384: 260 and 51). */
__global__ __launch_bounds__(256) void k_estimate(const double* ext, const double* pw, const int32_t* goff,
                                                   const double* gw, int Np, const int32_t* poff, int rig0,
                                                   double* out) {
    __shared__ double sh[4 * 13];
    __shared__ double s_mu[12];
    __shared__ double bws[4];
    __shared__ int bis[4];
    const int row = blockIdx.x; /* of the covariance */
    if (poff) { /* the rig's */
        const int rig = rig0 + blockIdx.y;
        const int64_t P0 = poff[rig];
        Np = poff[rig + 1] - poff[rig];
        ext += P0 * 12;
        pw += P0;
        goff += P0;
        out += (int64_t)rig * EST_DOUBLES;
    }
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    double s1[13];
#pragma unroll
    for (int c = 0; c < 13; ++c) s1[c] = 0.0;
    double bw = -1.0;
    int bi = 0x7fffffff;
    for (int p = t; p < Np; p += 256) {
        const double w = pw[p];
        s1[12] += w;
#pragma unroll
        for (int c = 0; c < 12; ++c) s1[c] += w * ext[(int64_t)p * 12 + c];
        if (w > bw) { /* p ascending within a thread: strict > keeps the first */
            bw = w;
            bi = p;
        }
    }
    /* first maximum: larger weight, then smaller index */
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double ow = __shfl_xor(bw, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        if (ow > bw || (ow == bw && oi < bi)) {
            bw = ow;
            bi = oi;
        }
    }
    if (lane == 0) {
        bws[wv] = bw;
        bis[wv] = bi;
    }
    block_sum_n<13>(s1, sh);
    const double W = s1[12];
    const double r = W > 0 ? 1.0 / W : 0.0;
    double mu[12];
#pragma unroll
    for (int c = 0; c < 12; ++c) mu[c] = s1[c] * r;
    if (t == 0) {
#pragma unroll
        for (int c = 0; c < 12; ++c) s_mu[c] = mu[c];
    }
    __syncthreads();
    const double mi = s_mu[row];
    double v[12];
#pragma unroll
    for (int j = 0; j < 12; ++j) v[j] = 0.0;
    for (int p = t; p < Np; p += 256) {
        const double* x = ext + (int64_t)p * 12;
        const double wdi = pw[p] * (x[row] - mi);
#pragma unroll
        for (int j = 0; j < 12; ++j) v[j] += wdi * (x[j] - mu[j]);
    }
    block_sum_n<12>(v, sh);
    if (t == 0) {
#pragma unroll
        for (int j = 0; j < 12; ++j) out[12 + row * 12 + j] = v[j] * r;
    }
    if (row != 0) return;
    int best = bis[0];
    double bestw = bws[0];
    for (int k = 1; k < 4; ++k)
        if (bws[k] > bestw || (bws[k] == bestw && bis[k] < best)) {
            bestw = bws[k];
            best = bis[k];
        }
    double card[1] = {0.0};
    if (best < Np)
        for (int64_t g = goff[best] + t; g < goff[best + 1]; g += 256) card[0] += gw[g];
    block_sum_n<1>(card, sh);
    if (t < 12) out[t] = s_mu[t];
    if (t == 0) out[156] = card[0];
}

/* ---------------------------------------------------- posterior samples */
/* the block of merged Gaussian gm: a dropped non-detection term's block
 * while there are any, else the next one after them */
__device__ inline int64_t posterior_block(const int32_t* holes, int64_t nholes, int64_t post_base, int64_t gm) {
    return gm < nholes ? (int64_t)holes[gm] : post_base + (gm - nholes);
}

/* Sixteen lanes (one row of a wavefront) per merged Gaussian, four per
 * wavefront: S draws x = L z + mu with L the Cholesky factor of the merged
 * covariance (sample_disparity_gaussian, src/scphdcameracalibration.cu:640-690),
 * factored once per lane and used for every sample the lane draws, mapped
 * to the world by the parent's camera (disparityToWorldKernel,
 * src/kernels.cu:49-80), sample weight 1/S (:2009-2010).  Merged Gaussian
 * gm's cloud goes to the block of a dropped non-detection term while there
 * are any (holes), else after them (posterior_block).  The parent is the same
 * for every row, its data in scalar registers. */
template <typename T, typename A>
__device__ inline void sample_row(const SampleArgs& a, const ParentCtx& pc, int64_t rec, int k, T* to) {
    constexpr bool F32 = std::is_same_v<A, float>;
    const int lane = threadIdx.x & 15;
    double mu[6], P[21], L[21];
#pragma unroll
    for (int c = 0; c < 6; ++c) mu[c] = a.mmu[c * a.scap + rec];
#pragma unroll
    for (int e = 0; e < 21; ++e) P[e] = a.mP[e * a.scap + rec];
    chol6(P, L);
    /* the FP32-arithmetic variant: the factor and mean rounded to single
     * precision once, each draw and its unprojection in single precision */
    MeasF mf;
    PoseF pf;
    A Lf[21], muf[6];
    if constexpr (F32) {
        mf = meas_f(pc.meas);
        pf = pose_f(pc.pose);
    }
#pragma unroll
    for (int e = 0; e < 21; ++e) Lf[e] = (A)L[e];
#pragma unroll
    for (int c = 0; c < 6; ++c) muf[c] = (A)mu[c];
    const T w = (T)(1.0 / a.S);
    PosteriorCarry carry; /* normals carried between the two steps of a noise group */
    /* the lane's sample s, member J of its noise group */
    auto draw = [&](int s, auto member, T x[6]) {
        constexpr uint32_t J = decltype(member)::value;
        A z[6];
        NoiseKey key = pc.key; /* its round keys are formed anew, not held over the sweep */
        asm volatile("" : "+s"(key.k0), "+s"(key.k1));
        posterior_normals_seq(key, pc.step, (uint32_t)pc.pl, (uint32_t)k, (uint32_t)s, J, carry, z);
        if constexpr (F32) {
            float q[6], xf[6];
#pragma unroll
            for (int r = 0; r < 6; ++r) {
                float acc = muf[r];
#pragma unroll
                for (int c = 0; c <= r; ++c) acc = __builtin_fmaf(Lf[pidx(r, c)], z[c], acc);
                q[r] = acc;
            }
            world_from_disparity_f(mf, pf, q, xf);
#pragma unroll
            for (int c = 0; c < 6; ++c) x[c] = (T)xf[c];
        } else {
            double q[6];
#pragma unroll
            for (int r = 0; r < 6; ++r) {
                double acc = 0.0;
#pragma unroll
                for (int c = 0; c <= r; ++c) acc += Lf[pidx(r, c)] * z[c];
                q[r] = acc + muf[r];
            }
            const DisparityPoint d{q[0], q[1], q[2], q[3], q[4], q[5]};
            const EuclideanPoint e = world_from_disparity_fast(pc.meas, pc.pose, d);
            x[0] = (T)e.x; x[1] = (T)e.y; x[2] = (T)e.z; x[3] = (T)e.vx; x[4] = (T)e.vy; x[5] = (T)e.vz;
        }
    };
    auto put = [&](int s0, const T x[6]) {
        T* const o = to + 7 * s0 + lane;
        const int wd = min(a.S - s0, 16);
#pragma unroll
        for (int c = 0; c < 6; ++c) __builtin_nontemporal_store(x[c], &o[c * wd]); /* next read in the next update */
        __builtin_nontemporal_store(w, &o[6 * wd]);
    };
    for (int s0 = 0; s0 < a.S; s0 += 32) { /* a pair of steps is a noise group */
        T x[6];
        if (s0 + lane < a.S) {
            draw(s0 + lane, std::integral_constant<uint32_t, 0>(), x);
            put(s0, x);
        }
        if (s0 + 16 + lane < a.S) {
            draw(s0 + 16 + lane, std::integral_constant<uint32_t, 1>(), x);
            put(s0 + 16, x);
        }
    }
}

template <typename T, typename A = double>
__global__ __launch_bounds__(256) void k_sample(SampleKernArgs<T> ka) {
    const int w = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (w >= ka.a.n_waves) return;
    const int p = ((cint_t*)ka.a.wave_parent)[w];
    if (p < 0) return;
    cint_t* off = (cint_t*)ka.a.mergeoff + p;
    const int k = 4 * (w - first_wave(off[0], p)) + ((threadIdx.x & 63) >> 4);
    if (k >= off[1] - off[0]) return; /* whole rows */
    T* const to = ka.dst.block(posterior_block(ka.a.holes, ka.a.nholes, ka.a.post_base, off[0] + k));
    const SampleArgs& a = kernarg_late<SampleArgs>();
    const ParentCtx pc(a.pose, a.meas, a.rig_meas, a.key, a.ustep, p);
    const int64_t rec = (int64_t)((cint_t*)a.survoff)[p] + k;
    sample_row<T, A>(a, pc, rec, k, to);
}

/* -------------------------------------------------------- map assembly */
/* The kept non-detection entries of a parent at keepoff[p] on, ndlist, the
 * others' blocks in holes (at the entry's index less the kept ones before
 * it), and the posterior's wave_parent.  One wavefront per parent. */
__global__ __launch_bounds__(256) void k_lists(const int32_t* keep, const int32_t* keepoff, const int32_t* goff,
                                               int Np, int32_t* ndlist, int32_t* holes, const int32_t* mergeoff,
                                               int32_t* wave_parent) {
    const int p = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (p >= Np) return;
    write_wave_parents(mergeoff[p], mergeoff[p + 1], p, lane, wave_parent);
    const int g1 = goff[p + 1];
    int k0 = keepoff[p];
    for (int g0 = goff[p]; g0 < g1; g0 += 64) {
        const int g = g0 + lane;
        const bool in = g < g1, kept = in && keep[g] != 0;
        const uint64_t b = __ballot(kept);
        const int k = k0 + __popcll(b & ((1ull << lane) - 1ull));
        if (kept)
            ndlist[k] = g;
        else if (in)
            holes[g - k] = g;
        k0 += __popcll(b);
    }
}

/* New map table per parent: [merged posterior Gaussians | kept
 * non-detection Gaussians in input order] (recombineNonDetections,
 * src/scphdcameracalibration.cu:1422-1574, weights w (1 - pd) for the
 * non-detection terms, :1314-1318). */
__global__ void k_table(TableArgs a) {
    const int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= a.Nout) return;
    const int p = upper_parent(a.outoff, a.Np, o);
    const int j = (int)(o - a.outoff[p]);
    const int K = a.mergeoff[p + 1] - a.mergeoff[p];
    if (j < K) {
        a.gblock[o] = (int32_t)posterior_block(a.holes, a.nholes, a.post_base, (int64_t)a.mergeoff[p] + j);
        a.gwo[o] = a.mw[(int64_t)a.survoff[p] + j];
        a.gpd[o] = 1.0f;
    } else {
        const int g = a.ndlist[a.keepoff[p] + (j - K)];
        const double pdg = a.fit[(int64_t)FP_PD * a.Ng_in + g];
        a.gblock[o] = (int32_t)(a.nd_base + g);
        a.gwo[o] = a.gw[g] * (1 - pdg);
        a.gpd[o] = (float)pdg;
    }
    a.gparent[o] = p;
}

/* ---------------------------------------------------------- resampling */
/* n_eff = 1 / (N sum w^2) (computeNeff :2641-2649); when below min_neff,
 * systematic resampling with points u + j/N against the sequential
 * cumulative sum of the weights (resample :2651-2702), the overrun fallback
 * to the first maximum of exp(w), gather of parent states, and weights 1/N.
 *
 * k_resample, one workgroup a rig: n_eff, the decision, the cumulative sum
 * and the fallback.  The sum keeps the reference's left-to-right rounding,
 * so it is a chain of N additions: the first wavefront adds sixteen weights
 * at a time out of LDS in registers, while the others store the chunk before
 * and load the next.  k_resample_draw, a parent a thread: its point's search
 * (a chain of log2 N reads, so over the whole chip) and the gather.  16384
 * parents: 620 us with the chain's sums stored one by one and the searches
 * and gathers in the same workgroup; 100 so (a frame on average, half of
 * which resample). */
static constexpr int RS_CH = 2048, RS_STEP = 16;

__global__ __launch_bounds__(1024) void k_resample(ResampleArgs a) {
    __shared__ double red[16];
    __shared__ __attribute__((aligned(16))) double chunk[2][RS_CH];
    __shared__ double s_em[16];
    __shared__ int s_am[16];
    const int rig = blockIdx.x;
    const int N = a.poff ? a.poff[rig + 1] - a.poff[rig] : a.Np;
    const int64_t P0 = a.poff ? a.poff[rig] : 0;
    const double* const pw = a.pw + P0;
    double* const cum = a.cum + P0;
    const int t = threadIdx.x;
    double ss = 0.0;
    for (int p = t; p < N; p += blockDim.x) ss += pw[p] * pw[p];
    ss = block_sum(ss, red);
    const double neff = 1.0 / (N * ss);
    const bool go = !(neff >= a.min_neff);
    if (t == 0) {
        a.neff[rig] = neff;
        a.rflag[rig] = go ? 1 : 0;
    }
    if (!go) return;
    /* first index of the maximum of exp(w) */
    double em = -1.0;
    int am = -1;
    for (int i = t; i < N; i += blockDim.x) {
        const double w = pw[i], e = exp(w);
        if (i < RS_CH) chunk[0][i] = w;
        if (e > em) {
            em = e;
            am = i;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double e2 = __shfl_xor(em, o, 64);
        const int a2 = __shfl_xor(am, o, 64);
        if (e2 > em || (e2 == em && a2 >= 0 && (am < 0 || a2 < am))) {
            em = e2;
            am = a2;
        }
    }
    if ((t & 63) == 0) {
        s_em[t >> 6] = em;
        s_am[t >> 6] = am;
    }
    __syncthreads();
    if (t == 0) {
        int amax = -1;
        double bm = -1.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
            if (s_am[w] >= 0 && (s_em[w] > bm || (s_em[w] == bm && s_am[w] < amax))) {
                bm = s_em[w];
                amax = s_am[w];
            }
        }
        a.amax[rig] = amax;
    }
    /* sequential cumulative sum */
    double c = 0.0;
    int b = 0;
    for (int c0 = 0; c0 < N; c0 += RS_CH, b ^= 1) {
        if (t < 64) {
            const int n = min(RS_CH, N - c0);
            double* const x = chunk[b];
            int i = 0;
            double v[RS_STEP];
            if (RS_STEP <= n) {
#pragma unroll
                for (int k = 0; k < RS_STEP; ++k) v[k] = x[k];
            }
            for (; i + RS_STEP <= n; i += RS_STEP) {
                double w[RS_STEP]; /* the next, while this one's sums wait */
                const int j = min(i + RS_STEP, RS_CH - RS_STEP);
#pragma unroll
                for (int k = 0; k < RS_STEP; ++k) w[k] = x[j + k];
#pragma unroll
                for (int k = 0; k < RS_STEP; ++k) v[k] = c += v[k];
                if (t == 0) {
#pragma unroll
                    for (int k = 0; k < RS_STEP; ++k) x[i + k] = v[k];
                }
#pragma unroll
                for (int k = 0; k < RS_STEP; ++k) v[k] = w[k];
            }
            for (; i < n; ++i) {
                c += x[i];
                if (t == 0) x[i] = c;
            }
        } else {
            double* const x = chunk[b ^ 1];
            for (int i = t - 64; i < RS_CH; i += blockDim.x - 64) {
                const int at = c0 + i;
                if (c0 > 0) cum[at - RS_CH] = x[i];
                if (at + RS_CH < N) x[i] = pw[at + RS_CH];
            }
        }
        __syncthreads();
    }
    const int last = (N - 1) / RS_CH * RS_CH;
    for (int i = t; last + i < N; i += blockDim.x) cum[last + i] = chunk[b ^ 1][i];
}

__global__ __launch_bounds__(256) void k_resample_draw(ResampleArgs a) {
    __shared__ int s_anc[256];
    const int t = threadIdx.x, j0 = blockIdx.x * 256, n = min(256, a.Np - j0);
    int any = 0;
    for (int r = t; r < a.nrigs; r += 256) any |= a.rflag[r];
    if (t < n) {
        const int g = j0 + t;
        const int rig = a.prig ? a.prig[g] : 0;
        const int P0 = a.poff ? a.poff[rig] : 0, N = a.poff ? a.poff[rig + 1] - P0 : a.Np;
        int anc = g;
        if (a.rflag[rig]) {
            const NoiseKey key = a.keys ? a.keys[rig] : a.key;
            /* the rig's own resample count: the handle's less its count at joining */
            const uint64_t rstep = a.rstep - (a.sbase ? a.sbase[SC_COUNT * rig + SC_RESAMPLE] : 0u);
            uint32_t x[4];
            noise_block(key, NS_RESAMPLE, rstep, 0, 0, 0, 0, x);
            const double u = uniform_co(x[0], x[1]) * (1.0 / N);
            const double interval = 1.0 / N;
            const int j = g - P0;
            const double r = u + j * interval;
            int lo = 0, hi = N;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (!(r > a.cum[P0 + mid]))
                    hi = mid;
                else
                    lo = mid + 1;
            }
            anc = P0 + (lo < N ? lo : a.amax[rig]);
            if (!a.defer) a.pw[g] = 1.0 / N;
        }
        a.anc[g] = anc;
        a.newcnt[g] = a.goff[anc + 1] - a.goff[anc];
        s_anc[t] = anc;
    }
    if (!__syncthreads_or(any)) return;
    for (int i = t; i < 12 * n; i += 256) a.ext_tmp[(int64_t)j0 * 12 + i] = a.ext[(int64_t)s_anc[i / 12] * 12 + i % 12];
}

__global__ void k_resample_commit(double* ext, const double* ext_tmp, double* pw, int32_t* anc_out,
                                  const int32_t* anc, int N, int go) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= N) return;
    anc_out[j] = anc[j];
    if (go) {
        for (int q = 0; q < 12; ++q) ext[(int64_t)j * 12 + q] = ext_tmp[(int64_t)j * 12 + q];
        pw[j] = 1.0 / N;
    }
}

__global__ void k_fill_i32(int32_t* x, int32_t v, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = v;
}

__global__ void k_iota(int32_t* x, int64_t n, int32_t start) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = start + (int32_t)i;
}

/* ---------------------------------------------- ensemble membership */
/* The map table without one rig's Gaussians [G0, G0 + Gr): entry i of the
 * result is entry i below G0, else entry i + Gr, whose parent index (at or
 * after the removed rig's parents, which end at P1) moves down by Nr. */
__global__ void k_table_remove(const int32_t* gparent, const int32_t* gblock, const double* gw, const float* gpd,
                               int64_t G0, int64_t Gr, int64_t Ng_new, int P1, int Nr, int32_t* gparent_out,
                               int32_t* gblock_out, double* gw_out, float* gpd_out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= Ng_new) return;
    const int64_t j = i < G0 ? i : i + Gr;
    const int32_t p = gparent[j];
    gparent_out[i] = p >= P1 ? p - Nr : p;
    gblock_out[i] = gblock[j];
    gw_out[i] = gw[j];
    if (gpd_out) gpd_out[i] = gpd[j];
}

__global__ void k_goff_remove(const int32_t* goff, int P0, int Nr, int32_t Gr, int Np_new, int32_t* goff_out) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p > Np_new) return;
    goff_out[p] = p < P0 ? goff[p] : goff[p + Nr] - Gr;
}

__global__ void k_index_shift(int32_t* x, int64_t n, int P1, int Nr) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && x[i] >= P1) x[i] -= Nr;
}

__global__ void k_table_resample(const int32_t* anc, const int32_t* goff_old, const int32_t* goff_new,
                                 const int32_t* gblock_old, const double* gw_old, int Np, int64_t Nnew,
                                 int32_t* gparent, int32_t* gblock, double* gw, const float* gpd_old,
                                 float* gpd) {
    const int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= Nnew) return;
    const int p = upper_parent(goff_new, Np, o);
    const int64_t src = (int64_t)goff_old[anc[p]] + (o - goff_new[p]);
    gparent[o] = p;
    gblock[o] = gblock_old[src];
    gw[o] = gw_old[src];
    if (gpd) gpd[o] = gpd_old[src];
}

/* ------------------------------------------------------------ read-back */
/* The map's clouds into consecutive blocks: block g of dst <- block
 * gblock[g] of src.  A wavefront a cloud at a time, in workgroups that fill
 * the chip once: a map has more values than a launch may have threads, and
 * short clouds cost more in workgroups than in copies (scphd_compact of
 * 102,400 clouds of 100 samples: 0.46 ms with a thread a value, 0.19 so). */
template <typename T>
__global__ __launch_bounds__(256) void k_gather(Clouds<T> src, Clouds<T> dst, const int32_t* gblock, int64_t Ng,
                                                int S) {
    const int n = 7 * S;
    for (int64_t g = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); g < Ng; g += (int64_t)gridDim.x * 4) {
        const T* const from = src.block(gblock[g]);
        T* const to = dst.block(g);
        for (int e = threadIdx.x & 63; e < n; e += 64) to[e] = from[e];
    }
}

template <typename T>
__global__ void k_extract(Clouds<T> src, const int32_t* gblock, int64_t Ng, int S, double* out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n = Ng * S;
    if (i >= n) return;
    const int64_t g = i / S;
    T r[7];
    load_sample<T>(src.block(gblock[g]), S, (int)(i - g * S), r);
#pragma unroll
    for (int c = 0; c < 7; ++c) out[c * n + i] = (double)r[c];
}

template <typename T>
__global__ void k_inject(const double* in, int64_t Ng, int S, Clouds<T> dst) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n = Ng * S;
    if (i >= n) return;
    const int64_t g = i / S;
    const int s = (int)(i - g * S);
    T* const b = dst.block(g);
#pragma unroll
    for (int c = 0; c < 7; ++c) b[cloud_at(S, s, c)] = (T)in[c * n + i];
}

/* ----------------------------------------------------------------- scan */
/* Up to SCAN_ONE values in one workgroup: a launch instead of the three or
 * four of the tiled scan and the read-out (256 values: 12.4 us in three
 * launches, 7.4 in one; 4096: 22.8 in four, 9.7 in one; 16384: 23.6 and 21,
 * and 45 for the update's two scans, the time of their eight launches). */
static constexpr int SCAN_ONE_T = 1024, SCAN_ONE_I = 8, SCAN_ONE = SCAN_ONE_T * SCAN_ONE_I;

/* SCAN_ONE_I consecutive values a thread, from base on */
__device__ inline int scan_load(const int32_t* in, int n, int base, int (&v)[SCAN_ONE_I]) {
    int s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ONE_I; ++i) {
        v[i] = base + i < n ? in[base + i] : 0;
        s += v[i];
    }
    return s;
}

/* what a read-out leaves in host memory: the offsets' end, the largest
 * segment, the segments over limit, the largest of x0[0, n0) and x1 */
__device__ inline void read_out(int total, int mx, int over, const int32_t* x0, int n0, const int32_t* x1,
                                volatile int32_t* out) {
    __shared__ int smax[16], scnt[16];
    int any = 0;
    for (int i = threadIdx.x; i < n0; i += blockDim.x) any = max(any, x0[i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        mx = max(mx, __shfl_xor(mx, o, 64));
        over += __shfl_xor(over, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        smax[threadIdx.x >> 6] = mx;
        scnt[threadIdx.x >> 6] = over;
    }
    __shared__ int s_any;
    if (threadIdx.x == 0) s_any = 0;
    __syncthreads();
    if (any) atomicMax(&s_any, any);
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
            mx = max(mx, smax[w]);
            over += scnt[w];
        }
        out[0] = total;
        out[1] = mx;
        out[2] = over;
        out[3] = s_any;
        out[4] = x1 ? *x1 : 0;
    }
}

__global__ __launch_bounds__(SCAN_ONE_T) void k_scan_readout(const int32_t* in, int32_t* off, int n, int32_t limit,
                                                             const int32_t* x0, int n0, const int32_t* x1,
                                                             volatile int32_t* out) {
    __shared__ int sh[SCAN_ONE_T / 64];
    const int items = (n + SCAN_ONE_T - 1) / SCAN_ONE_T; /* a thread */
    const int base = threadIdx.x * items, end = min(n, base + items);
    int v[SCAN_ONE_I], tot, mx = 0, over = 0;
    int o = block_exscan(scan_load(in, end, base, v), sh, &tot);
#pragma unroll
    for (int i = 0; i < SCAN_ONE_I; ++i) {
        if (base + i < end) off[base + i] = o;
        o += v[i];
        mx = max(mx, v[i]);
        over += limit > 0 && v[i] > limit ? 1 : 0;
    }
    if (threadIdx.x == 0) off[n] = tot;
    read_out(tot, mx, over, x0, n0, x1, out);
}

/* The update's output offsets: mergeoff of the merged terms' counts, keepoff
 * of the kept non-detection terms', off of both. */
__global__ __launch_bounds__(SCAN_ONE_T) void k_outputs(const int32_t* nmerged, const int32_t* nkeep, int n,
                                                        int32_t limit, const int32_t* x1, int32_t* mergeoff,
                                                        int32_t* keepoff, int32_t* off, volatile int32_t* out) {
    __shared__ int sh[SCAN_ONE_T / 64];
    __shared__ int s_merged;
    const int items = (n + SCAN_ONE_T - 1) / SCAN_ONE_T;
    const int base = threadIdx.x * items, end = min(n, base + items);
    int v[SCAN_ONE_I], w[SCAN_ONE_I], tv, tw, mx = 0, over = 0;
    int ov = block_exscan(scan_load(nmerged, end, base, v), sh, &tv);
    int ow = block_exscan(scan_load(nkeep, end, base, w), sh, &tw);
#pragma unroll
    for (int i = 0; i < SCAN_ONE_I; ++i) {
        if (base + i < end) {
            mergeoff[base + i] = ov;
            keepoff[base + i] = ow;
            off[base + i] = ov + ow;
        }
        ov += v[i];
        ow += w[i];
        mx = max(mx, v[i] + w[i]);
        over += limit > 0 && v[i] + w[i] > limit ? 1 : 0;
    }
    if (threadIdx.x == 0) {
        mergeoff[n] = s_merged = tv;
        keepoff[n] = tw;
        off[n] = tv + tw;
    }
    __syncthreads();
    read_out(tv + tw, mx, over, &s_merged, 1, x1, out);
}

/* off = mergeoff + keepoff, n + 1 of them */
__global__ void k_add_offsets(const int32_t* mergeoff, const int32_t* keepoff, int n, int32_t* off) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i <= n) off[i] = mergeoff[i] + keepoff[i];
}

static constexpr int SCAN_T = 256, SCAN_I = 8, SCAN_TILE = SCAN_T * SCAN_I;

__global__ __launch_bounds__(SCAN_T) void k_scan_tiles(const int32_t* in, int32_t* out, int64_t n, int32_t* sums) {
    __shared__ int sh[8];
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_I;
    int v[SCAN_I];
    int s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_I; ++i) {
        v[i] = (base + i < n) ? in[base + i] : 0;
        s += v[i];
    }
    int tot;
    int off = block_exscan(s, sh, &tot);
#pragma unroll
    for (int i = 0; i < SCAN_I; ++i) {
        if (base + i < n) out[base + i] = off;
        off += v[i];
    }
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

__global__ __launch_bounds__(SCAN_T) void k_scan_sums(int32_t* sums, int64_t nb, int32_t* total_out) {
    __shared__ int sh[8];
    int carry = 0;
    for (int64_t c0 = 0; c0 < nb; c0 += SCAN_T) {
        const int64_t i = c0 + threadIdx.x;
        const int v = i < nb ? sums[i] : 0;
        int tot;
        const int o = block_exscan(v, sh, &tot);
        if (i < nb) sums[i] = carry + o;
        carry += tot;
    }
    if (threadIdx.x == 0) *total_out = carry;
}

__global__ void k_scan_add(int32_t* out, int64_t n, const int32_t* sums) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] += sums[i / SCAN_TILE];
}

/* ============================================================ launchers */
static inline unsigned nblocks(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

/* the same, of a kernel whose workgroups stride over what is left: no more
 * than the 2^32 - 1 threads a launch may have (more are taken modulo 2^32,
 * without an error) */
static inline unsigned nblocks_strided(int64_t n, int t) {
    return (unsigned)std::min<int64_t>((n + t - 1) / t, 0xFFFFFFFFll / t);
}

#define LAUNCH_CHECK() return hipGetLastError()

hipError_t launch_prior(hipStream_t s, double* ext, double* pw, int Np, const double* a12, const double* b12,
                        NoiseKey key) {
    Bounds12 ab;
    for (int i = 0; i < 12; ++i) {
        ab.a[i] = a12[i];
        ab.b[i] = b12[i];
    }
    k_prior<<<nblocks(Np, 256), 256, 0, s>>>(ext, pw, Np, ab, key);
    LAUNCH_CHECK();
}

hipError_t launch_parent_predict(hipStream_t s, double* ext, int Np, OrientedLinearCVMotionModel3D cam, double dt,
                                 RigKeys key, uint64_t step) {
    k_parent_predict<<<nblocks(Np, 256), 256, 0, s>>>(ext, Np, cam, dt, key, step);
    LAUNCH_CHECK();
}

hipError_t launch_scale(hipStream_t s, double* x, int64_t n, double a) {
    if (n <= 0) return hipSuccess;
    k_scale<<<nblocks(n, 256), 256, 0, s>>>(x, n, a);
    LAUNCH_CHECK();
}

int64_t wave_count(int64_t n, int Np) { return n / 4 + Np; }

hipError_t launch_pose(hipStream_t s, const double* ext, double* pose, int Np, int fixed, const int32_t* prig,
                       const int32_t* rfixed, const int32_t* goff, int32_t* wave_parent, int32_t* counters) {
    if (rfixed && !prig) return hipErrorInvalidValue;
    k_pose<<<nblocks(Np, 4), 256, 0, s>>>(ext, pose, Np, fixed, prig, rfixed, goff, wave_parent, counters);
    LAUNCH_CHECK();
}

template <typename T>
hipError_t launch_materialize(hipStream_t s, Clouds<T> src, Clouds<T> dst, const int32_t* gblock,
                              const int32_t* gparent, const int32_t* goff, int64_t Ng, int S,
                              LinearCVMotionModel3D feat, double dt, RigKeys key, uint64_t step, bool arith32) {
    if (Ng <= 0) return hipSuccess;
    if (arith32 && !std::is_same_v<T, float>) return hipErrorInvalidValue;
    k_materialize<T><<<nblocks_strided(Ng * S, 256), 256, 0, s>>>(src, dst, gblock, gparent, goff, Ng, S, feat, dt,
                                                                  key, step, arith32 ? 1 : 0);
    LAUNCH_CHECK();
}

template <typename T>
hipError_t launch_fit(hipStream_t s, const FitArgs& a, Clouds<T> src, Clouds<T> dst) {
    if (a.Ng <= 0) return hipSuccess;
    const unsigned nb = nblocks(a.n_waves, 4);
    if constexpr (std::is_same_v<T, float>) {
        if (a.arith32) {
            k_fit<T, float><<<nb, 256, 0, s>>>(FitKernArgs<T>{a, src, dst});
            LAUNCH_CHECK();
        }
    } else if (a.arith32) {
        return hipErrorInvalidValue;
    }
    k_fit<T><<<nb, 256, 0, s>>>(FitKernArgs<T>{a, src, dst});
    LAUNCH_CHECK();
}

template <typename T>
hipError_t launch_fit_fix(hipStream_t s, const FitArgs& a, Clouds<T> src, Clouds<T> dst) {
    if (a.Ng <= 0) return hipSuccess;
    const unsigned nb = (unsigned)std::min<int64_t>(nblocks(a.Ng, 16), 256);
    if constexpr (std::is_same_v<T, float>) {
        if (a.arith32) {
            if (a.rig_meas)
                k_fit_fix<T, true, float><<<nb, 256, 0, s>>>(a, src, dst);
            else
                k_fit_fix<T, false, float><<<nb, 256, 0, s>>>(a, src, dst);
            LAUNCH_CHECK();
        }
    } else if (a.arith32) {
        return hipErrorInvalidValue;
    }
    if (a.rig_meas)
        k_fit_fix<T, true><<<nb, 256, 0, s>>>(a, src, dst);
    else
        k_fit_fix<T, false><<<nb, 256, 0, s>>>(a, src, dst);
    LAUNCH_CHECK();
}

template <typename T>
hipError_t launch_nd_fill(hipStream_t s, const FitArgs& a, Clouds<T> src, Clouds<T> dst) {
    if (a.Ng <= 0) return hipSuccess;
    const int64_t blocks = std::min<int64_t>(nblocks(a.Ng, 16), 2048); /* the list is at most Ng long */
    if constexpr (std::is_same_v<T, float>) {
        if (a.arith32) {
            if (a.rig_meas)
                k_nd_fill<T, true, float><<<blocks, 256, 0, s>>>(a, src, dst);
            else
                k_nd_fill<T, false, float><<<blocks, 256, 0, s>>>(a, src, dst);
            LAUNCH_CHECK();
        }
    } else if (a.arith32) {
        return hipErrorInvalidValue;
    }
    if (a.rig_meas)
        k_nd_fill<T, true><<<blocks, 256, 0, s>>>(a, src, dst);
    else
        k_nd_fill<T, false><<<blocks, 256, 0, s>>>(a, src, dst);
    LAUNCH_CHECK();
}

hipError_t launch_precompute(hipStream_t s, const double* fit, const double* gw, int64_t Ng, double var_u,
                             double var_v, double* pre, double* lik) {
    if (Ng <= 0) return hipSuccess;
    k_precompute<<<nblocks(Ng, 128), 128, 0, s>>>(fit, gw, Ng, var_u, var_v, pre, lik);
    LAUNCH_CHECK();
}

hipError_t launch_eta(hipStream_t s, EtaArgs a, int max_map) {
    /* an odd stride: a word of all places lies in all banks.  The list as
     * long as two workgroups of a CU's 160 KB allow (the kernel's own arrays
     * take 11 each): each round of a list costs the walk of its rows' masks by
     * few lanes (ten frames of 4096 parents, 200 landmarks: 11.6 ms with 1024
     * terms, 10.5 with 2048, 9.6 with 4096; a denser scene, where 4096 leave
     * room for one: 10.7, 8.5, 10.8). */
    a.mask_stride = ((std::min(max_map, ETA_CHUNK) + 31) / 32) | 1;
    const size_t mask = (size_t)std::min(std::max(a.M, 1), NT) * a.mask_stride * sizeof(uint32_t);
    a.list = mask + 4096 * sizeof(double) <= 68 * 1024 ? 4096 : 2048;
    k_eta<<<a.Np, NT, a.list * sizeof(double) + mask, s>>>(a);
    if (max_map > ETA_CHUNK && !a.no_lists) k_eta_list<<<a.Np, NT, sizeof(LateList), s>>>(a);
    LAUNCH_CHECK();
}

hipError_t launch_survivors(hipStream_t s, const SurvArgs& a) {
    k_survivors<<<a.e.Np, NT, 0, s>>>(a);
    LAUNCH_CHECK();
}

hipError_t launch_merge(hipStream_t s, const MergeArgs& a, int max_surv) {
    /* a launch's LDS is that of its largest parent: one for those of which
     * two share a CU, one for those that take a CU each, and the rest in
     * global scratch */
    const int cap2 = std::min(a.lds_cap, GROUPS_CAP2), cap1 = std::min(a.lds_cap, GROUPS_CAP1);
    k_merge_groups<false><<<a.Np, NT, groups_lds_bytes(std::min(max_surv, cap2)), s>>>(a, -1, cap2);
    if (max_surv > cap2 && cap1 > cap2)
        k_merge_groups<false><<<a.Np, NT, groups_lds_bytes(std::min(max_surv, cap1)), s>>>(a, cap2, cap1);
    if (max_surv > cap1) k_merge_groups<true><<<a.Np, NT, 0, s>>>(a, cap1, INT32_MAX);
    if (a.Stot > 0) k_merge_moments<<<nblocks(a.Stot, 128), 128, 0, s>>>(a);
    k_merge_rounds<false><<<a.Np, NT, merge_lds_bytes(std::max(1, std::min(max_surv, a.rounds_cap))), s>>>(a);
    if (max_surv > a.rounds_cap) k_merge_rounds<true><<<a.Np, NT, 0, s>>>(a);
    LAUNCH_CHECK();
}

hipError_t launch_parent_weights(hipStream_t s, double* pw, const double* loglik, int Np, const int32_t* poff,
                                 int nrigs, const int32_t* rfixed) {
    if (rfixed && !poff) return hipErrorInvalidValue;
    k_parent_weights<<<poff ? nrigs : 1, 1024, 0, s>>>(pw, loglik, Np, poff, rfixed);
    LAUNCH_CHECK();
}

hipError_t launch_debug_normals(hipStream_t s, NoiseKey key, uint32_t stream, uint64_t step, uint32_t parent,
                                uint32_t gauss, int n, double* out) {
    if (n <= 0) return hipSuccess;
    k_debug_normals<<<nblocks(n, 256), 256, 0, s>>>(key, stream, step, parent, gauss, n, out);
    LAUNCH_CHECK();
}

hipError_t launch_estimate(hipStream_t s, const double* ext, const double* pw, const int32_t* goff,
                           const double* gw, int Np, const int32_t* poff, int nrigs, double* out) {
    if (poff ? nrigs <= 0 : Np <= 0) return hipErrorInvalidValue;
    constexpr int SLICE = 65535; /* a grid's y has at most 65536 */
    for (int r = 0; r < (poff ? nrigs : 1); r += SLICE)
        k_estimate<<<dim3(12, poff ? std::min(nrigs - r, SLICE) : 1), 256, 0, s>>>(ext, pw, goff, gw, Np, poff, r, out);
    LAUNCH_CHECK();
}

template <typename T>
hipError_t launch_sample(hipStream_t s, const SampleArgs& a, Clouds<T> dst) {
    if (a.Kt <= 0) return hipSuccess;
    const unsigned nb = nblocks(a.n_waves, 4);
    if constexpr (std::is_same_v<T, float>) {
        if (a.arith32) {
            k_sample<T, float><<<nb, 256, 0, s>>>(SampleKernArgs<T>{a, dst});
            LAUNCH_CHECK();
        }
    } else if (a.arith32) {
        return hipErrorInvalidValue;
    }
    k_sample<T><<<nb, 256, 0, s>>>(SampleKernArgs<T>{a, dst});
    LAUNCH_CHECK();
}

hipError_t launch_lists(hipStream_t s, const int32_t* keep, const int32_t* keepoff, const int32_t* goff, int Np,
                        int32_t* ndlist, int32_t* holes, const int32_t* mergeoff, int32_t* wave_parent) {
    k_lists<<<nblocks(Np, 4), 256, 0, s>>>(keep, keepoff, goff, Np, ndlist, holes, mergeoff, wave_parent);
    LAUNCH_CHECK();
}

hipError_t launch_table(hipStream_t s, const TableArgs& a) {
    if (a.Nout <= 0) return hipSuccess;
    k_table<<<nblocks(a.Nout, 256), 256, 0, s>>>(a);
    LAUNCH_CHECK();
}

hipError_t launch_resample(hipStream_t s, const ResampleArgs& a) {
    k_resample<<<a.poff ? a.nrigs : 1, 1024, 0, s>>>(a);
    k_resample_draw<<<nblocks(a.Np, 256), 256, 0, s>>>(a);
    LAUNCH_CHECK();
}

/* Scalars the host needs after a scan, written by the device straight into
 * mapped host memory, so that a read-back costs no copy-engine transfer:
 * out[0] = off[n], out[1] = the largest segment off[p + 1] - off[p],
 * out[2] = the number of segments above `limit` (0 when limit <= 0),
 * out[3] = the largest of x0[0, n0) (0 when n0 = 0) and out[4] = *x1 (0 for a
 * null pointer).  One workgroup. */
__global__ __launch_bounds__(1024) void k_readout(const int32_t* off, int n, int32_t limit, const int32_t* x0, int n0,
                                                  const int32_t* x1, volatile int32_t* out) {
    int mx = 0, c = 0;
    for (int p = threadIdx.x; p < n; p += blockDim.x) {
        const int seg = off[p + 1] - off[p];
        mx = max(mx, seg);
        c += (limit > 0 && seg > limit) ? 1 : 0;
    }
    read_out(off[n], mx, c, x0, n0, x1, out);
}

/* out = the number of NaN entries of w[0, n) (checkStuff,
 * src/scphdcameracalibration.cu:812-821, without the host copy).  One
 * workgroup. */
__global__ __launch_bounds__(1024) void k_nan_count(const double* w, int n, volatile int32_t* out) {
    __shared__ int sc[16];
    int c = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) c += w[i] != w[i] ? 1 : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if ((threadIdx.x & 63) == 0) sc[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < (int)(blockDim.x >> 6); ++k) c += sc[k];
        *out = c;
    }
}

/* Detection pairs of an ensemble update: the sum over rigs of the rig's
 * map size times its measurement count (exact in FP64 below 2^53).  One
 * workgroup. */
__global__ __launch_bounds__(256) void k_pair_count(const int32_t* goff, const int32_t* moff, const int32_t* poff,
                                                    int nrigs, volatile double* out) {
    __shared__ double red[16];
    double c = 0.0;
    for (int r = threadIdx.x; r < nrigs; r += blockDim.x)
        c += (double)(goff[poff[r + 1]] - goff[poff[r]]) * (double)(moff[r + 1] - moff[r]);
    c = block_sum(c, red);
    if (threadIdx.x == 0) *out = c;
}

hipError_t launch_pair_count(hipStream_t s, const int32_t* goff, const int32_t* moff, const int32_t* poff,
                             int nrigs, double* out) {
    k_pair_count<<<1, 256, 0, s>>>(goff, moff, poff, nrigs, out);
    LAUNCH_CHECK();
}

hipError_t launch_nan_count(hipStream_t s, const double* w, int n, int32_t* out) {
    k_nan_count<<<1, 1024, 0, s>>>(w, n, out);
    LAUNCH_CHECK();
}

hipError_t launch_resample_commit(hipStream_t s, double* ext, const double* ext_tmp, double* pw, int32_t* anc_out,
                                  const int32_t* anc, int N, int go) {
    if (N <= 0) return hipSuccess;
    k_resample_commit<<<nblocks(N, 256), 256, 0, s>>>(ext, ext_tmp, pw, anc_out, anc, N, go);
    LAUNCH_CHECK();
}

hipError_t launch_fill_i32(hipStream_t s, int32_t* x, int32_t v, int64_t n) {
    if (n <= 0) return hipSuccess;
    k_fill_i32<<<nblocks(n, 256), 256, 0, s>>>(x, v, n);
    LAUNCH_CHECK();
}

hipError_t launch_iota(hipStream_t s, int32_t* x, int64_t n, int32_t start) {
    if (n <= 0) return hipSuccess;
    k_iota<<<nblocks(n, 256), 256, 0, s>>>(x, n, start);
    LAUNCH_CHECK();
}

hipError_t launch_table_remove(hipStream_t s, const int32_t* gparent, const int32_t* gblock, const double* gw,
                               const float* gpd, int64_t G0, int64_t Gr, int64_t Ng_new, int P1, int Nr,
                               int32_t* gparent_out, int32_t* gblock_out, double* gw_out, float* gpd_out) {
    if (Ng_new <= 0) return hipSuccess;
    if ((gpd_out != nullptr) != (gpd != nullptr)) return hipErrorInvalidValue;
    k_table_remove<<<nblocks(Ng_new, 256), 256, 0, s>>>(gparent, gblock, gw, gpd, G0, Gr, Ng_new, P1, Nr,
                                                        gparent_out, gblock_out, gw_out, gpd_out);
    LAUNCH_CHECK();
}

hipError_t launch_goff_remove(hipStream_t s, const int32_t* goff, int P0, int Nr, int32_t Gr, int Np_new,
                              int32_t* goff_out) {
    k_goff_remove<<<nblocks((int64_t)Np_new + 1, 256), 256, 0, s>>>(goff, P0, Nr, Gr, Np_new, goff_out);
    LAUNCH_CHECK();
}

hipError_t launch_index_shift(hipStream_t s, int32_t* x, int64_t n, int P1, int Nr) {
    if (n <= 0) return hipSuccess;
    k_index_shift<<<nblocks(n, 256), 256, 0, s>>>(x, n, P1, Nr);
    LAUNCH_CHECK();
}

hipError_t launch_table_resample(hipStream_t s, const int32_t* anc, const int32_t* goff_old,
                                 const int32_t* goff_new, const int32_t* gblock_old, const double* gw_old, int Np,
                                 int64_t Nnew, int32_t* gparent, int32_t* gblock, double* gw,
                                 const float* gpd_old, float* gpd) {
    if (Nnew <= 0) return hipSuccess;
    k_table_resample<<<nblocks(Nnew, 256), 256, 0, s>>>(anc, goff_old, goff_new, gblock_old, gw_old, Np, Nnew,
                                                         gparent, gblock, gw, gpd_old, gpd);
    LAUNCH_CHECK();
}

template <typename T>
hipError_t launch_gather(hipStream_t s, Clouds<T> src, Clouds<T> dst, const int32_t* gblock, int64_t Ng, int S) {
    if (Ng <= 0) return hipSuccess;
    k_gather<T><<<(unsigned)std::min<int64_t>((Ng + 3) / 4, 2048), 256, 0, s>>>(src, dst, gblock, Ng, S);
    LAUNCH_CHECK();
}

template <typename T>
hipError_t launch_extract(hipStream_t s, Clouds<T> src, const int32_t* gblock, int64_t Ng, int S, double* out) {
    if (Ng <= 0) return hipSuccess;
    k_extract<T><<<nblocks(Ng * S, 256), 256, 0, s>>>(src, gblock, Ng, S, out);
    LAUNCH_CHECK();
}

template <typename T>
hipError_t launch_inject(hipStream_t s, const double* in, int64_t Ng, int S, Clouds<T> dst) {
    if (Ng <= 0) return hipSuccess;
    k_inject<T><<<nblocks(Ng * S, 256), 256, 0, s>>>(in, Ng, S, dst);
    LAUNCH_CHECK();
}

int64_t scan_tmp_size(int64_t n) { return (n + SCAN_TILE - 1) / SCAN_TILE + 1; }

static void scan(hipStream_t s, const int32_t* in, int32_t* out, int64_t n, int32_t* tmp) {
    const int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    if (nb > 0) k_scan_tiles<<<(unsigned)nb, SCAN_T, 0, s>>>(in, out, n, tmp);
    k_scan_sums<<<1, SCAN_T, 0, s>>>(tmp, nb, out + n);
    if (nb > 1) k_scan_add<<<nblocks(n, 256), 256, 0, s>>>(out, n, tmp);
}

hipError_t launch_scan_readout(hipStream_t s, const int32_t* in, int32_t* off, int n, int32_t* tmp, int32_t limit,
                               const int32_t* x0, int n0, const int32_t* x1, int32_t* out) {
    if (n <= SCAN_ONE) {
        k_scan_readout<<<1, SCAN_ONE_T, 0, s>>>(in, off, n, limit, x0, n0, x1, out);
    } else {
        scan(s, in, off, n, tmp);
        k_readout<<<1, 1024, 0, s>>>(off, n, limit, x0, n0, x1, out);
    }
    LAUNCH_CHECK();
}

hipError_t launch_outputs(hipStream_t s, const int32_t* nmerged, const int32_t* nkeep, int n, int32_t* tmp,
                          int32_t limit, const int32_t* x1, int32_t* mergeoff, int32_t* keepoff, int32_t* off,
                          int32_t* out) {
    if (n <= SCAN_ONE) {
        k_outputs<<<1, SCAN_ONE_T, 0, s>>>(nmerged, nkeep, n, limit, x1, mergeoff, keepoff, off, out);
    } else {
        scan(s, nmerged, mergeoff, n, tmp);
        scan(s, nkeep, keepoff, n, tmp);
        k_add_offsets<<<nblocks((int64_t)n + 1, 256), 256, 0, s>>>(mergeoff, keepoff, n, off);
        k_readout<<<1, 1024, 0, s>>>(off, n, limit, mergeoff + n, 1, x1, out);
    }
    LAUNCH_CHECK();
}

/* explicit instantiations */
template hipError_t launch_materialize<float>(hipStream_t, Clouds<float>, Clouds<float>, const int32_t*,
                                              const int32_t*, const int32_t*, int64_t, int, LinearCVMotionModel3D,
                                              double, RigKeys, uint64_t, bool);
template hipError_t launch_materialize<double>(hipStream_t, Clouds<double>, Clouds<double>, const int32_t*,
                                               const int32_t*, const int32_t*, int64_t, int, LinearCVMotionModel3D,
                                               double, RigKeys, uint64_t, bool);
template hipError_t launch_fit<float>(hipStream_t, const FitArgs&, Clouds<float>, Clouds<float>);
template hipError_t launch_fit<double>(hipStream_t, const FitArgs&, Clouds<double>, Clouds<double>);
template hipError_t launch_fit_fix<float>(hipStream_t, const FitArgs&, Clouds<float>, Clouds<float>);
template hipError_t launch_fit_fix<double>(hipStream_t, const FitArgs&, Clouds<double>, Clouds<double>);
template hipError_t launch_nd_fill<float>(hipStream_t, const FitArgs&, Clouds<float>, Clouds<float>);
template hipError_t launch_nd_fill<double>(hipStream_t, const FitArgs&, Clouds<double>, Clouds<double>);
template hipError_t launch_sample<float>(hipStream_t, const SampleArgs&, Clouds<float>);
template hipError_t launch_sample<double>(hipStream_t, const SampleArgs&, Clouds<double>);
template hipError_t launch_gather<float>(hipStream_t, Clouds<float>, Clouds<float>, const int32_t*, int64_t, int);
template hipError_t launch_gather<double>(hipStream_t, Clouds<double>, Clouds<double>, const int32_t*, int64_t,
                                          int);
template hipError_t launch_extract<float>(hipStream_t, Clouds<float>, const int32_t*, int64_t, int, double*);
template hipError_t launch_extract<double>(hipStream_t, Clouds<double>, const int32_t*, int64_t, int, double*);
template hipError_t launch_inject<float>(hipStream_t, const double*, int64_t, int, Clouds<float>);
template hipError_t launch_inject<double>(hipStream_t, const double*, int64_t, int, Clouds<double>);

}  // namespace scphd

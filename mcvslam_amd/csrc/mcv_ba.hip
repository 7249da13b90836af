// Bundle-adjustment linearization kernels for gfx950.
//
//   k_ba_linearize  EdgeSE3XYZ2Camera::computeError + linearizeOplus
//                   (include/OptimizeTypes.hpp:80-113), chi2 and the Huber
//                   weight (ThirdParty/g2o/g2o/core/base_edge.h:94-97,
//                   core/robust_kernel_impl.cpp:65-78), all edges at once
//   k_ba_linearize_group  the same for one (frame, camera) edge group
//   k_ba_stereo_linearize EdgeStereoSE3ProjectXYZ (3-row stereo edge)
//   k_ba_outliers   the chi2 outlier test of FilterCallBack_Chi2
//   k_ba_point_adj  sum_obs J_point^T g per point (CSR by point)
//   k_ba_pose_adj   sum_obs J_pose^T g per frame (observation list by frame)
//
// Arithmetic is FP32.  The residual e = (u - cx) - fx * X / Z subtracts two
// numbers of a few hundred pixels to get about one pixel, so the camera-frame
// point and the projection are carried as unevaluated float pairs
// (hi + lo, error-free transforms with fmaf): the point and pose state come
// in as such pairs too, which keeps the FP64 state of the optimizer.  The
// Jacobians, chi2 and weight are plain FP32.
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mcv {

struct f2 {
    float hi, lo;
};

__device__ __forceinline__ f2 two_sum(float a, float b) {
    const float s = a + b;
    const float bb = s - a;
    const float e = (a - (s - bb)) + (b - bb);
    return {s, e};
}
__device__ __forceinline__ f2 fast_two_sum(float a, float b) {
    const float s = a + b;
    return {s, b - (s - a)};
}
__device__ __forceinline__ f2 two_prod(float a, float b) {
    const float p = a * b;
    return {p, __builtin_fmaf(a, b, -p)};
}
__device__ __forceinline__ f2 df_add(f2 a, f2 b) {
    f2 s = two_sum(a.hi, b.hi);
    const f2 t = two_sum(a.lo, b.lo);
    s.lo += t.hi;
    s = fast_two_sum(s.hi, s.lo);
    s.lo += t.lo;
    return fast_two_sum(s.hi, s.lo);
}
__device__ __forceinline__ f2 df_neg(f2 a) { return {-a.hi, -a.lo}; }
__device__ __forceinline__ f2 df_mul(f2 a, f2 b) {
    f2 p = two_prod(a.hi, b.hi);
    p.lo = __builtin_fmaf(a.hi, b.lo, p.lo);
    p.lo = __builtin_fmaf(a.lo, b.hi, p.lo);
    return fast_two_sum(p.hi, p.lo);
}
__device__ __forceinline__ f2 df_mul_f(f2 a, float b) {
    f2 p = two_prod(a.hi, b);
    p.lo = __builtin_fmaf(a.lo, b, p.lo);
    return fast_two_sum(p.hi, p.lo);
}
__device__ __forceinline__ f2 df_div(f2 a, f2 b) {
    const float q1 = a.hi / b.hi;
    f2 r = df_add(a, df_neg(df_mul_f(b, q1)));
    const float q2 = r.hi / b.hi;
    r = df_add(r, df_neg(df_mul_f(b, q2)));
    const float q3 = r.hi / b.hi;
    const f2 q = fast_two_sum(q1, q2);
    return df_add(q, f2{q3, 0.f});
}

// Per (frame, camera) pair.  Tcw = Tcb * Tbw as float pairs for the
// residual; Tbw and Rcb in float for the Jacobians.
struct BAPair {
    float Rh[9], Rl[9];   // R_cw hi / lo, row-major
    float th[3], tl[3];   // t_cw hi / lo
    float Rbw[9], tbw[3]; // body from world
    float Rcb[9];         // camera from body
    float fx, fy, cx, cy, delta;
    float pad[3];
};

struct BAObs {
    const float2* uv;       // M
    const uint32_t* pt;     // M point index
    const uint32_t* pair;   // M (frame, camera) pair index
    const float* isig;      // M inverse level sigma^2
    int M;
};

struct BAOut {
    float* planes;   // 22 planes of M floats: e_u e_v chi2 w Jpose[12] Jpoint[6]
    long long stride;
};

// a / b as a float pair, from inv ~ 1 / b.hi (v_rcp_f32, 1 ulp): three
// quotient digits, each remainder taken exactly, so the result carries the
// accuracy of the pair arithmetic and no division is correctly rounded
__device__ __forceinline__ f2 df_div_rcp(f2 a, f2 b, float inv) {
    const float q1 = a.hi * inv;
    f2 r = df_add(a, df_neg(df_mul_f(b, q1)));
    const float q2 = r.hi * inv;
    r = df_add(r, df_neg(df_mul_f(b, q2)));
    const float q3 = r.hi * inv;
    return df_add(fast_two_sum(q1, q2), f2{q3, 0.f});
}

constexpr int kPairWords = (int)(sizeof(BAPair) / 4);
constexpr int kLdsPairs = 192;  // (frame, camera) pairs that fit the LDS copy

// Inputs of one observation: the streamed record and its gathered point.
struct BAIn {
    float2 uv;
    uint32_t pt, pair;
    float isig;
    float4 ph, pl;
};

__device__ __forceinline__ void ba_load_obs(int i, const BAObs& ob, BAIn& in) {
    in.uv = ob.uv[i];
    in.pt = ob.pt[i];
    in.pair = ob.pair[i];
    in.isig = ob.isig[i];
}

__device__ __forceinline__ void ba_load_point(const float4* __restrict__ pts_hi, const float4* __restrict__ pts_lo,
                                              BAIn& in) {
    in.ph = pts_hi[in.pt];
    in.pl = pts_lo[in.pt];
}

// kNt: streaming (non-temporal) stores for the output planes; this kernel
// never reads them back
// Plane k of observation i: the plane base is uniform (scalar registers) and
// the byte offset 4 i a 32-bit lane value, so each store takes one address
// register instead of a 64-bit pointer per plane.
template <bool kNt>
__device__ __forceinline__ void ba_store(const BAOut& out, int k, uint32_t off, float v) {
    float* p = reinterpret_cast<float*>(reinterpret_cast<char*>(out.planes + (long long)k * out.stride) + off);
    if (kNt) __builtin_nontemporal_store(v, p);
    else *p = v;
}

// Linearization modes: every plane; e, chi2 and w only (the LM trials'
// computeActiveErrors); everything but J_point (edges whose point is fixed:
// EdgeSE3XYZ2CameraOnlyPose, include/OptimizeTypes.hpp:20-68, has the same
// residual and J_pose, and a fixed point's J_point is never used).
constexpr int kBaFull = 0, kBaResidual = 1, kBaPoseOnly = 2;

// e, chi2 and the Huber weight of one edge, and the camera-frame point and
// reciprocal depth its Jacobians start from
struct BAEdge {
    float e0, e1, chi2, w, x, y, iz;
};

__device__ __forceinline__ BAEdge ba_residual(const BAIn& in, const BAPair& T) {
    const float2 uv = in.uv;
    const float isig = in.isig;
    const float4 ph = in.ph, pl = in.pl;
    const f2 P[3] = {{ph.x, pl.x}, {ph.y, pl.y}, {ph.z, pl.z}};
    // P_c = R_cw P_w + t_cw (float pairs)
    f2 C[3];
#pragma unroll
    for (int r = 0; r < 3; r++) {
        f2 acc = {T.th[r], T.tl[r]};
#pragma unroll
        for (int k = 0; k < 3; k++) acc = df_add(acc, df_mul(f2{T.Rh[3 * r + k], T.Rl[3 * r + k]}, P[k]));
        C[r] = acc;
    }
    // e = (obs - c) - f * X / Z
    const float iz = __builtin_amdgcn_rcpf(C[2].hi);
    const f2 qx = df_div_rcp(C[0], C[2], iz);
    const f2 qy = df_div_rcp(C[1], C[2], iz);
    const f2 eu = df_add(two_sum(uv.x, -T.cx), df_neg(df_mul_f(qx, T.fx)));
    const f2 ev = df_add(two_sum(uv.y, -T.cy), df_neg(df_mul_f(qy, T.fy)));
    const float e0 = eu.hi + eu.lo, e1 = ev.hi + ev.lo;
    const float chi2 = e0 * (isig * e0) + e1 * (isig * e1);
    const float d2 = T.delta * T.delta;
    const float w = chi2 <= d2 ? 1.f : T.delta * __builtin_amdgcn_rsqf(chi2);
    return BAEdge{e0, e1, chi2, w, C[0].hi, C[1].hi, iz};
}

// J_pose (2x6) of one edge (FP32).  Jpi = [[fx/z, 0, -fx x/z^2], [0, fy/z, -fy y/z^2]]:
// j00, j02, j11, j12
__device__ __forceinline__ void ba_jpi(const BAEdge& E, const BAPair& T, float& j00, float& j02, float& j11, float& j12) {
    j00 = T.fx * E.iz;
    j02 = -T.fx * E.x * (E.iz * E.iz);
    j11 = T.fy * E.iz;
    j12 = -T.fy * E.y * (E.iz * E.iz);
}

__device__ __forceinline__ void ba_jpose(const BAIn& in, const BAEdge& E, const BAPair& T, float (&Jp)[12]) {
    float j00, j02, j11, j12;
    ba_jpi(E, T, j00, j02, j11, j12);
    const float4 ph = in.ph;
    // P_b = R_bw P_w + t_bw; M = Jpi R_cb; J_pose = [M [P_b]x | -M]
    float pb[3];
#pragma unroll
    for (int r = 0; r < 3; r++) pb[r] = T.Rbw[3 * r] * ph.x + T.Rbw[3 * r + 1] * ph.y + T.Rbw[3 * r + 2] * ph.z + T.tbw[r];
    float Mr[6];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        Mr[k] = j00 * T.Rcb[k] + j02 * T.Rcb[6 + k];
        Mr[3 + k] = j11 * T.Rcb[3 + k] + j12 * T.Rcb[6 + k];
    }
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const float m0 = Mr[3 * r], m1 = Mr[3 * r + 1], m2 = Mr[3 * r + 2];
        // M * [p]x, [p]x = [[0,-z,y],[z,0,-x],[-y,x,0]]
        Jp[6 * r + 0] = m1 * pb[2] - m2 * pb[1];
        Jp[6 * r + 1] = m2 * pb[0] - m0 * pb[2];
        Jp[6 * r + 2] = m0 * pb[1] - m1 * pb[0];
        Jp[6 * r + 3] = -m0;
        Jp[6 * r + 4] = -m1;
        Jp[6 * r + 5] = -m2;
    }
}

template <bool kNt>
__device__ __forceinline__ void ba_edge(int i, const BAIn& in, const BAPair& T, BAOut out, int mode) {
    const BAEdge E = ba_residual(in, T);
    const uint32_t off = (uint32_t)i * 4u;
    ba_store<kNt>(out, 0, off, E.e0);
    ba_store<kNt>(out, 1, off, E.e1);
    ba_store<kNt>(out, 2, off, E.chi2);
    ba_store<kNt>(out, 3, off, E.w);
    if (mode == kBaResidual) return;
    // J_point = -Jpi R_cw
    if (mode != kBaPoseOnly) {
        float j00, j02, j11, j12;
        ba_jpi(E, T, j00, j02, j11, j12);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            ba_store<kNt>(out, 16 + k, off, -(j00 * T.Rh[k] + j02 * T.Rh[6 + k]));
            ba_store<kNt>(out, 19 + k, off, -(j11 * T.Rh[3 + k] + j12 * T.Rh[6 + k]));
        }
    }
    float Jp[12];
    ba_jpose(in, E, T, Jp);
#pragma unroll
    for (int k = 0; k < 12; k++) ba_store<kNt>(out, 4 + k, off, Jp[k]);
}

// One observation per thread per step, grid-stride.  kLds: the (frame,
// camera) table (npairs <= kLdsPairs) is copied to dynamic LDS once per
// workgroup, so the per-observation parameter reads are LDS gathers
// (53-word records: odd stride, distinct records fall in distinct banks)
// instead of ~50 scattered global loads.  kIlp observations are in flight
// per thread: all their loads are issued before the first is computed.
template <bool kLds, int kIlp, bool kNt>
__global__ __launch_bounds__(1024) void k_ba_linearize(BAObs ob, const float4* __restrict__ pts_hi,
                                                       const float4* __restrict__ pts_lo,
                                                       const BAPair* __restrict__ pairs, int npairs, BAOut out,
                                                       int mode) {
    extern __shared__ float s_pairs[];  // npairs * kPairWords floats when kLds
    if (kLds) {
        const float* src = reinterpret_cast<const float*>(pairs);
        for (int k = threadIdx.x; k < npairs * kPairWords; k += blockDim.x) s_pairs[k] = src[k];
        __syncthreads();
    }
    const int stride = gridDim.x * blockDim.x;
    if (kIlp == 1) {
        for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < ob.M; i += stride) {
            const uint32_t pr = ob.pair[i];
            const BAPair& T = kLds ? *reinterpret_cast<const BAPair*>(s_pairs + pr * kPairWords) : pairs[pr];
            BAIn in;
            ba_load_obs(i, ob, in);
            ba_load_point(pts_hi, pts_lo, in);
            ba_edge<kNt>(i, in, T, out, mode);
        }
        return;
    }
    for (int i0 = blockIdx.x * blockDim.x + threadIdx.x; i0 < ob.M; i0 += kIlp * stride) {
        BAIn in[kIlp];
#pragma unroll
        for (int u = 0; u < kIlp; u++)
            if (i0 + u * stride < ob.M) ba_load_obs(i0 + u * stride, ob, in[u]);
#pragma unroll
        for (int u = 0; u < kIlp; u++)
            if (i0 + u * stride < ob.M) ba_load_point(pts_hi, pts_lo, in[u]);
#pragma unroll
        for (int u = 0; u < kIlp; u++) {
            const int i = i0 + u * stride;
            if (i >= ob.M) break;
            const BAPair& T = kLds ? *reinterpret_cast<const BAPair*>(s_pairs + in[u].pair * kPairWords)
                                   : pairs[in[u].pair];
            ba_edge<kNt>(i, in[u], T, out, mode);
        }
    }
}

// The plain launch pattern: the observations of one (frame, camera) edge
// group (list[0..n)), one launch per group.
__global__ __launch_bounds__(256) void k_ba_linearize_group(BAObs ob, const float4* __restrict__ pts_hi,
                                                            const float4* __restrict__ pts_lo,
                                                            const BAPair* __restrict__ pairs, const int* list, int n,
                                                            BAOut out, int mode) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int i = list[k];
    BAIn in;
    ba_load_obs(i, ob, in);
    ba_load_point(pts_hi, pts_lo, in);
    ba_edge<false>(i, in, pairs[in.pair], out, mode);
}

// ---------------------------------------------------------------------------
// Stereo edge EdgeStereoSE3ProjectXYZ (include/OptimizeTypes.hpp:119-157,
// src/OptimizeTypes.cpp:12-58).  The pose vertex is the keyframe pose (the
// left camera is the body).  cam_project_uv_u rounds the inverse depth to
// float and forms bf * invz as a float product; the rest is double in the
// reference, float pairs here.  32 output planes of M floats:
// e_u e_v e_ur chi2 w J_pose[3x6] J_point[3x3].
struct FramePose {
    float Rh[9], Rl[9];  // R_cw hi / lo
    float th[3], tl[3];  // t_cw hi / lo
};

struct StereoCam {
    float fx, fy, cx, cy, bf, delta;
};

struct BAStereoObs {
    const float* obs;       // M x 3: u, v, u_right
    const uint32_t* pt;
    const uint32_t* fr;
    const float* isig;
    int M;
};

struct StereoEdge {
    float e[3], chi2, w, x, y, z;
};

__device__ __forceinline__ StereoEdge stereo_residual(const BAStereoObs& ob, int i, const float4* __restrict__ pts_hi,
                                                      const float4* __restrict__ pts_lo, const FramePose& T,
                                                      const StereoCam& cam) {
    const float ou = ob.obs[3 * i], ov = ob.obs[3 * i + 1], our = ob.obs[3 * i + 2];
    const float isig = ob.isig[i];
    const uint32_t pi = ob.pt[i];
    const float4 ph = pts_hi[pi], pl = pts_lo[pi];
    const f2 P[3] = {{ph.x, pl.x}, {ph.y, pl.y}, {ph.z, pl.z}};
    f2 C[3];
#pragma unroll
    for (int r = 0; r < 3; r++) {
        f2 acc = {T.th[r], T.tl[r]};
#pragma unroll
        for (int k = 0; k < 3; k++) acc = df_add(acc, df_mul(f2{T.Rh[3 * r + k], T.Rl[3 * r + k]}, P[k]));
        C[r] = acc;
    }
    // invz = (float)(1 / z), rounded from the pair quotient
    const f2 q = df_div_rcp(f2{1.f, 0.f}, C[2], __builtin_amdgcn_rcpf(C[2].hi));
    const float invz = q.hi + q.lo;
    const f2 ru = df_add(df_mul_f(df_mul_f(C[0], invz), cam.fx), f2{cam.cx, 0.f});
    const f2 rv = df_add(df_mul_f(df_mul_f(C[1], invz), cam.fy), f2{cam.cy, 0.f});
    const float bfi = cam.bf * invz;
    const f2 eu = df_add(f2{ou, 0.f}, df_neg(ru));
    const f2 ev = df_add(f2{ov, 0.f}, df_neg(rv));
    const f2 er = df_add(df_add(f2{our, 0.f}, df_neg(ru)), f2{bfi, 0.f});
    const float e0 = eu.hi + eu.lo, e1 = ev.hi + ev.lo, e2 = er.hi + er.lo;
    const float chi2 = isig * (e0 * e0 + e1 * e1 + e2 * e2);
    const float w = chi2 <= cam.delta * cam.delta ? 1.f : cam.delta * __builtin_amdgcn_rsqf(chi2);
    return StereoEdge{{e0, e1, e2}, chi2, w, C[0].hi, C[1].hi, C[2].hi};
}

// J_pose (3x6) of a stereo edge
__device__ __forceinline__ void stereo_jpose(const StereoEdge& E, const StereoCam& cam, float (&J)[18]) {
    const float x = E.x, y = E.y;
    const float iz = __builtin_amdgcn_rcpf(E.z), iz2 = iz * iz;
    const float fx = cam.fx, fy = cam.fy, bf = cam.bf;
    float *J0 = J, *J1 = J + 6, *J2 = J + 12;
    J0[0] = x * y * iz2 * fx;
    J0[1] = -(1.f + x * x * iz2) * fx;
    J0[2] = y * iz * fx;
    J0[3] = -iz * fx;
    J0[4] = 0.f;
    J0[5] = x * iz2 * fx;
    J1[0] = (1.f + y * y * iz2) * fy;
    J1[1] = -x * y * iz2 * fy;
    J1[2] = -x * iz * fy;
    J1[3] = 0.f;
    J1[4] = -iz * fy;
    J1[5] = y * iz2 * fy;
    J2[0] = J0[0] - bf * y * iz2;
    J2[1] = J0[1] + bf * x * iz2;
    J2[2] = J0[2];
    J2[3] = J0[3];
    J2[4] = 0.f;
    J2[5] = J0[5] - bf * iz2;
}

__global__ __launch_bounds__(256) void k_ba_stereo_linearize(BAStereoObs ob, const float4* __restrict__ pts_hi,
                                                             const float4* __restrict__ pts_lo,
                                                             const FramePose* __restrict__ poses, StereoCam cam,
                                                             BAOut out, int mode) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ob.M) return;
    const FramePose& T = poses[ob.fr[i]];
    const StereoEdge E = stereo_residual(ob, i, pts_hi, pts_lo, T, cam);
    const long long S = out.stride;
    float* o = out.planes + i;
    o[0] = E.e[0];
    o[S] = E.e[1];
    o[2 * S] = E.e[2];
    o[3 * S] = E.chi2;
    o[4 * S] = E.w;
    if (mode == kBaResidual) return;
    float J[18];
    stereo_jpose(E, cam, J);
#pragma unroll
    for (int k = 0; k < 18; k++) o[(5 + k) * S] = J[k];
    if (mode == kBaPoseOnly) return;
    const float x = E.x, y = E.y;
    const float iz = __builtin_amdgcn_rcpf(E.z), iz2 = iz * iz;
    const float fx = cam.fx, fy = cam.fy, bf = cam.bf;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float a = -fx * T.Rh[k] * iz + fx * x * T.Rh[6 + k] * iz2;
        const float b = -fy * T.Rh[3 + k] * iz + fy * y * T.Rh[6 + k] * iz2;
        o[(23 + k) * S] = a;
        o[(26 + k) * S] = b;
        o[(29 + k) * S] = a - bf * T.Rh[6 + k] * iz2;
    }
}

// FilterCallBack_Chi2 (src/PoseEstimation.cpp:132-151): flag = chi2 >= threshold.
__global__ __launch_bounds__(256) void k_ba_outliers(const float* chi2, int M, float threshold, uint8_t* flags) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < M) flags[i] = chi2[i] >= threshold ? 1 : 0;
}

// grad_point[p] = sum over the observations of p (CSR, observation order) of
// J_point^T g.  One thread per point, fixed summation order.
__global__ __launch_bounds__(256) void k_ba_point_adj(const float* planes, long long S, const float2* g,
                                                      const int* ptr, int P, float* gout) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    float a0 = 0.f, a1 = 0.f, a2 = 0.f;
    for (int i = ptr[p]; i < ptr[p + 1]; i++) {
        const float2 gi = g[i];
        a0 += planes[16 * S + i] * gi.x + planes[19 * S + i] * gi.y;
        a1 += planes[17 * S + i] * gi.x + planes[20 * S + i] * gi.y;
        a2 += planes[18 * S + i] * gi.x + planes[21 * S + i] * gi.y;
    }
    gout[3 * p] = a0;
    gout[3 * p + 1] = a1;
    gout[3 * p + 2] = a2;
}

// grad_pose[f][c] = sum over the observations of frame f of row c of J_pose^T
// g, one workgroup per frame and kC of the six components; each thread sums a
// strided slice, then a fixed-order tree reduction: deterministic.  A frame's
// observations lie some F apart in the planes, so what bounds it is whole lines
// of the planes pulled through a CU for a few values each.  The cut by component
// spreads them over more CUs, 4 loads in flight per thread; it costs the
// observation list and g once per component (pose_adj_shape).
template <int kThreads, int kC>
__global__ __launch_bounds__(kThreads) void k_ba_pose_adj(const float* planes, long long S, const float2* g,
                                                          const int* fptr, const int* fobs, float* gout) {
    constexpr int kLoads = kC == 1 ? 4 : 2;
    __shared__ float red[kC][kThreads / 64];
    const int f = blockIdx.x, c0 = kC * blockIdx.y;
    const float* pu = planes + (4 + c0) * S;
    const float* pv = planes + (10 + c0) * S;
    const int k1 = fptr[f + 1];
    float a[kC][kLoads] = {};
    for (int k = fptr[f] + threadIdx.x; k < k1; k += kLoads * kThreads) {
        int i[kLoads];
#pragma unroll
        for (int u = 0; u < kLoads; u++) i[u] = k + u * kThreads < k1 ? fobs[k + u * kThreads] : -1;
#pragma unroll
        for (int u = 0; u < kLoads; u++)
            if (i[u] >= 0) {
                const float2 gi = g[i[u]];
#pragma unroll
                for (int c = 0; c < kC; c++) a[c][u] += pu[c * S + i[u]] * gi.x + pv[c * S + i[u]] * gi.y;
            }
    }
#pragma unroll
    for (int c = 0; c < kC; c++) {
        float s = 0.f;
        if constexpr (kLoads == 4) s = (a[c][0] + a[c][1]) + (a[c][2] + a[c][3]);
        else s = a[c][0] + a[c][1];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if ((threadIdx.x & 63) == 0) red[c][threadIdx.x >> 6] = s;
    }
    __syncthreads();
    if (threadIdx.x < kC) {
        float t = 0.f;
        for (int w = 0; w < kThreads / 64; w++) t += red[threadIdx.x][w];
        gout[6 * f + c0 + threadIdx.x] = t;
    }
}

// Components per workgroup and threads.  Below about 500k observations the
// planes stay in L2 and the cut by component pays at any number of frames; above,
// only while it does not make more workgroups than CUs, which otherwise pull the
// same lines at different times.  us of an adjoint, <256, 6> / <256, 3> / <256, 1>
// / <1024, 1>: 10 frames of 15k observations 86 59 36 31, 5 of 300k 991 673 523
// 275, 42 of 36k 408 259 142 211, 100 of 20k 306 201 304 397, 200 of 10k 203 320
// 369 394, 1000 of 1000 194 206 241 239, 400 of 250 19 18 18 22, 2000 of 200 83
// 78 66 79.
struct PoseAdjShape {
    int threads, comps;
};
inline PoseAdjShape pose_adj_shape(int M, int F) {
    if (F <= 21) return {1024, 1};
    if (F <= 42 || M <= 500000) return {256, 1};
    return {256, F <= 128 ? 3 : 6};
}

// the residual planes as rows (e_u, e_v)
__global__ __launch_bounds__(256) void k_ba_residual_rows(const float* planes, long long S, float2* out) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < S) out[i] = make_float2(planes[i], planes[S + i]);
}

}  // namespace mcv

namespace mcv {

// ---------------------------------------------------------------------------
// Schur complement of the point blocks (BlockSolver::buildSystem +
// BlockSolver::solve, ThirdParty/g2o/g2o/core/block_solver.hpp:315-449,
// 463-520; quadratic form of BaseBinaryEdge::constructQuadraticForm,
// core/base_binary_edge.hpp:64-136), FP32, fixed summation orders, over the
// active mono (2-row, k_ba_linearize planes) and stereo (3-row,
// k_ba_stereo_linearize planes) edges; edge index i < M is mono edge i,
// i >= M stereo edge i - M.  Fixed points have no edge lists (their edges
// still enter H_pp and b_p through the frame lists); fixed frames have no
// pose block.  W = Huber weight * inv sigma^2.
//   k_schur_points  per point: H_ll = sum W J_x^T J_x, b_l = -sum W J_x^T e,
//       the Cholesky factor C of D = H_ll + lambda I and y = C^-1 b_l; per
//       (point, free frame) entry H_pl = sum W J_p^T J_x (6x3), kept as
//       Z = H_pl C^-T, so that H_pl,i D^-1 H_pl,j^T = Z_i Z_j^T and
//       H_pl D^-1 b_l = Z y
//   k_schur_edges, k_schur_edge_sums  per free frame: H_pp = sum W J_p^T J_p,
//       b_p = -sum W J_p^T e
//   k_schur_items, k_schur_assemble  per free-frame pair block (i <= j):
//       S_ij = [i == j](H_pp + lambda I) - sum over shared points Z_i Z_j^T,
//       b_schur = b_p - sum Z y
//   k_schur_backsub  x_l = C^-T (y - sum Z^T x_p)
// What bounds them: the planes (88 B per mono edge) and the entry rows (96 B)
// from memory; every plane is read in edge order, so that a wave's loads are
// whole lines.  50 keyframes, 200k points, 1.5M edges, 1.2M entries, 5.4M
// items: points 131, edges 47 + 9, items 139, assembly 6 us (one thread per
// point, one workgroup per frame and per pair block: 391, 675 and 806 us).
constexpr int kZRow = 24;          // floats per entry row: Z (6x3 row-major), Z y (6)
constexpr int kPointRec = 12;      // floats per point: c10 c20 c21, 1/c00 1/c11 1/c22, y, b_l
constexpr int kEdgeChunk = 512;    // edges per workgroup of k_schur_edges
constexpr int kItemSums = 40;      // sums of an item chunk (36, or 27 on the diagonal)
constexpr int kFrameSums = 27;     // per frame: H_pp upper triangle by rows, each row followed by b_p's entry
// Rows of frame sums take 0.2 Fp bytes an edge with one per chunk.  Below this
// bound every chunk has its own (1.5M edges, 50 frames: 16 MB); it leaves a row
// for each CU up to kMaxFreeFrames.
constexpr size_t kEpartBytes = 256u << 20;

struct ItemChunk {
    int i0, i1;  // items [i0, i1) of one frame-pair block
    int out;     // row of ipart: the chunks of a block in order, blocks in order
    int diag;
};

// ---- edge lists of the Schur complement, built on the device ------------------
// From the edges in point order (mono: CSR pptr; stereo: CSR sptr over slist)
// and every edge's free frame: per free point its active edges and, by free
// frame, its entries and their edges; the entries' rows by (frame, point); per
// frame pair the items (row_i, row_j) in point order.  All orders are fixed.
// Bound by the edge and entry arrays, read a few times; 1.5M edges, 1.2M
// entries, 5.4M items: the host loops this replaces took 50 ms.
constexpr int kWindows = 32;  // windows of a frame's rows, for the item chunks

// frame-pair blocks (i <= j): the upper triangle by rows
__host__ __device__ __forceinline__ int block_of(int i, int j, int Fp) { return i * Fp - i * (i - 1) / 2 + (j - i); }

struct SchurBuild {
    const int* pptr;
    const int* sptr;          // null without stereo edges
    const int* slist;
    const uint32_t* pair;     // mono: frame * C + cam
    const uint32_t* sfr;      // stereo: frame
    const uint8_t* act_m;     // or null: every edge active
    const uint8_t* act_s;
    const uint8_t* pfix;      // or null: no point fixed
    const int* fidx;          // frame -> free frame or -1
    int M, Ms, P, C, Fp, words, ntile;  // words: u64 per frame mask; ntile: tiles of 256 entries (stride of thist)
    int* ef;                  // M + Ms: the edge's free frame, -1 fixed frame, -2 inactive
    unsigned long long* mask; // P x words: the free frames that see a point
    int *pe_ptr, *po_ptr, *pf_ptr;      // P + 1 each
    int* btot;                // per 256 points: (edges, edges of free frames, entries), then their totals
    int *pe, *pf_obs, *pf_obs_ptr, *pf_frame, *pf_point, *pf_row, *row_q;
    int* thist;               // Fp x ntile
    int* fbase;               // Fp + 1: first row of a frame
    int* tbase;               // Fp + 1: first 64-row tile of a frame
    int* tcount;              // row tiles x Fp
    int* win;                 // nblk x (kWindows + 1): items before each window, then all; or null:
    int* btotal;              // nblk: all items
    const int* blk_ptr;       // nblk
    int2* items;
    uint16_t *eptr, *elist;
    int nchunk_m;             // chunks of the mono edges; the stereo edges' follow
};

__global__ __launch_bounds__(256) void k_sb_edges(SchurBuild b) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= b.M + b.Ms) return;
    const bool mono = e < b.M;
    const uint8_t* act = mono ? b.act_m : b.act_s;
    const int k = mono ? e : e - b.M;
    b.ef[e] = act && !act[k] ? -2 : b.fidx[mono ? b.pair[k] / (uint32_t)b.C : b.sfr[k]];
}

// f(edge, its free frame) for every active edge of point p, mono first
template <typename F>
__device__ __forceinline__ void point_edges(const SchurBuild& b, int p, F f) {
    for (int e = b.pptr[p]; e < b.pptr[p + 1]; e++)
        if (b.ef[e] != -2) f(e, b.ef[e]);
    if (b.sptr)
        for (int t = b.sptr[p]; t < b.sptr[p + 1]; t++) {
            const int e = b.M + b.slist[t];
            if (b.ef[e] != -2) f(e, b.ef[e]);
        }
}

// exclusive scan of one int per thread over the workgroup; ws: 17 ints
__device__ __forceinline__ int wg_excl(int v, int* ws, int& total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) ws[w] = x;
    __syncthreads();
    int base = 0;
    total = 0;
    for (int k = 0; k < nw; k++) {
        base += k < w ? ws[k] : 0;
        total += ws[k];
    }
    __syncthreads();
    return base + x - v;
}

// per point: counts (their scans within the 256 points), and the frame mask
__global__ __launch_bounds__(256) void k_sb_points(SchurBuild b) {
    __shared__ int ws[17];
    const int p = blockIdx.x * 256 + threadIdx.x;
    int n = 0, nf = 0, nd = 0;
    if (p < b.P) {
        unsigned long long* m = b.mask + (long long)p * b.words;
        for (int k = 0; k < b.words; k++) m[k] = 0;
        if (!(b.pfix && b.pfix[p])) {
            unsigned long long m0 = 0;
            point_edges(b, p, [&](int, int f) {
                n++;
                if (f < 0) return;
                nf++;
                if (f < 64) m0 |= 1ull << f;
                else m[f >> 6] |= 1ull << (f & 63);
            });
            if (b.words) m[0] = m0;
            for (int k = 0; k < b.words; k++) nd += __popcll(m[k]);
        }
    }
    int t0, t1, t2;
    const int a0 = wg_excl(n, ws, t0), a1 = wg_excl(nf, ws, t1), a2 = wg_excl(nd, ws, t2);
    if (p < b.P) {
        b.pe_ptr[p] = a0;
        b.po_ptr[p] = a1;
        b.pf_ptr[p] = a2;
    }
    if (threadIdx.x == 0) {
        b.btot[3 * blockIdx.x] = t0;
        b.btot[3 * blockIdx.x + 1] = t1;
        b.btot[3 * blockIdx.x + 2] = t2;
    }
}

// the 256-point blocks' offsets, the totals after them (one workgroup)
__global__ __launch_bounds__(1024) void k_sb_offsets(SchurBuild b, int nb) {
    __shared__ int ws[17];
    int run[3] = {0, 0, 0};
    for (int k0 = 0; k0 < nb; k0 += 1024) {
        const int k = k0 + threadIdx.x;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            int tot;
            const int x = wg_excl(k < nb ? b.btot[3 * k + c] : 0, ws, tot);
            if (k < nb) b.btot[3 * k + c] = run[c] + x;
            run[c] += tot;
        }
    }
    if (threadIdx.x == 0)
        for (int c = 0; c < 3; c++) b.btot[3 * nb + c] = run[c];
}

// per point: final offsets, its edge list, its entries by frame and their edges
__global__ __launch_bounds__(256) void k_sb_fill(SchurBuild b, int nb) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= b.P) return;
    const int* bo = b.btot + 3 * blockIdx.x;
    int n = b.pe_ptr[p] + bo[0], o = b.po_ptr[p] + bo[1], q = b.pf_ptr[p] + bo[2];
    b.pe_ptr[p] = n;
    b.pf_ptr[p] = q;
    if (p == b.P - 1) {
        b.pe_ptr[b.P] = b.btot[3 * nb];
        b.pf_ptr[b.P] = b.btot[3 * nb + 2];
        b.pf_obs_ptr[b.btot[3 * nb + 2]] = b.btot[3 * nb + 1];
    }
    if (b.pfix && b.pfix[p]) return;
    point_edges(b, p, [&](int e, int) { b.pe[n++] = e; });
    for (int k = 0; k < b.words; k++)
        for (unsigned long long m = b.mask[(long long)p * b.words + k]; m; m &= m - 1, q++) {
            const int f = 64 * k + __builtin_ctzll(m);
            b.pf_obs_ptr[q] = o;
            b.pf_frame[q] = f;
            b.pf_point[q] = p;
            point_edges(b, p, [&](int e, int fe) {
                if (fe == f) b.pf_obs[o++] = e;
            });
        }
}

// entries per frame of 256 entries
__global__ __launch_bounds__(256) void k_sb_hist(SchurBuild b, int nb) {
    extern __shared__ int s_cnt[];  // Fp
    const int npf = b.btot[3 * nb + 2], q = blockIdx.x * 256 + threadIdx.x;
    for (int f = threadIdx.x; f < b.Fp; f += 256) s_cnt[f] = 0;
    __syncthreads();
    if (q < npf) atomicAdd(&s_cnt[b.pf_frame[q]], 1);
    __syncthreads();
    for (int f = threadIdx.x; f < b.Fp; f += 256) b.thist[(long long)f * b.ntile + blockIdx.x] = s_cnt[f];
}

// per frame: the tiles' offsets; the frame's entries to fbase[f + 1]
__global__ __launch_bounds__(1024) void k_sb_frames(SchurBuild b) {
    __shared__ int ws[17];
    int* h = b.thist + (long long)blockIdx.x * b.ntile;
    int run = 0;
    for (int k0 = 0; k0 < b.ntile; k0 += 1024) {
        const int k = k0 + threadIdx.x;
        int tot;
        const int x = wg_excl(k < b.ntile ? h[k] : 0, ws, tot);
        if (k < b.ntile) h[k] = run + x;
        run += tot;
    }
    if (threadIdx.x == 0) b.fbase[blockIdx.x + 1] = run;
}

__global__ __launch_bounds__(1024) void k_sb_bases(SchurBuild b) {
    __shared__ int ws[17];
    int r0 = 0, r1 = 0;
    for (int k0 = 0; k0 < b.Fp; k0 += 1024) {
        const int k = k0 + threadIdx.x;
        const int n = k < b.Fp ? b.fbase[k + 1] : 0;
        int t0, t1;
        const int x0 = wg_excl(n, ws, t0), x1 = wg_excl((n + 63) / 64, ws, t1);
        if (k < b.Fp) {
            b.fbase[k + 1] = r0 + x0 + n;
            b.tbase[k + 1] = r1 + x1 + (n + 63) / 64;
        }
        r0 += t0;
        r1 += t1;
    }
    if (threadIdx.x == 0) b.fbase[0] = b.tbase[0] = 0;
}

// row of every entry: rank among the tile's earlier entries of its frame
__global__ __launch_bounds__(256) void k_sb_rows(SchurBuild b, int nb) {
    __shared__ int s_f[256];
    const int npf = b.btot[3 * nb + 2], q = blockIdx.x * 256 + threadIdx.x;
    const int f = q < npf ? b.pf_frame[q] : -1;
    s_f[threadIdx.x] = f;
    __syncthreads();
    if (q >= npf) return;
    int r = 0;
    for (int k = 0; k < (int)threadIdx.x; k++) r += s_f[k] == f ? 1 : 0;
    r += b.fbase[f] + b.thist[(long long)f * b.ntile + blockIdx.x];
    b.pf_row[q] = r;
    b.row_q[r] = q;
}

// Items of 64 rows of one frame i (one wave; rows are in point order): with
// frame j, row l has an item when its point sees j, and its place among the
// tile's items of (i, j) is the number of earlier rows that do.
template <bool kFill>
__global__ __launch_bounds__(256) void k_sb_items(SchurBuild b) {
    const int tile = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (tile >= b.tbase[b.Fp]) return;
    int lo = 0, hi = b.Fp - 1;  // the last frame whose first tile is <= tile (frames without rows have none)
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (b.tbase[mid] <= tile) lo = mid; else hi = mid - 1;
    }
    const int i = lo, r = b.fbase[i] + 64 * (tile - b.tbase[i]) + lane;
    const bool on = r < b.fbase[i + 1];
    int q = on ? b.row_q[r] : 0;
    const unsigned long long* m = b.mask + (long long)(on ? b.pf_point[q] : 0) * b.words;
    for (int w = i >> 6; w < b.words; w++) {
        unsigned long long mw = on ? m[w] : 0;
        if (w == i >> 6) mw &= ~0ull << (i & 63);
        for (int j = max(i, 64 * w); j < min(b.Fp, 64 * w + 64); j++) {
            const bool has = (mw >> (j & 63)) & 1ull;
            const unsigned long long v = __ballot(has);
            if constexpr (kFill) {
                if (v == 0) continue;
                const int at = b.blk_ptr[block_of(i, j, b.Fp)] + b.tcount[(long long)tile * b.Fp + j];
                // q walks the point's entries from frame i on
                if (has) b.items[at + (int)lanes_below(v)] = make_int2(r, b.pf_row[q++]);
            } else if (lane == 0) {
                b.tcount[(long long)tile * b.Fp + j] = __popcll(v);
            }
        }
    }
}

// per block (i, j): the tiles' offsets, and the items before each window of
// frame i's tiles (win[kWindows]: all of them).  One wave per block.
__global__ __launch_bounds__(64) void k_sb_blocks(SchurBuild b) {
    const int i = blockIdx.y, j = blockIdx.x;
    if (j < i) return;
    const int t0 = b.tbase[i], nt = b.tbase[i + 1] - t0, lane = threadIdx.x;
    const int blk = block_of(i, j, b.Fp);
    int* win = b.win ? b.win + (long long)blk * (kWindows + 1) : nullptr;
    int run = 0;
    for (int k0 = 0; k0 < nt; k0 += 64) {
        const int k = k0 + lane;
        int* c = b.tcount + (long long)(t0 + k) * b.Fp + j;
        const int v = k < nt ? *c : 0;
        int x = v;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (k < nt) {
            *c = run + x - v;
            // windows whose first tile (w * nt / kWindows) is k
            if (win)
                for (int w = (int)(((long long)k * kWindows + nt - 1) / nt);
                     w < kWindows && (int)((long long)w * nt / kWindows) == k; w++)
                    win[w] = run + x - v;
        }
        run += __shfl(x, 63, 64);
    }
    if (!win) {
        if (lane == 0) b.btotal[blk] = run;
        return;
    }
    if (nt == 0 && lane < kWindows) win[lane] = 0;
    if (lane == 0) win[kWindows] = run;
}

// the windows of some blocks (i, j) that have items, from the tiles' offsets
__global__ __launch_bounds__(256) void k_sb_windows(SchurBuild b, const int2* blocks, int n, int* win) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n * kWindows) return;
    const int2 ij = blocks[k / kWindows];
    const int w = k % kWindows, t0 = b.tbase[ij.x], nt = b.tbase[ij.x + 1] - t0;
    win[k] = b.tcount[(t0 + (long long)w * nt / kWindows) * b.Fp + ij.y];
}

// the frame-sorted edge lists of k_schur_edges' chunks
__global__ __launch_bounds__(512) void k_sb_chunks(SchurBuild b) {
    extern __shared__ int s_cnt[];  // Fp + 1, after it kEdgeChunk frames
    int* s_f = s_cnt + b.Fp + 1;
    const bool st = (int)blockIdx.x >= b.nchunk_m;
    const int k = (int)(st ? blockIdx.x - b.nchunk_m : blockIdx.x) * kEdgeChunk + threadIdx.x;
    int f = -1;
    if (k < (st ? b.Ms : b.M)) f = max(b.ef[st ? b.M + k : k], -1);
    for (int i = threadIdx.x; i <= b.Fp; i += 512) s_cnt[i] = 0;
    s_f[threadIdx.x] = f;
    __syncthreads();
    if (f >= 0) atomicAdd(&s_cnt[f + 1], 1);
    __syncthreads();
    if (threadIdx.x < 64) {
        int run = 0;
        for (int i0 = 0; i0 <= b.Fp; i0 += 64) {
            const int i = i0 + threadIdx.x;
            int x = i <= b.Fp ? s_cnt[i] : 0;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(x, o, 64);
                if ((int)threadIdx.x >= o) x += y;
            }
            if (i <= b.Fp) s_cnt[i] = run + x;
            run += __shfl(x, 63, 64);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i <= b.Fp; i += 512)
        b.eptr[(long long)blockIdx.x * (b.Fp + 1) + i] = (uint16_t)s_cnt[i];
    if (f >= 0) {
        int r = s_cnt[f];
        for (int t = 0; t < (int)threadIdx.x; t++) r += s_f[t] == f ? 1 : 0;
        b.elist[(long long)blockIdx.x * kEdgeChunk + r] = (uint16_t)threadIdx.x;
    }
}

struct SchurArgs {
    const float* planes;    // mono planes (22 of stride S)
    long long S;
    const float* isig;
    int M;
    const float* splanes;   // stereo planes (32 of stride SS)
    long long SS;
    const float* sisig;
    const int* pe_ptr;      // P + 1: active edges of free point p
    const int* pe;
    const int* pf_ptr;      // per point: first pf entry (P + 1)
    const int* pf_obs_ptr;  // per pf entry: range in pf_obs (npf + 1)
    const int* pf_obs;      // edge indices grouped by pf
    const int* pf_frame;    // free frame of each pf entry
    const int* pf_row;      // row of each pf entry: rows are ordered by (frame, point)
    // chunks of kEdgeChunk consecutive edges, the mono edges' first: the local
    // numbers of its active edges of free frames, by frame
    const uint16_t* eptr;   // per chunk, Fp + 1: the frames' ranges in its list
    const uint16_t* elist;  // per chunk, kEdgeChunk
    int nchunk_m, Ms;
    const ItemChunk* ichunk;
    const int* blk_chunk;   // per block: its first item chunk (nblk + 1)
    const int2* items;      // (row_i, row_j), by block, then by point
    int P, Fp, nechunk, esub, nichunk;
    int egroup, nerow;      // chunks per workgroup of k_schur_edges, its workgroups
    float lambda;
    float* prec;            // P x kPointRec
    float* hd;              // P x 3: diagonal of H_ll
    float* Z;               // npf x kZRow
    float* epart;           // (nerow * esub) x (kFrameSums * Fp)
    float* ipart;           // nichunk x kItemSums
    float* Hpp;             // Fp x 36 (without lambda)
    float* bs;              // Fp x 6 (b_schur)
    float* bp;              // Fp x 6 (b_p)
    float* Sout;            // (6 Fp)^2 row-major
};

// one edge's planes: e row r at base[r * st], J_pose (r, c) at
// base[(jp + 6 r + c) * st], J_point (r, c) at base[(jx + 3 r + c) * st]
struct EdgeRef {
    const float* base;
    long long st;
    int rows, jp, jx;
    float W;
    __device__ __forceinline__ float e(int r) const { return base[r * st]; }
    __device__ __forceinline__ float Jp(int r, int c) const { return base[(jp + 6 * r + c) * st]; }
    __device__ __forceinline__ float Jx(int r, int c) const { return base[(jx + 3 * r + c) * st]; }
};

__device__ __forceinline__ EdgeRef edge_ref(const SchurArgs& a, int i) {
    if (i < a.M) return EdgeRef{a.planes + i, a.S, 2, 4, 16, a.planes[3 * a.S + i] * a.isig[i]};
    const int j = i - a.M;
    return EdgeRef{a.splanes + j, a.SS, 3, 5, 23, a.splanes[4 * a.SS + j] * a.sisig[j]};
}

template <int R>
struct RowCount {
    static constexpr int value = R;
};

// f(row count, edge) for edge i
template <typename F>
__device__ __forceinline__ void with_edge(const SchurArgs& a, int i, F f) {
    const EdgeRef E = edge_ref(a, i);
    if (i < a.M) f(RowCount<2>{}, E);
    else f(RowCount<3>{}, E);
}

template <int kCtrl>
__device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xF, 0xF, false));
}

// sum over aligned groups of 8 lanes, in every lane of the group
__device__ __forceinline__ float sum8(float v) {
    v += dpp_f<0xB1>(v);   // lane ^ 1
    v += dpp_f<0x4E>(v);   // lane ^ 2
    v += dpp_f<0x141>(v);  // the other quad of the half row
    return v;
}

// 8 lanes per point: they take its edges in turn (a wave's loads of a plane
// then cover the edges of 8 neighbouring points, a few whole lines, where one
// thread per point read the same lines once per edge of a point), and after
// the sums and the factorization its entries in turn.
__global__ __launch_bounds__(256) void k_schur_points(SchurArgs a) {
    const int xb = xcd_block((a.P + 31) / 32);
    if (xb < 0) return;
    const int p = xb * 32 + (threadIdx.x >> 3), g = threadIdx.x & 7;
    float h00 = 0.f, h01 = 0.f, h02 = 0.f, h11 = 0.f, h12 = 0.f, h22 = 0.f, b0 = 0.f, b1 = 0.f, b2 = 0.f;
    int e0 = 0, e1 = 0;
    if (p < a.P) {
        e0 = a.pe_ptr[p];
        e1 = a.pe_ptr[p + 1];
    }
    for (int t = e0 + g; t < e1; t += 8)
        with_edge(a, a.pe[t], [&](auto rows, const EdgeRef& E) {
            // all of the edge's loads before the sums
            constexpr int R = decltype(rows)::value;
            float er[R], x[R], y[R], z[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                er[r] = E.e(r);
                x[r] = E.Jx(r, 0);
                y[r] = E.Jx(r, 1);
                z[r] = E.Jx(r, 2);
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                b0 -= E.W * (x[r] * er[r]);
                b1 -= E.W * (y[r] * er[r]);
                b2 -= E.W * (z[r] * er[r]);
                h00 += E.W * (x[r] * x[r]);
                h01 += E.W * (x[r] * y[r]);
                h02 += E.W * (x[r] * z[r]);
                h11 += E.W * (y[r] * y[r]);
                h12 += E.W * (y[r] * z[r]);
                h22 += E.W * (z[r] * z[r]);
            }
        });
    h00 = sum8(h00); h01 = sum8(h01); h02 = sum8(h02);
    h11 = sum8(h11); h12 = sum8(h12); h22 = sum8(h22);
    b0 = sum8(b0); b1 = sum8(b1); b2 = sum8(b2);
    if (p >= a.P) return;
    // D = H_ll + lambda I = C C^T.  H_ll is positive semidefinite, so a pivot of
    // D is at least lambda, which holds it against cancellation.  Where it is
    // within rounding of zero all the same (lambda of 0 or next to it: a point
    // of one mono edge has an H_ll of rank 2) its direction carries nothing and
    // is left out, as in a pseudo-inverse: the rounding error over such a
    // pivot's root would reach S and b_schur of every frame that sees the point.
    // (A lambda below zero that leaves D indefinite gives NaN.)
    float c10 = 0.f, c20 = 0.f, c21 = 0.f, i00 = 0.f, i11 = 0.f, i22 = 0.f;
    if (e1 > e0) {
        auto inv_root = [&](float pivot, float diag) {
            const float v = fmaxf(pivot, a.lambda);
            return a.lambda >= 0.f && v <= __FLT_EPSILON__ * diag ? 0.f : 1.f / sqrtf(v);
        };
        const float d0 = h00 + a.lambda, d1 = h11 + a.lambda, d2 = h22 + a.lambda;
        i00 = inv_root(d0, d0);
        c10 = h01 * i00;
        c20 = h02 * i00;
        i11 = inv_root(d1 - c10 * c10, d1);
        c21 = (h12 - c20 * c10) * i11;
        i22 = inv_root(d2 - c20 * c20 - c21 * c21, d2);
    }
    const float y0 = b0 * i00, y1 = (b1 - c10 * y0) * i11, y2 = (b2 - c20 * y0 - c21 * y1) * i22;
    if (g == 0) {
        float4* o = reinterpret_cast<float4*>(a.prec + (long long)kPointRec * p);
        o[0] = make_float4(c10, c20, c21, i00);
        o[1] = make_float4(i11, i22, y0, y1);
        o[2] = make_float4(y2, b0, b1, b2);
        a.hd[3 * p] = h00;
        a.hd[3 * p + 1] = h11;
        a.hd[3 * p + 2] = h22;
    }
    const int q1 = a.pf_ptr[p + 1];
    for (int q = a.pf_ptr[p] + g; q < q1; q += 8) {
        float H[18];
#pragma unroll
        for (int k = 0; k < 18; k++) H[k] = 0.f;
        for (int t = a.pf_obs_ptr[q]; t < a.pf_obs_ptr[q + 1]; t++)
            with_edge(a, a.pf_obs[t], [&](auto rows, const EdgeRef& E) {
                constexpr int R = decltype(rows)::value;
                float B[R][6], A[R][3];
#pragma unroll
                for (int r = 0; r < R; r++) {
#pragma unroll
                    for (int k = 0; k < 6; k++) B[r][k] = E.Jp(r, k);
#pragma unroll
                    for (int k = 0; k < 3; k++) A[r][k] = E.Jx(r, k);
                }
#pragma unroll
                for (int r = 0; r < R; r++)
#pragma unroll
                    for (int i = 0; i < 6; i++)
#pragma unroll
                        for (int c = 0; c < 3; c++) H[3 * i + c] += E.W * (B[r][i] * A[r][c]);
            });
        float zy[6];
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const float z0 = H[3 * i] * i00;
            const float z1 = (H[3 * i + 1] - z0 * c10) * i11;
            const float z2 = (H[3 * i + 2] - z0 * c20 - z1 * c21) * i22;
            H[3 * i] = z0;
            H[3 * i + 1] = z1;
            H[3 * i + 2] = z2;
            zy[i] = z0 * y0 + z1 * y1 + z2 * y2;
        }
        float4* o = reinterpret_cast<float4*>(a.Z + (long long)kZRow * a.pf_row[q]);
        o[0] = make_float4(H[0], H[1], H[2], H[3]);
        o[1] = make_float4(H[4], H[5], H[6], H[7]);
        o[2] = make_float4(H[8], H[9], H[10], H[11]);
        o[3] = make_float4(H[12], H[13], H[14], H[15]);
        o[4] = make_float4(H[16], H[17], zy[0], zy[1]);
        o[5] = make_float4(zy[2], zy[3], zy[4], zy[5]);
    }
}

// Frame sums of one chunk of edges: the chunk's planes are read in edge order
// into LDS (per edge W, then per row J_pose and e: an odd number of words, so
// that different edges start in different banks), then a thread takes one of
// a frame's 27 sums and walks the frame's edges of the chunk.  With few
// frames, esub threads share a sum.  (A frame's edges gathered straight from
// the planes put every 4-byte read in a line of its own.)  A workgroup takes
// egroup chunks in turn and adds their sums in its row of epart: one, unless a
// row per chunk would take more than kEpartBytes (kMany; with the loop for every
// problem 47.0 us instead of 45.5, 50 frames and 1.5M edges).
template <bool kMany>
__global__ __launch_bounds__(512) void k_schur_edges(SchurArgs a) {
    constexpr int kWords = 23;  // 1 + 7 * 3 rows, and one to make it odd
    __shared__ float s_e[kEdgeChunk * kWords];
    __shared__ uint16_t s_list[kEdgeChunk];
    const int cols = kFrameSums * a.Fp;
    const int c0 = kMany ? (int)blockIdx.x * a.egroup : (int)blockIdx.x;
    const int c1 = kMany ? min(a.nechunk, c0 + a.egroup) : c0 + 1;
    for (int chunk = c0; chunk < c1; chunk++) {
        const bool st = chunk >= a.nchunk_m;
        const int rows = st ? 3 : 2, words = st ? kWords : 15;
        const int e0 = (st ? chunk - a.nchunk_m : chunk) * kEdgeChunk, n = min(kEdgeChunk, (st ? a.Ms : a.M) - e0);
        const uint16_t* ptr = a.eptr + (long long)chunk * (a.Fp + 1);
        const int nl = ptr[a.Fp];
        if (kMany && chunk > c0) __syncthreads();  // the previous chunk's LDS is read
        for (int i = threadIdx.x; i < nl; i += 512) s_list[i] = a.elist[(long long)chunk * kEdgeChunk + i];
        for (int i = threadIdx.x; i < n; i += 512) {
            const EdgeRef E = edge_ref(a, st ? a.M + e0 + i : e0 + i);
            float* o = s_e + i * words;
            o[0] = E.W;
            for (int r = 0; r < rows; r++) {
#pragma unroll
                for (int k = 0; k < 6; k++) o[1 + 7 * r + k] = E.Jp(r, k);
                o[7 + 7 * r] = E.e(r);
            }
        }
        __syncthreads();
        for (int t = threadIdx.x; t < cols * a.esub; t += 512) {
            const int sub = t / cols, col = t - sub * cols, f = col / kFrameSums;
            // sum k of a frame is element (i, c) of the rows (i, i .. 6), i = 0..5
            int i = 0, c = col - kFrameSums * f;
            while (c >= 7 - i) {
                c -= 7 - i;
                i++;
            }
            c += i;
            float acc = 0.f;
            const int l1 = ptr[f + 1];
            for (int l = ptr[f] + sub; l < l1; l += a.esub) {
                const float* e = s_e + (int)s_list[l] * words;
                const float W = e[0];
                acc += W * (e[1 + i] * e[1 + c]);
                acc += W * (e[8 + i] * e[8 + c]);
                if (rows == 3) acc += W * (e[15 + i] * e[15 + c]);
            }
            if (c == 6) acc = -acc;
            float* sum = a.epart + ((long long)blockIdx.x * a.esub + sub) * cols + col;
            *sum = !kMany || chunk == c0 ? acc : *sum + acc;
        }
    }
}

// H_pp and b_p from the chunks' sums: 16 sums per workgroup, 64 threads to a
// sum, chunk order fixed
__global__ __launch_bounds__(1024) void k_schur_edge_sums(SchurArgs a) {
    __shared__ float red[64][17];
    const int cols = kFrameSums * a.Fp, rows = a.nerow * a.esub;
    const int cl = threadIdx.x & 15, sl = threadIdx.x >> 4;
    const int col = blockIdx.x * 16 + cl;
    float acc = 0.f;
    if (col < cols) {
        int r = sl;
        for (; r + 192 < rows; r += 256) {
            const float v0 = a.epart[(long long)r * cols + col], v1 = a.epart[(long long)(r + 64) * cols + col],
                        v2 = a.epart[(long long)(r + 128) * cols + col], v3 = a.epart[(long long)(r + 192) * cols + col];
            acc += v0;
            acc += v1;
            acc += v2;
            acc += v3;
        }
        for (; r < rows; r += 64) acc += a.epart[(long long)r * cols + col];
    }
    red[sl][cl] = acc;
    __syncthreads();
    for (int s = 32; s > 0; s >>= 1) {
        if (sl < s) red[sl][cl] += red[sl + s][cl];
        __syncthreads();
    }
    if (sl != 0 || col >= cols) return;
    const int f = col / kFrameSums;
    int i = 0, c = col - kFrameSums * f;
    while (c >= 7 - i) {
        c -= 7 - i;
        i++;
    }
    c += i;
    if (c == 6) {
        a.bp[6 * f + i] = red[0][cl];
    } else {
        a.Hpp[36 * f + 6 * i + c] = red[0][cl];
        a.Hpp[36 * f + 6 * c + i] = red[0][cl];
    }
}

// halves the sums a lane keeps: [0, N) or, with hi, [N, 2N), with the DPP
// partner's share of them added
template <int kCtrl, int N>
__device__ __forceinline__ void sum_fold(float* v, int hi) {
#pragma unroll
    for (int k = 0; k < N; k++) {
        const float send = hi ? v[k] : v[k + N], keep = hi ? v[k + N] : v[k];
        v[k] = keep + dpp_f<kCtrl>(send);
    }
}

// rows (one per lane, 16-byte pieces [0, Q) of each) into the wave's LDS, at
// 16 Q bytes a row: consecutive lanes fetch consecutive pieces, so that a row
// is fetched by one instruction
typedef float mcv_f4 __attribute__((ext_vector_type(4)));

template <int Q>
__device__ __forceinline__ void rows_load(const mcv_f4* Z, int row, mcv_f4 (&v)[Q]) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < Q; k++) {
        const int e = 64 * k + lane, r = e / Q;
        v[k] = Z[(long long)__shfl(row, r, 64) * (kZRow / 4) + (e - Q * r)];
    }
}

template <bool kDiag>
__device__ __forceinline__ void schur_items(const SchurArgs& a, const ItemChunk& C, mcv_f4* lds) {
    constexpr int Q = kDiag ? 6 : 5;  // the diagonal also takes Z y
    const int lane = threadIdx.x & 63;
    const mcv_f4* Z = reinterpret_cast<const mcv_f4*>(a.Z);
    // S_ij row-major, or on the diagonal its upper triangle by rows and Z y;
    // padded to 8 n for the folds
    constexpr int kN = kDiag ? 4 : 5;
    float acc[8 * kN];
#pragma unroll
    for (int k = 0; k < 8 * kN; k++) acc[k] = 0.f;
    int2 it = a.items[min(C.i0 + lane, C.i1 - 1)];
    for (int t = C.i0; t < C.i1; t += 64) {
        mcv_f4 vi[Q], vj[Q];
        rows_load<Q>(Z, it.x, vi);
        if constexpr (!kDiag) rows_load<Q>(Z, it.y, vj);
        it = a.items[min(t + 64 + lane, C.i1 - 1)];
        wave_lds_sync();  // the previous rows are read
#pragma unroll
        for (int k = 0; k < Q; k++) {
            lds[64 * k + lane] = vi[k];
            if constexpr (!kDiag) lds[64 * (Q + k) + lane] = vj[k];
        }
        wave_lds_sync();
        // a lane past the end holds the last row again, with weight zero
        const float on = t + lane < C.i1 ? 1.f : 0.f;
        const float2* li = reinterpret_cast<const float2*>(lds + Q * lane);
        const float2* lj = reinterpret_cast<const float2*>(lds + 64 * Q + Q * lane);
        float A[18], B[18];
#pragma unroll
        for (int k = 0; k < 18; k += 2) {
            const float2 v = li[k >> 1];
            A[k] = v.x * on;
            A[k + 1] = v.y * on;
            if constexpr (!kDiag) {
                const float2 w = lj[k >> 1];
                B[k] = w.x;
                B[k + 1] = w.y;
            }
        }
        if constexpr (kDiag) {
#pragma unroll
            for (int k = 0; k < 6; k += 2) {
                const float2 v = li[9 + (k >> 1)];
                acc[21 + k] += v.x * on;
                acc[22 + k] += v.y * on;
            }
        }
        int o = 0;
#pragma unroll
        for (int r = 0; r < 6; r++)
#pragma unroll
            for (int c = kDiag ? r : 0; c < 6; c++, o++) {
                const float* b = kDiag ? A + 3 * c : B + 3 * c;
                acc[o] = fmaf(A[3 * r], b[0], fmaf(A[3 * r + 1], b[1], fmaf(A[3 * r + 2], b[2], acc[o])));
            }
    }
    // the 64 lanes' sums: each fold halves the sums a lane keeps, by lane bits
    // 3, 2 and 1 (a third of the instructions of one butterfly per sum), and
    // lanes 0, 2, .. 14 end with kN sums each
    sum_fold<0x140, 4 * kN>(acc, lane & 8);
    sum_fold<0x141, 2 * kN>(acc, lane & 4);
    sum_fold<0x1B, kN>(acc, lane & 2);
#pragma unroll
    for (int k = 0; k < kN; k++) {
        float v = acc[k];
        v += dpp_f<0xB1>(v);
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        acc[k] = v;
    }
    if (lane < 16 && (lane & 1) == 0) {
        float* o = a.ipart + (long long)kItemSums * C.out + (lane & 8 ? 4 * kN : 0) + (lane & 4 ? 2 * kN : 0) +
                   (lane & 2 ? kN : 0);
#pragma unroll
        for (int k = 0; k < kN; k++) o[k] = acc[k];
    }
}

// sum of Z_i Z_j^T (and, on the diagonal, Z y) over one chunk of a block's
// items, one wave per chunk and one item per lane.  Bound by the entry rows
// from memory (1.1 GB asked for by 5.4M items, 0.11 GB of rows).  The chunks
// run in the order of their first point, neighbours on one XCD, so that all
// blocks read the same points' rows while its L2 holds them: 142 us, against
// 290 us in block order and 806 us with one workgroup per block.
__global__ __launch_bounds__(256) void k_schur_items(SchurArgs a) {
    __shared__ mcv_f4 s_rows[4][640];
    const int xb = xcd_block((a.nichunk + 3) / 4);
    if (xb < 0) return;
    const int chunk = xb * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (chunk >= a.nichunk) return;
    const ItemChunk C = a.ichunk[chunk];
    mcv_f4* lds = s_rows[__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)];
    if (C.diag) schur_items<true>(a, C, lds);
    else schur_items<false>(a, C, lds);
}

// S and b_schur from the chunks' sums, one workgroup per block: 8 threads to
// a sum, chunk order fixed
__global__ __launch_bounds__(8 * kItemSums) void k_schur_assemble(SchurArgs a) {
    __shared__ float red[8][kItemSums];
    const int2 ij = make_int2((int)blockIdx.y, (int)blockIdx.x);
    if (ij.y < ij.x) return;
    const int blk = block_of(ij.x, ij.y, a.Fp), t = threadIdx.x % kItemSums, sl = threadIdx.x / kItemSums;
    const bool diag = ij.x == ij.y;
    float sum = 0.f;
    if (t < (diag ? 27 : 36))
        for (int c = a.blk_chunk[blk] + sl; c < a.blk_chunk[blk + 1]; c += 8) sum += a.ipart[(long long)kItemSums * c + t];
    red[sl][t] = sum;
    __syncthreads();
    if (sl == 0) {
#pragma unroll
        for (int k = 1; k < 8; k++) sum += red[k][t];
        red[0][t] = sum;
    }
    __syncthreads();
    if (threadIdx.x < 36) {
        const int r = threadIdx.x / 6, c = threadIdx.x % 6, lo = min(r, c), hi = max(r, c);
        const int n = 6 * a.Fp;
        float v = -red[0][diag ? lo * 6 - lo * (lo - 1) / 2 + hi - lo : (int)threadIdx.x];
        if (diag) v += a.Hpp[36 * ij.x + threadIdx.x] + (r == c ? a.lambda : 0.f);
        a.Sout[(long long)(6 * ij.x + r) * n + 6 * ij.y + c] = v;
        if (!diag) a.Sout[(long long)(6 * ij.y + c) * n + 6 * ij.x + r] = v;
    } else if (diag && threadIdx.x < 42) {
        const int r = threadIdx.x - 36;
        a.bs[6 * ij.x + r] = a.bp[6 * ij.x + r] - red[0][21 + r];
    }
}

// fixed-order sum of one double per thread over the workgroup (256)
__device__ __forceinline__ double block_sum_d(double v, double* red) {
    red[threadIdx.x] = v;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    return red[0];
}

// x_l = C^-T (y - sum over the point's entries of Z^T x_p) per point (0 for
// points without edges), 8 lanes per point, and per workgroup the partial sum
// of x_l . (lambda x_l + b_l) (the points' share of the LM scale).
__global__ __launch_bounds__(256) void k_schur_backsub(SchurArgs a, const float* xp, float* xl, double* partial) {
    __shared__ double red[256];
    const int p = blockIdx.x * 32 + (threadIdx.x >> 3), g = threadIdx.x & 7;
    double sc = 0.0;
    float s0 = 0.f, s1 = 0.f, s2 = 0.f;
    if (p < a.P) {
        const int q1 = a.pf_ptr[p + 1];
        for (int q = a.pf_ptr[p] + g; q < q1; q += 8) {
            const float4* z = reinterpret_cast<const float4*>(a.Z + (long long)kZRow * a.pf_row[q]);
            const float* x = xp + 6 * a.pf_frame[q];
            float A[20];
#pragma unroll
            for (int k = 0; k < 5; k++) {
                const float4 v = z[k];
                A[4 * k] = v.x; A[4 * k + 1] = v.y; A[4 * k + 2] = v.z; A[4 * k + 3] = v.w;
            }
#pragma unroll
            for (int k = 0; k < 6; k++) {
                s0 += A[3 * k] * x[k];
                s1 += A[3 * k + 1] * x[k];
                s2 += A[3 * k + 2] * x[k];
            }
        }
    }
    s0 = sum8(s0);
    s1 = sum8(s1);
    s2 = sum8(s2);
    if (p < a.P && g == 0) {
        const float4* rec = reinterpret_cast<const float4*>(a.prec + (long long)kPointRec * p);
        const float4 r0 = rec[0], r1 = rec[1], r2 = rec[2];
        const float c10 = r0.x, c20 = r0.y, c21 = r0.z, i00 = r0.w, i11 = r1.x, i22 = r1.y;
        const float x2 = (r2.x - s2) * i22, x1 = (r1.w - s1 - c21 * x2) * i11,
                    x0 = (r1.z - s0 - c10 * x1 - c20 * x2) * i00;
        const float v[3] = {x0, x1, x2}, b[3] = {r2.y, r2.z, r2.w};
#pragma unroll
        for (int k = 0; k < 3; k++) {
            xl[3 * p + k] = v[k];
            sc += (double)v[k] * ((double)a.lambda * (double)v[k] + (double)b[k]);
        }
    }
    const double t = block_sum_d(sc, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// Huber rho of chi2 (core/robust_kernel_impl.cpp:65-78) summed over the
// active edges, per workgroup: mono edge i takes delta from its (frame,
// camera) pair, stereo edges the stereo delta; an infinite delta is the
// edge without a robust kernel (rho = chi2).
__device__ __forceinline__ double huber_rho(float chi2, float delta) {
    const double e = chi2, d = delta;
    return e <= d * d ? e : 2.0 * sqrt(e) * d - d * d;
}

__global__ __launch_bounds__(256) void k_ba_rho_sum(const float* chi2, const uint32_t* pair, const BAPair* pairs,
                                                    const uint8_t* act, int M, const float* schi2,
                                                    const uint8_t* sact, int Ms, float sdelta, double* partial) {
    __shared__ double red[256];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (i < M) {
        if (!act || act[i]) v = huber_rho(chi2[i], pairs[pair[i]].delta);
    } else if (i - M < Ms) {
        const int j = i - M;
        if (!sact || sact[j]) v = huber_rho(schi2[j], sdelta);
    }
    const double t = block_sum_d(v, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// ---- a keyframe's pose, on the host and on the device --------------------------
// double -> (hi, lo) float pair
__host__ __device__ inline void split(double v, float& hi, float& lo) {
    hi = (float)v;
    lo = (float)(v - (double)hi);
}

__host__ __device__ inline void quat_to_R(const double* q, double R[9]) {
    const double x = q[0], y = q[1], z = q[2], w = q[3];
    const double tx = 2 * x, ty = 2 * y, tz = 2 * z;
    const double twx = tx * w, twy = ty * w, twz = tz * w;
    const double txx = tx * x, txy = ty * x, txz = tz * x;
    const double tyy = ty * y, tyz = tz * y, tzz = tz * z;
    R[0] = 1 - (tyy + tzz); R[1] = txy - twz; R[2] = txz + twy;
    R[3] = txy + twz; R[4] = 1 - (txx + tzz); R[5] = tyz - twx;
    R[6] = txz - twy; R[7] = tyz + twx; R[8] = 1 - (txx + tyy);
}

// One frame's records from its FP64 state: the pose for the stereo edges, and
// per camera (cm: fx fy cx cy, quaternion, translation, Huber delta) that of the
// mono edges.  Without the robust kernel the Huber deltas are infinite (w = 1,
// rho = chi2).
__host__ __device__ inline void frame_rotation(const double* fq, double Rbw[9]) {
    // g2o SE3Quat keeps a normalised quaternion with w >= 0 (se3quat.h:280-285)
    const double qn = sqrt(fq[0] * fq[0] + fq[1] * fq[1] + fq[2] * fq[2] + fq[3] * fq[3]);
    const double q[4] = {fq[0] / qn, fq[1] / qn, fq[2] / qn, fq[3] / qn};
    quat_to_R(q, Rbw);
}

__host__ __device__ inline void pose_record(const double Rbw[9], const double* tbw, FramePose& fp) {
    for (int i = 0; i < 9; i++) split(Rbw[i], fp.Rh[i], fp.Rl[i]);
    for (int i = 0; i < 3; i++) split(tbw[i], fp.th[i], fp.tl[i]);
}

__host__ __device__ inline void pair_record(const double Rbw[9], const double* tbw, const double* cm, bool robust,
                                            BAPair& P) {
    double Rcb[9];
    const double qn = sqrt(cm[4] * cm[4] + cm[5] * cm[5] + cm[6] * cm[6] + cm[7] * cm[7]);
    const double qc[4] = {cm[4] / qn, cm[5] / qn, cm[6] / qn, cm[7] / qn};
    quat_to_R(qc, Rcb);
    const double* tcb = cm + 8;
    // Tcw = Tcb * Tbw
    for (int r = 0; r < 3; r++) {
        for (int cc = 0; cc < 3; cc++) {
            double v = 0;
            for (int m = 0; m < 3; m++) v += Rcb[3 * r + m] * Rbw[3 * m + cc];
            split(v, P.Rh[3 * r + cc], P.Rl[3 * r + cc]);
        }
        double tv = tcb[r];
        for (int m = 0; m < 3; m++) tv += Rcb[3 * r + m] * tbw[m];
        split(tv, P.th[r], P.tl[r]);
    }
    for (int i = 0; i < 9; i++) { P.Rbw[i] = (float)Rbw[i]; P.Rcb[i] = (float)Rcb[i]; }
    for (int i = 0; i < 3; i++) P.tbw[i] = (float)tbw[i];
    P.fx = (float)cm[0]; P.fy = (float)cm[1]; P.cx = (float)cm[2]; P.cy = (float)cm[3];
    P.delta = robust ? (float)cm[11] : INFINITY;
    P.pad[0] = P.pad[1] = P.pad[2] = 0.f;
}

// Pose increment T <- exp(x) * T of VertexSE3Expmap::oplusImpl
// (types/sba/types_six_dof_expmap.h:98-101): SE3Quat::exp
// (types/slam3d/se3quat.h:218-257) with Eigen's matrix -> quaternion
// conversion, then the product with a normalised (w >= 0) quaternion.
struct Qd { double x, y, z, w; };

__host__ __device__ inline Qd qd_mul(const Qd& a, const Qd& b) {
    return Qd{a.w * b.x + a.x * b.w + a.y * b.z - a.z * b.y, a.w * b.y + a.y * b.w + a.z * b.x - a.x * b.z,
              a.w * b.z + a.z * b.w + a.x * b.y - a.y * b.x, a.w * b.w - a.x * b.x - a.y * b.y - a.z * b.z};
}

__host__ __device__ inline void qd_rotate(const Qd& q, const double v[3], double o[3]) {
    double uv[3] = {q.y * v[2] - q.z * v[1], q.z * v[0] - q.x * v[2], q.x * v[1] - q.y * v[0]};
    for (double& c : uv) c += c;
    o[0] = v[0] + q.w * uv[0] + (q.y * uv[2] - q.z * uv[1]);
    o[1] = v[1] + q.w * uv[1] + (q.z * uv[0] - q.x * uv[2]);
    o[2] = v[2] + q.w * uv[2] + (q.x * uv[1] - q.y * uv[0]);
}

__host__ __device__ inline void qd_normalize(Qd& q) {
    if (q.w < 0) q = Qd{-q.x, -q.y, -q.z, -q.w};
    const double n = sqrt(q.x * q.x + q.y * q.y + q.z * q.z + q.w * q.w);
    q = Qd{q.x / n, q.y / n, q.z / n, q.w / n};
}

// the case of the largest diagonal entry I (indices known when compiled: the
// device keeps no array in memory)
template <int I>
__host__ __device__ inline Qd qd_from_diagonal(const double* m) {
    constexpr int J = (I + 1) % 3, K = (J + 1) % 3;
    double c[3];
    double t = sqrt(m[4 * I] - m[4 * J] - m[4 * K] + 1.0);
    c[I] = 0.5 * t;
    t = 0.5 / t;
    c[J] = (m[3 * J + I] + m[3 * I + J]) * t;
    c[K] = (m[3 * K + I] + m[3 * I + K]) * t;
    return Qd{c[0], c[1], c[2], (m[3 * K + J] - m[3 * J + K]) * t};
}

__host__ __device__ inline Qd qd_from_R(const double* m) {
    Qd q{};
    double t = m[0] + m[4] + m[8];
    if (t > 0) {
        t = sqrt(t + 1.0);
        q.w = 0.5 * t;
        t = 0.5 / t;
        q.x = (m[7] - m[5]) * t;
        q.y = (m[2] - m[6]) * t;
        q.z = (m[3] - m[1]) * t;
    } else {
        const bool y = m[4] > m[0];
        if (m[8] > (y ? m[4] : m[0])) q = qd_from_diagonal<2>(m);
        else q = y ? qd_from_diagonal<1>(m) : qd_from_diagonal<0>(m);
    }
    return q;
}

__host__ __device__ inline void se3_oplus(double* frame, const double* xi) {
    const double w[3] = {xi[0], xi[1], xi[2]};
    const double th = sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
    const double W[9] = {0, -w[2], w[1], w[2], 0, -w[0], -w[1], w[0], 0};
    double W2[9];
    for (int r = 0; r < 3; r++)
        for (int c = 0; c < 3; c++) W2[3 * r + c] = W[3 * r] * W[c] + W[3 * r + 1] * W[3 + c] + W[3 * r + 2] * W[6 + c];
    double R[9], V[9];
    for (int k = 0; k < 9; k++) {
        const double I = (k % 4 == 0) ? 1.0 : 0.0;
        if (th < 0.00001) {
            R[k] = I + W[k] + 0.5 * W2[k];
            V[k] = I + 0.5 * W[k] + (1.0 / 6.0) * W2[k];
        } else {
            R[k] = I + sin(th) / th * W[k] + (1 - cos(th)) / (th * th) * W2[k];
            V[k] = I + (1 - cos(th)) / (th * th) * W[k] + (th - sin(th)) / (th * th * th) * W2[k];
        }
    }
    Qd dq = qd_from_R(R);
    qd_normalize(dq);
    double dt[3];
    for (int r = 0; r < 3; r++) dt[r] = V[3 * r] * xi[3] + V[3 * r + 1] * xi[4] + V[3 * r + 2] * xi[5];
    // exp(x) * T
    const Qd q{frame[0], frame[1], frame[2], frame[3]};
    double rt[3];
    qd_rotate(dq, frame + 4, rt);
    Qd nq = qd_mul(dq, q);
    qd_normalize(nq);
    frame[0] = nq.x; frame[1] = nq.y; frame[2] = nq.z; frame[3] = nq.w;
    for (int r = 0; r < 3; r++) frame[4 + r] = dt[r] + rt[r];
}

// The optimizer on a problem whose only unknown is one keyframe's pose (every
// point and every other frame fixed), in one launch of one workgroup: the
// iterations, trials and rules of mcv_ba_optimize.  An evaluation of a state
// gives chi2 (sum of rho), H_pp and b_p at once, FP64 sums of the edges' FP32
// terms in a fixed order, so a trial that is accepted has already linearized
// the next iteration, and one that is rejected leaves the last H_pp and b_p in
// hand.  Wave 0 solves the 6 x 6 system, moves the frame and writes its records;
// all waves evaluate.  A frame has at most a few thousand edges, so a trial is
// bound by its chain, not by the edges' arithmetic: with the optimizer on the
// host and a launch and a wait per trial it took 26 us.
constexpr int kPoseThreads = 512;
constexpr int kPoseCams = 8;       // cameras whose records fit the workgroup's state
constexpr int kPoseMaxEdges = 16384;
constexpr int kPoseSums = 28;      // H_pp's upper triangle by rows, each row followed by b_p's entry; chi2
constexpr int kPoseIters = 16;     // iterations of one launch

struct PoseState {
    BAPair pair[kPoseCams];  // (frame, camera) records of the free frame
    FramePose pose;
};

struct PoseArgs {
    BAObs ob;
    BAStereoObs so;
    const float4 *hi, *lo;
    const BAPair* pairs;     // the other frames'
    const FramePose* poses;
    const uint8_t *act_m, *act_s;  // or null
    StereoCam scam;
    int frame, C;            // the free frame
};

struct PoseRun {             // in: where the optimizer stands; out: where it stopped
    double fr[7], lambda, ni;
    int iters;               // in: to run (at most kPoseIters); out: run
    int stop;                // in: nonzero on a problem's first launch; out: no further iteration
};

struct PoseSetup {
    double cams[12 * kPoseCams];
    double tau;
    int max_trials, robust;
};

template <int kCtrl, int N>
__device__ __forceinline__ void sum_fold_d(double* v, int hi) {
#pragma unroll
    for (int k = 0; k < N; k++) {
        const double send = hi ? v[k] : v[k + N], keep = hi ? v[k + N] : v[k];
        const int lo32 = __builtin_amdgcn_update_dpp(0, __double2loint(send), kCtrl, 0xF, 0xF, false);
        const int hi32 = __builtin_amdgcn_update_dpp(0, __double2hiint(send), kCtrl, 0xF, 0xF, false);
        v[k] = keep + __hiloint2double(hi32, lo32);
    }
}

// acc += W times the outer products of kRows rows of J with themselves (upper
// triangle by rows) and, negated, with e, in FP64
template <int kRows>
__device__ __forceinline__ void pose_terms(double (&acc)[32], const float* J, const float* e, float W) {
#pragma unroll
    for (int row = 0; row < kRows; row++) {
        double j[6], w[6];
#pragma unroll
        for (int r = 0; r < 6; r++) {
            j[r] = (double)J[6 * row + r];
            w[r] = (double)W * j[r];
        }
        const double m = -(double)e[row];
        int o = 0;
#pragma unroll
        for (int r = 0; r < 6; r++) {
#pragma unroll
            for (int k = r; k < 6; k++, o++) acc[o] = __builtin_fma(w[r], j[k], acc[o]);
            acc[o] = __builtin_fma(w[r], m, acc[o]);
            o++;
        }
    }
}

// The sums of state S into sums (LDS).  The mono edges go to the threads in
// order, kPoseBatch of them loaded at once, the stereo edges from the last
// thread down, whose waves have fewer.
constexpr int kPoseBatch = 3;
__device__ __forceinline__ void pose_eval(const PoseArgs& a, const PoseState& S, double (*s_sum)[32], double* sums) {
    double acc[32];
#pragma unroll
    for (int k = 0; k < 32; k++) acc[k] = 0.0;
    for (int i0 = threadIdx.x; i0 < a.ob.M; i0 += kPoseBatch * kPoseThreads) {
        BAIn in[kPoseBatch];
        bool on[kPoseBatch];
#pragma unroll
        for (int u = 0; u < kPoseBatch; u++) {
            const int i = i0 + u * kPoseThreads;
            on[u] = i < a.ob.M && !(a.act_m && !a.act_m[i]);
            ba_load_obs(min(i, a.ob.M - 1), a.ob, in[u]);
        }
#pragma unroll
        for (int u = 0; u < kPoseBatch; u++) ba_load_point(a.hi, a.lo, in[u]);
#pragma unroll
        for (int u = 0; u < kPoseBatch; u++) {
            if (!on[u]) continue;
            const int f = (int)in[u].pair / a.C, c = (int)in[u].pair - f * a.C;
            const BAPair& T = f == a.frame ? S.pair[c] : a.pairs[in[u].pair];
            const BAEdge E = ba_residual(in[u], T);
            acc[27] += huber_rho(E.chi2, T.delta);
            if (f != a.frame) continue;
            float J[12];
            ba_jpose(in[u], E, T, J);
            const float e[2] = {E.e0, E.e1};
            pose_terms<2>(acc, J, e, E.w * in[u].isig);
        }
    }
    for (int i = kPoseThreads - 1 - threadIdx.x; i < a.so.M; i += kPoseThreads) {
        if (a.act_s && !a.act_s[i]) continue;
        const int f = (int)a.so.fr[i];
        const FramePose& T = f == a.frame ? S.pose : a.poses[f];
        const StereoEdge E = stereo_residual(a.so, i, a.hi, a.lo, T, a.scam);
        acc[27] += huber_rho(E.chi2, a.scam.delta);
        if (f != a.frame) continue;
        float J[18];
        stereo_jpose(E, a.scam, J);
        pose_terms<3>(acc, J, E.e, E.w * a.so.isig[i]);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    sum_fold_d<0x140, 16>(acc, lane & 8);
    sum_fold_d<0x141, 8>(acc, lane & 4);
    sum_fold_d<0x1B, 4>(acc, lane & 2);
    sum_fold_d<0xB1, 2>(acc, lane & 1);
#pragma unroll
    for (int k = 0; k < 2; k++) {
        acc[k] += __shfl_xor(acc[k], 16, 64);
        acc[k] += __shfl_xor(acc[k], 32, 64);
    }
    if (lane < 16) {
        const int o = (lane & 8 ? 16 : 0) + (lane & 4 ? 8 : 0) + (lane & 2 ? 4 : 0) + (lane & 1 ? 2 : 0);
        s_sum[wave][o] = acc[0];
        s_sum[wave][o + 1] = acc[1];
    }
    __syncthreads();
    if (threadIdx.x < kPoseSums) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < kPoseThreads / 64; w++) v += s_sum[w][threadIdx.x];
        sums[threadIdx.x] = v;
    }
}

// x = S^-1 b by Cholesky (mcv_solve_llt for n = 6, with the diagonal's
// reciprocals: a chain of 33 divisions otherwise), S = H_pp + lambda I from the
// sums of an evaluation; false when S is not positive definite
__device__ __forceinline__ bool pose_solve(const double* sums, double lambda, double (&b)[6], double (&x)[6]) {
    double L[6][6], inv[6];
    int o = 0;
#pragma unroll
    for (int r = 0; r < 6; r++) {
#pragma unroll
        for (int k = r; k < 6; k++) L[k][r] = sums[o++];
        L[r][r] += lambda;
        b[r] = sums[o++];
    }
#pragma unroll
    for (int j = 0; j < 6; j++) {
        double d = L[j][j];
#pragma unroll
        for (int k = 0; k < j; k++) d -= L[j][k] * L[j][k];
        if (!(d > 0)) return false;
        inv[j] = 1.0 / sqrt(d);
#pragma unroll
        for (int i = j + 1; i < 6; i++) {
            double v = L[i][j];
#pragma unroll
            for (int k = 0; k < j; k++) v -= L[i][k] * L[j][k];
            L[i][j] = v * inv[j];
        }
    }
    double y[6];
#pragma unroll
    for (int i = 0; i < 6; i++) {
        double v = b[i];
#pragma unroll
        for (int k = 0; k < i; k++) v -= L[i][k] * y[k];
        y[i] = v * inv[i];
    }
#pragma unroll
    for (int i = 5; i >= 0; i--) {
        double v = y[i];
#pragma unroll
        for (int k = i + 1; k < 6; k++) v -= L[k][i] * x[k];
        x[i] = v * inv[i];
    }
    return true;
}

// the optimizer's state, in LDS between its steps (the evaluations need the
// registers)
struct PoseStep {
    double fr[7], fr0[7], lambda, ni, rho, scale;
    int it, qmax;
    bool begin, pending, done, stop;
};

__global__ __launch_bounds__(kPoseThreads) void k_pose_optimize(PoseArgs a, PoseSetup q, PoseRun in, PoseRun* out,
                                                                double* stats) {
    __shared__ PoseState s_state;
    __shared__ double s_sum[kPoseThreads / 64][32];
    __shared__ double s_new[kPoseSums], s_cur[kPoseSums];
    __shared__ PoseStep s_step;
    const int lane = threadIdx.x & 63;
    const bool ctl = threadIdx.x < 64;  // wave 0: the optimizer, every lane alike
    // the frame's records: camera `lane`, or the pose
    auto records = [&](const double* fr) {
        double Rbw[9];
        frame_rotation(fr, Rbw);
        if (lane < a.C) pair_record(Rbw, fr + 4, q.cams + 12 * lane, q.robust != 0, s_state.pair[lane]);
        else if (lane == kPoseCams) pose_record(Rbw, fr + 4, s_state.pose);
    };
    if (ctl) {
        records(in.fr);
        PoseStep T{};
#pragma unroll
        for (int k = 0; k < 7; k++) T.fr[k] = in.fr[k];
        T.lambda = in.lambda;
        T.ni = in.ni;
        T.begin = true;
        if (lane == 0) s_step = T;
    }
    __syncthreads();
    pose_eval(a, s_state, s_sum, s_cur);
    for (;;) {
        __syncthreads();
        if (ctl) {
            PoseStep T = s_step;
            // the trial's verdict; at an iteration's end, whether to go on
            auto judge = [&](double chi) {
                T.rho = (s_cur[27] - chi) / T.scale;
                bool last = false;
                if (T.rho > 0 && isfinite(chi)) {
                    const double g = 2 * T.rho - 1;
                    T.lambda *= fmax(1. / 3., fmin(1. - g * g * g, 2. / 3.));
                    T.ni = 2;
                    wave_lds_sync();
                    if (lane < kPoseSums) s_cur[lane] = s_new[lane];
                    wave_lds_sync();
                } else {
                    T.lambda *= T.ni;
                    T.ni *= 2;
#pragma unroll
                    for (int k = 0; k < 7; k++) T.fr[k] = T.fr0[k];
                    last = !isfinite(T.lambda);
                }
                if (!last) {
                    T.qmax++;
                    if (T.rho < 0 && T.qmax < q.max_trials) return;
                }
                if (lane == 0) {
                    stats[4 * T.it + 1] = s_cur[27];
                    stats[4 * T.it + 2] = T.lambda;
                    stats[4 * T.it + 3] = T.qmax;
                }
                T.it++;
                T.stop = T.qmax == q.max_trials || T.rho == 0 || !isfinite(T.lambda);
                T.done = T.stop || T.it == in.iters;
                T.begin = true;
            };
            if (T.pending) judge(s_new[27]);
            T.pending = false;
            while (!T.done) {
                if (T.begin) {
                    T.begin = false;
                    if (lane == 0) stats[4 * T.it] = s_cur[27];
                    if (in.stop && T.it == 0) {
                        // computeLambdaInit: the diagonal entries of H_pp
                        const double mx =
                            fmax(fmax(fmax(fabs(s_cur[0]), fabs(s_cur[7])), fmax(fabs(s_cur[13]), fabs(s_cur[18]))),
                                 fmax(fabs(s_cur[22]), fabs(s_cur[25])));
                        T.lambda = q.tau * mx;
                    }
                    T.rho = 0;
                    T.qmax = 0;
                }
#pragma unroll
                for (int k = 0; k < 7; k++) T.fr0[k] = T.fr[k];
                double b[6], x[6];
                T.scale = 1e-3;
                if (pose_solve(s_cur, T.lambda, b, x)) {
#pragma unroll
                    for (int k = 0; k < 6; k++) T.scale += x[k] * (T.lambda * x[k] + b[k]);
                    se3_oplus(T.fr, x);
                    records(T.fr);
                    T.pending = true;
                    break;
                }
                judge(DBL_MAX);
            }
            if (lane == 0) s_step = T;
        }
        __syncthreads();
        if (!s_step.pending) break;
        pose_eval(a, s_state, s_sum, s_new);
    }
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < 7; k++) out->fr[k] = s_step.fr[k];
        out->lambda = s_step.lambda;
        out->ni = s_step.ni;
        out->iters = s_step.it;
        out->stop = s_step.stop;
    }
}

// out[0] = sum of partial[0 .. n) in a fixed order (one workgroup)
__global__ __launch_bounds__(256) void k_sum_partials(const double* partial, int n, double* out) {
    __shared__ double red[256];
    double v = 0.0;
    for (int k = threadIdx.x; k < n; k += 256) v += partial[k];
    const double t = block_sum_d(v, red);
    if (threadIdx.x == 0) out[0] = t;
}

// largest |diagonal entry| of H_pp (free frames) and H_ll (points with
// edges), computeLambdaInit's maxDiagonal: per-workgroup maxima over a
// grid-stride loop into partial[blockIdx.x], then k_max_partials
__global__ __launch_bounds__(256) void k_ba_max_diag(const float* Hpp, int Fp, const float* hd, const int* pe_ptr,
                                                     int P, float* partial) {
    __shared__ float red[256];
    float m = 0.f;
    const int stride = gridDim.x * 256;
    for (int k = blockIdx.x * 256 + threadIdx.x; k < 6 * Fp; k += stride)
        m = fmaxf(m, fabsf(Hpp[36 * (k / 6) + 7 * (k % 6)]));
    for (int k = blockIdx.x * 256 + threadIdx.x; k < 3 * P; k += stride) {
        const int p = k / 3;
        if (pe_ptr[p + 1] > pe_ptr[p]) m = fmaxf(m, fabsf(hd[k]));
    }
    red[threadIdx.x] = m;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void k_max_partials(const float* partial, int n, float* out) {
    __shared__ float red[256];
    float m = 0.f;
    for (int k = threadIdx.x; k < n; k += 256) m = fmaxf(m, partial[k]);
    red[threadIdx.x] = m;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

// FP64 point estimates -> (hi, lo) float pairs; with xl, first the additive
// update P += x_l of the free points (VertexSBAPointXYZ::oplusImpl).  bak keeps
// the estimates from before it; restore: they come back from there.
template <typename T>
__global__ __launch_bounds__(256) void k_ba_points_apply(double* p64, double* bak, bool restore, const T* xl,
                                                         const uint8_t* fixed, int P, float4* hi, float4* lo) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= P) return;
    const double* src = restore ? bak : p64;
    double* dst = restore ? p64 : bak;
    double v[3] = {src[3 * p], src[3 * p + 1], src[3 * p + 2]};
    if (dst) {
#pragma unroll
        for (int k = 0; k < 3; k++) dst[3 * p + k] = v[k];
    }
    if (xl && !(fixed && fixed[p])) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            v[k] += (double)xl[3 * p + k];
            p64[3 * p + k] = v[k];
        }
    }
    float h[3], l[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        h[k] = (float)v[k];
        l[k] = (float)(v[k] - (double)h[k]);
    }
    hi[p] = make_float4(h[0], h[1], h[2], 0.f);
    lo[p] = make_float4(l[0], l[1], l[2], 0.f);
}

}  // namespace mcv

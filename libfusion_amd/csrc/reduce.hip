// ICP and photometric normal-equation reductions and the on-device
// Gauss-Newton step.
//
// Reference: src/tracking/pose_estimator.cu (ICPReduction :166-260,
// icp_reduce :267-307), src/tracking/m_estimator.cu (RgbReduction2 :313-430,
// rgb_step :437-482), include/tracking/reduce_sum.h (WarpReduce / BlockReduce
// :11-46, create_jtjjtr :48-61), src/tracking/icp_tracker.cpp
// (compute_transform :23-156).
//
// MI355X design:
//  * A tracking step evaluates both the ICP row and the RGB row of every reference
//    pixel (they share the projected vertex) and accumulates their combined normal
//    equations, 31 FP64 sums per lane; a stand-alone reduction has one kind of row
//    and 29 FP32 sums.
//  * A wavefront's sums are a transpose butterfly by DPP and permlane swaps, then the
//    8 wavefronts' partials meet in LDS; each workgroup writes one partial row.
//  * One lane per reference pixel, so a whole pyramid level is in flight at
//    once (the pass is bound by memory latency, not bandwidth); each pixel's
//    loads are issued in two rounds.
//  * A tracking iteration is one launch: every workgroup sums the previous
//    iteration's partial rows in a fixed order (deterministic), one lane builds
//    A = 1e6 H_icp + H_rgb, solves it with an FP64 LDL^T, applies T <- exp(dx) T
//    in FP64 and runs the reference's divergence / revert logic; then the
//    workgroup adds up its own partial row at the new pose.  The first launch of
//    a frame starts the estimate and a last one, of one workgroup, ends it: a
//    whole frame of tracking is a fixed sequence of launches with no host
//    round trip (the reference downloads the sums and solves on the host twice
//    per iteration).
//  * The stand-alone reductions of the C-ABI (lf_icp_reduce, lf_rgb_step) are
//    one launch, in which a workgroup that finds every row written sums them.
#include <atomic>
#include <cfloat>
#include <climits>
#include <functional>
#include <mutex>

#include "lf_common.h"
#include "lf_track.h"

using namespace lf;

namespace {

// Maximum workgroups of a reduction: the workgroups resident at once on
// MI355X (256 CUs x 2 workgroups of 512 lanes at the step kernel's register
// count).  A larger level loops over pixels with the next pixel's loads in
// flight, rather than waiting for a second round of workgroups.
constexpr int kGrid = 512;
constexpr int kStepGrid = 256;  // of a lone system's tracking step (step_grid)
constexpr int kThreads = 512;  // lanes per workgroup (8 wavefronts)
constexpr int kWaves = kThreads / 64;

struct ReduceArgs {
    LfTrackLevel lv;
    const float *pose12;   // float 3x4 (stand-alone reductions)
    float stddev;          // stand-alone RGB reduction
    float angle, dthr;
    float *partials;       // kGrid * kVals floats
    // tracking step
    LfTrackState *st;
    int step;              // index within the frame; 0: the estimate starts at init
    int first_iter;        // first iteration of a level
    int prev_first_iter;   // the previous step's first_iter,
    int prev_grid;         // and its workgroups (partial rows)
    int context_mode;      // compute_transform(ctx) semantics
    float icp_weight;
    double init[12];       // initial estimate (step 0)
    float init_f[12];      // the same in FP32 (the first step's pose, uniform across the grid)
};

// create_jtjjtr<6,7> plus {r^2, count} of one row, summed in FP32: the
// reference's sums (the stand-alone reductions lf_icp_reduce / lf_rgb_step).
LF_DEV void accumulate(float *s, const float *row) {
    int k = 0;
#pragma unroll
    for (int i = 0; i < 7; ++i)
#pragma unroll
        for (int j = i; j < 7; ++j) s[k++] += row[i] * row[j];
    s[28] += 1.0f;
}

constexpr int kVals = 29;
struct FloatSums {  // a stand-alone reduction's sums
    float s[32];    // kVals, padded to a power of two for the wavefront transpose
    LF_DEV void clear() {
#pragma unroll
        for (int k = 0; k < 32; ++k) s[k] = 0.0f;
    }
    LF_DEV void icp(const float *row) { accumulate(s, row); }
    LF_DEV void rgb(const float *row) { accumulate(s, row); }
};

// The tracking step's sums: the normal equations A = w H_icp + H_rgb,
// b = w g_icp + g_rgb of compute_transform (icp_tracker.cpp:89-96) combined
// per pixel and accumulated in FP64, plus each term's {r^2, count}.  A
// product of two FP32 row values is exact in FP64, the ICP weight costs one
// rounding at 2^-53 and every fused multiply-add one more, so a lane's serial
// sum and the tree above it stay within about 1e-13 of the exact sum of the
// FP32 rows (relative to the sum of magnitudes), where FP32 sums (the
// reference's, summed per term and combined in FP32) carry about 1e-6.
// Layout (kTrackVals): 0-26 the create_jtjjtr<6,7> order of A and b, 27 / 28
// ICP r^2 / count, 29 / 30 RGB r^2 / count.
constexpr int kTrackVals = 31;
struct CombinedSums {
    double s[32];  // kTrackVals, padded to a power of two for the wavefront transpose
    double w;      // the ICP weight
    unsigned n_icp, n_rgb;  // the counts, moved into s[28] / s[30] for the reduction
    LF_DEV void clear() {
#pragma unroll
        for (int k = 0; k < 32; ++k) s[k] = 0.0;
        n_icp = n_rgb = 0u;
    }
    LF_DEV void icp(const float *row) {
        double d[7], wd[6];
#pragma unroll
        for (int i = 0; i < 7; ++i) d[i] = (double)row[i];
#pragma unroll
        for (int i = 0; i < 6; ++i) wd[i] = w * d[i];
        int k = 0;
#pragma unroll
        for (int i = 0; i < 6; ++i)
#pragma unroll
            for (int j = i; j < 7; ++j) s[k] = __builtin_fma(wd[i], d[j], s[k]), ++k;
        s[27] = __builtin_fma(d[6], d[6], s[27]);
        ++n_icp;
    }
    LF_DEV void rgb(const float *row) {
        double d[7];
#pragma unroll
        for (int i = 0; i < 7; ++i) d[i] = (double)row[i];
        int k = 0;
#pragma unroll
        for (int i = 0; i < 6; ++i)
#pragma unroll
            for (int j = i; j < 7; ++j) s[k] = __builtin_fma(d[i], d[j], s[k]), ++k;
        s[29] = __builtin_fma(d[6], d[6], s[29]);
        ++n_rgb;
    }
};

// Both rows of one reference pixel — ICPReduction::searchPoint + getRow
// (pose_estimator.cu:168-222) and RgbReduction2::find_corresp +
// compute_jacobian with interp2 (m_estimator.cu:315-391) — with all loads in
// two rounds: the pixel's own vertex / normal / intensity first, then every
// gather (the ICP correspondence and the 12 bilinear taps of the photometric
// term) together.  The arithmetic follows the reference's operation order.
// A reference pixel's own inputs (its vertex, normal and intensity): they do
// not depend on the pose, so they are loaded before the pose is known.
struct Own {
    float4 lv, ln;
    float il;
};

// Element i of a map of float4 or of 4 x FP16 (kHalf), and of a plane of
// float or FP16: the mixed-precision maps widen to FP32 as they are loaded.
template <bool kHalf>
LF_DEV float4 map4(const float *p, size_t i) {
    if constexpr (kHalf) {
        const uint2 u = reinterpret_cast<const uint2 *>(p)[i];
        return make_float4(half_bits_to_float((unsigned short)u.x), half_bits_to_float((unsigned short)(u.x >> 16)),
                           half_bits_to_float((unsigned short)u.y), half_bits_to_float((unsigned short)(u.y >> 16)));
    } else {
        return reinterpret_cast<const float4 *>(p)[i];
    }
}
template <bool kHalf>
LF_DEV float plane1(const float *p, size_t i) {
    if constexpr (kHalf) return half_bits_to_float(reinterpret_cast<const unsigned short *>(p)[i]);
    else return p[i];
}

template <bool kIcp, bool kRgb, bool kHalf = false>
LF_DEV Own load_own(const LfTrackLevel &L, int i) {
    Own o;
    o.lv = map4<false>(L.last_vmap, i);  // vertices are FP32 in both precisions
    o.ln = make_float4(0.f, 0.f, 0.f, 0.f);
    o.il = 0.0f;
    if (kIcp) o.ln = map4<kHalf>(L.last_nmap, i);
    if (kRgb) o.il = plane1<kHalf>(L.last_I, i);
    return o;
}

// kHalf (mixed precision) also takes one hardware reciprocal of the depth for
// every projection and the hardware square root, where the FP32 path keeps
// the reference's correctly rounded divisions and roots.
LF_DEV float uniform_f(float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); }
LF_DEV float fast_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }

template <bool kIcp, bool kRgb, bool kHalf, class Sums>
LF_DEV void pixel_rows(const ReduceArgs &a, const Own &o, const float *P, float stddev, float th, Sums &sums) {
    const LfTrackLevel &L = a.lv;
    const float4 lv = o.lv, ln = o.ln;
    const float il = o.il;
    const f3 vg = xform(P, f3{lv.x, lv.y, lv.z});
    const float iz = kHalf ? __builtin_amdgcn_rcpf(vg.z) : 0.0f;
    // ICP correspondence (pose_estimator.cu:168-193)
    bool icp_ok = false;
    size_t j = 0;
    if (kIcp) {
        const float invz = kHalf ? iz : 1.0f / vg.z;
        const int u = proj_floor(vg.x * invz * L.K.fx + L.K.cx + 0.5f);
        const int v = proj_floor(vg.y * invz * L.K.fy + L.K.cy + 0.5f);
        icp_ok = !isnan(lv.x) && u >= 0 && v >= 0 && u < L.cols && v < L.rows;
        if (icp_ok) j = (size_t)v * L.cols + u;
    }
    // photometric correspondence (m_estimator.cu:315-338)
    bool rgb_ok = false;
    float u0 = 0.0f, v0 = 0.0f;
    size_t t0 = 0;
    if (kRgb) {
        u0 = (kHalf ? vg.x * iz : vg.x / vg.z) * L.K.fx + L.K.cx;
        v0 = (kHalf ? vg.y * iz : vg.y / vg.z) * L.K.fy + L.K.cy;
        rgb_ok = !(lv.w < 0.0f || isnan(lv.x)) && isfinite(il) && u0 >= 2.0f && u0 < (float)(L.cols - 2) &&
                 v0 >= 2.0f && v0 < (float)(L.rows - 2);
        if (rgb_ok) t0 = (size_t)(int)floorf(v0) * L.cols + (int)floorf(u0);
    }
    // gathers
    float4 cv = make_float4(0.f, 0.f, 0.f, 0.f), cn = cv;
    if (kIcp) {
        cv = map4<false>(L.curr_vmap, j);
        cn = map4<kHalf>(L.curr_nmap, j);
    }
    float tI[4], tx[4], ty[4];
    if (kRgb) {
        const size_t o[4] = {t0, t0 + 1, t0 + L.cols, t0 + L.cols + 1};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            tI[k] = plane1<kHalf>(L.curr_I, o[k]);
            tx[k] = plane1<kHalf>(L.dIdx, o[k]);
            ty[k] = plane1<kHalf>(L.dIdy, o[k]);
        }
    }
    float row[7];
    if (kIcp && icp_ok) {
        const f3 vc = {cv.x, cv.y, cv.z};
        const f3 ng = rotate(P, f3{ln.x, ln.y, ln.z});
        const f3 nc = {cn.x, cn.y, cn.z};
        const f3 dv = sub(vg, vc), cn3 = cross(nc, ng);
        const float dist = kHalf ? fast_sqrt(dot(dv, dv)) : norm(dv);
        const float sine = kHalf ? fast_sqrt(dot(cn3, cn3)) : norm(cn3);
        if (sine < a.angle && dist <= a.dthr && !isnan(nc.x) && !isnan(ng.x)) {
            const f3 c = cross(vg, ng);
            row[0] = ng.x; row[1] = ng.y; row[2] = ng.z;
            row[3] = c.x; row[4] = c.y; row[5] = c.z;
            row[6] = dot(ng, sub(vc, vg));
            sums.icp(row);
        }
    }
    if (kRgb && rgb_ok) {
        const float cx = u0 - floorf(u0), cy = v0 - floorf(v0);
        const float ic = (tI[0] * (1.0f - cx) + tI[1] * cx) * (1.0f - cy) + (tI[2] * (1.0f - cx) + tI[3] * cx) * cy;
        const float dx = (tx[0] * (1.0f - cx) + tx[1] * cx) * (1.0f - cy) + (tx[2] * (1.0f - cx) + tx[3] * cx) * cy;
        const float dy = (ty[0] * (1.0f - cx) + ty[1] * cx) * (1.0f - cy) + (ty[2] * (1.0f - cx) + ty[3] * cx) * cy;
        if ((dx > 2.0f || dy > 2.0f) && isfinite(ic) && isfinite(dx) && isfinite(dy)) {
            const float zi = kHalf ? iz : 1.0f / vg.z;
            f3 l;
            l.x = dx * L.K.fx * zi;
            l.y = dy * L.K.fy * zi;
            l.z = -(l.x * vg.x + l.y * vg.y) * zi;
            float r = ic - il;
            const double sd = (double)stddev;
            if (sd > 10e-5) r = kHalf ? r * __builtin_amdgcn_rcpf(stddev) : r / stddev;
            float w = 1.0f;
            if (fabsf(r) > th && sd > 10e-6)
                w = kHalf ? fast_sqrt(th * __builtin_amdgcn_rcpf(fabsf(r))) : sqrtf(th / fabsf(r));
            const f3 c = cross(vg, l);
            row[6] = w * (-r);
            row[0] = l.x * w; row[1] = l.y * w; row[2] = l.z * w;
            row[3] = c.x * w; row[4] = c.y * w; row[5] = c.z * w;
            sums.rgb(row);
        }
    }
}

// ---------------------------------------------------------- FP64 SE(3) helpers
// The FP64 helpers let the compiler fuse multiply-adds (one rounding instead
// of two, half the instructions of the serial step); the FP32 row arithmetic
// above keeps the reference's separate roundings.
LF_DEV void m34_identity(double *T) {
    for (int i = 0; i < 12; ++i) T[i] = (i == 0 || i == 5 || i == 10) ? 1.0 : 0.0;
}
LF_DEV void m34_mul(const double *A, const double *B, double *C) {
#pragma clang fp contract(fast)
    double t[12];
    for (int i = 0; i < 3; ++i) {
        for (int j = 0; j < 3; ++j) t[i * 4 + j] = A[i * 4] * B[j] + A[i * 4 + 1] * B[4 + j] + A[i * 4 + 2] * B[8 + j];
        t[i * 4 + 3] = A[i * 4] * B[3] + A[i * 4 + 1] * B[7] + A[i * 4 + 2] * B[11] + A[i * 4 + 3];
    }
    for (int i = 0; i < 12; ++i) C[i] = t[i];
}
LF_DEV void m34_inv(const double *A, double *C) {
#pragma clang fp contract(fast)
    double t[12];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) t[i * 4 + j] = A[j * 4 + i];
    for (int i = 0; i < 3; ++i) t[i * 4 + 3] = -(t[i * 4] * A[3] + t[i * 4 + 1] * A[7] + t[i * 4 + 2] * A[11]);
    for (int i = 0; i < 12; ++i) C[i] = t[i];
}
// SE(3) exponential, tangent [upsilon; omega] (Sophus order); Barfoot sec. 7.1.
// The coefficients A = sin t / t, B = (1 - cos t) / t^2, C = (t - sin t) / t^3:
// below t = 0.02 (every step of a converging track) their Maclaurin series to
// the t^8 term, whose remainder is below 1e-20 relative there and which avoids
// the cancellation of 1 - cos t; above it one sincos and one division.
LF_DEV void se3_exp(const double *xi, double *T) {
#pragma clang fp contract(fast)
    const double *u = xi, *w = xi + 3;
    const double th2 = w[0] * w[0] + w[1] * w[1] + w[2] * w[2];
    const double W[9] = {0, -w[2], w[1], w[2], 0, -w[0], -w[1], w[0], 0};
    double W2[9];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) W2[i * 3 + j] = W[i * 3] * W[j] + W[i * 3 + 1] * W[3 + j] + W[i * 3 + 2] * W[6 + j];
    double A, B, C;
    if (th2 < 4e-4) {
        const double t = th2;
        A = 1.0 - t * (1.0 / 6) * (1.0 - t * (1.0 / 20) * (1.0 - t * (1.0 / 42) * (1.0 - t * (1.0 / 72))));
        B = 0.5 * (1.0 - t * (1.0 / 12) * (1.0 - t * (1.0 / 30) * (1.0 - t * (1.0 / 56) * (1.0 - t * (1.0 / 90)))));
        C = (1.0 / 6) * (1.0 - t * (1.0 / 20) * (1.0 - t * (1.0 / 42) * (1.0 - t * (1.0 / 72) * (1.0 - t * (1.0 / 110)))));
    } else {
        const double th = sqrt(th2), r = 1.0 / th;
        double s, c;
        sincos(th, &s, &c);
        A = s * r;
        B = (1.0 - c) * r * r;
        C = (th - s) * r * r * r;
    }
    double V[9];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) {
            const double I = i == j ? 1.0 : 0.0;
            T[i * 4 + j] = I + A * W[i * 3 + j] + B * W2[i * 3 + j];
            V[i * 3 + j] = I + B * W[i * 3 + j] + C * W2[i * 3 + j];
        }
    for (int i = 0; i < 3; ++i) T[i * 4 + 3] = V[i * 3] * u[0] + V[i * 3 + 1] * u[1] + V[i * 3 + 2] * u[2];
}
// Norm of the SE(3) logarithm (Barfoot sec. 7.1.3).
LF_DEV double se3_log_norm(const double *T) {
#pragma clang fp contract(fast)
    double c = (T[0] + T[5] + T[10] - 1) * 0.5;
    c = fmax(-1.0, fmin(1.0, c));
    double th = acos(c);
    const double v[3] = {T[9] - T[6], T[2] - T[8], T[4] - T[1]};
    double w[3];
    if (th < 1e-8) {
        for (int i = 0; i < 3; ++i) w[i] = 0.5 * v[i];
    } else if (M_PI - th < 1e-6) {
        // k = index of the largest diagonal entry (first one on ties); the
        // row of R is selected without a runtime array index
        const int k1 = T[5] > T[0] ? 1 : 0;
        const int k = T[10] > (k1 ? T[5] : T[0]) ? 2 : k1;
        const double r0 = k == 0 ? T[0] : k == 1 ? T[4] : T[8];
        const double r1 = k == 0 ? T[1] : k == 1 ? T[5] : T[9];
        const double r2 = k == 0 ? T[2] : k == 1 ? T[6] : T[10];
        const double rkk = k == 0 ? r0 : k == 1 ? r1 : r2;
        const double axk = sqrt(fmax(0.0, (rkk + 1) * 0.5));
        const double ax0 = k == 0 ? axk : r0 / (2 * axk);
        const double ax1 = k == 1 ? axk : r1 / (2 * axk);
        const double ax2 = k == 2 ? axk : r2 / (2 * axk);
        w[0] = ax0 * th;
        w[1] = ax1 * th;
        w[2] = ax2 * th;
    } else {
        const double s = th / (2 * sin(th));
        for (int i = 0; i < 3; ++i) w[i] = s * v[i];
    }
    const double th2 = w[0] * w[0] + w[1] * w[1] + w[2] * w[2];
    th = sqrt(th2);
    const double W[9] = {0, -w[2], w[1], w[2], 0, -w[0], -w[1], w[0], 0};
    double W2[9];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) W2[i * 3 + j] = W[i * 3] * W[j] + W[i * 3 + 1] * W[3 + j] + W[i * 3 + 2] * W[6 + j];
    const double D = th < 1e-8 ? 1.0 / 12 : (1 - th * sin(th) / (2 * (1 - cos(th)))) / th2;
    double n2 = th2;
    for (int i = 0; i < 3; ++i) {
        double s = 0;
        for (int j = 0; j < 3; ++j) {
            const double Vi = (i == j ? 1.0 : 0.0) - 0.5 * W[i * 3 + j] + D * W2[i * 3 + j];
            s += Vi * T[j * 4 + 3];
        }
        n2 += s * s;
    }
    return sqrt(n2);
}
// LDL^T solve of a symmetric positive definite 6x6 (no pivoting); one
// division per pivot (its reciprocal scales the column and the solution).
LF_DEV void ldlt6(const double *A, const double *b, double *x) {
#pragma clang fp contract(fast)
    double L[36], D[6], Dinv[6];
#pragma unroll
    for (int i = 0; i < 36; ++i) L[i] = 0.0;
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        // row j of L D, shared by the updates of the rows below it
        double LD[6];
        double d = A[j * 6 + j];
#pragma unroll
        for (int k = 0; k < j; ++k) {
            LD[k] = L[j * 6 + k] * D[k];
            d -= L[j * 6 + k] * LD[k];
        }
        D[j] = d;
        Dinv[j] = d != 0.0 ? 1.0 / d : 0.0;
        L[j * 6 + j] = 1.0;
#pragma unroll
        for (int i = j + 1; i < 6; ++i) {
            double s = A[i * 6 + j];
#pragma unroll
            for (int k = 0; k < j; ++k) s -= L[i * 6 + k] * LD[k];
            L[i * 6 + j] = s * Dinv[j];
        }
    }
    double y[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        double s = b[i];
#pragma unroll
        for (int k = 0; k < i; ++k) s -= L[i * 6 + k] * y[k];
        y[i] = s;
    }
#pragma unroll
    for (int i = 0; i < 6; ++i) y[i] *= Dinv[i];
#pragma unroll
    for (int i = 5; i >= 0; --i) {
        double s = y[i];
#pragma unroll
        for (int k = i + 1; k < 6; ++k) s -= L[k * 6 + i] * x[k];
        x[i] = s;
    }
}
// create_jtjjtr<6,7> (reduce_sum.h:48-61) of the combined sums: A and b.
LF_DEV void unpack27(const double *s, double *A, double *b) {
    int k = 0;
    for (int i = 0; i < 6; ++i)
        for (int j = i; j < 7; ++j) {
            const double v = s[k++];
            if (j == 6) b[i] = v;
            else A[j * 6 + i] = A[i * 6 + j] = v;
        }
}

// One Gauss-Newton step of compute_transform (icp_tracker.cpp:50-139), run by
// a single lane after the sums are final: updates g.
LF_DEV void gn_step(LfGnState &g, const double *sums, int first_iter, bool context_mode) {
    if (first_iter) {
        g.icp_error = FLT_MAX;
        g.rgb_error = FLT_MAX;
        g.icp_count = g.rgb_count = 0;
        g.active = 1;
    }
    double last[12];
    for (int k = 0; k < 12; ++k) last[k] = g.est[k];
    const float last_icp = g.icp_error, last_rgb = g.rgb_error;
    g.last_icp_error = last_icp;
    // the residual terms in FP32, as the reference's (m_estimator.cu:470-480)
    const float icp_r2 = (float)sums[27], icp_n = (float)sums[28];
    const float rgb_r2 = (float)sums[29], rgb_n = (float)sums[30];
    g.stddev = sqrtf(rgb_r2 / (rgb_n - 6.0f));
    double A[36], b[6], x[6];
    unpack27(sums, A, b);
    ldlt6(A, b, x);
    double E[12];
    se3_exp(x, E);
    m34_mul(E, last, g.est);
    g.iterations++;
    bool stop = false, revert = false;
    float icp_error = sqrtf(icp_r2) / icp_n;
    if (isnan(icp_error) && !context_mode) {
        g.invalid = 1;
        stop = true;
    } else if (icp_error > last_icp) {
        if (g.icp_count >= 2) {
            revert = stop = true;
        } else {
            g.icp_count++;
            icp_error = last_icp;
        }
    } else {
        g.icp_count = 0;
    }
    g.icp_error = icp_error;
    if (!stop) {
        float rgb_error = sqrtf(rgb_r2) / rgb_n;
        if (isnan(rgb_error) && !context_mode) {
            g.invalid = 1;
            stop = true;
        } else if (rgb_error > last_rgb) {
            if (g.rgb_count >= 2) {
                revert = stop = true;
            } else {
                g.rgb_count++;
                rgb_error = last_rgb;
            }
        } else {
            g.rgb_count = 0;
        }
        g.rgb_error = rgb_error;
    }
    // Revertable<SE3d>::revert: the estimate goes back to the one before the step
    if (revert)
        for (int k = 0; k < 12; ++k) g.est[k] = last[k];
    g.active = stop ? 0 : 1;
}

// A value (float or double) as its 32-bit words, lane l receiving lane l ^ o's.
// Within a row of 16 lanes by DPP; a ds_bpermute (__shfl_xor) goes through the
// LDS pipe, which the 64 shuffles of a block reduction's 8 wavefronts filled
// for 2.3 us of each tracking step.
template <int o>
LF_DEV int xor_word(int x) {
    static_assert(o == 1 || o == 2 || o == 4 || o == 8, "inside a row");
    if constexpr (o == 8) return __builtin_amdgcn_mov_dpp(x, 0x128, 0xF, 0xF, false);       // row_ror:8
    else if constexpr (o == 2) return __builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, false);   // quad_perm 2,3,0,1
    else if constexpr (o == 1) return __builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, false);   // quad_perm 1,0,3,2
    else return __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(x, 0x141, 0xF, 0xF, false), 0x1B, 0xF, 0xF,
                                         false);  // row_half_mirror (l ^ 7), then quad_perm 3,2,1,0 (l ^ 3)
}
template <int o>
LF_DEV float xor_lane(float v) { return __int_as_float(xor_word<o>(__float_as_int(v))); }
template <int o>
LF_DEV double xor_lane(double v) {
    return __hiloint2double(xor_word<o>(__double2hiint(v)), xor_word<o>(__double2loint(v)));
}
// a and b exchanged between lanes 32 (16) apart: the upper half (odd row) of a
// with the lower half (even row) of b.
template <int o>
LF_DEV void swap_word(unsigned int &a, unsigned int &b) {
    static_assert(o == 32 || o == 16, "halves or rows");
    const auto r = o == 32 ? __builtin_amdgcn_permlane32_swap(a, b, false, false)
                           : __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
template <int o>
LF_DEV float swap_sum(float a, float b) {
    unsigned int x = __float_as_uint(a), y = __float_as_uint(b);
    swap_word<o>(x, y);
    return __uint_as_float(x) + __uint_as_float(y);
}
template <int o>
LF_DEV double swap_sum(double a, double b) {
    unsigned int xl = (unsigned int)__double2loint(a), xh = (unsigned int)__double2hiint(a),
                 yl = (unsigned int)__double2loint(b), yh = (unsigned int)__double2hiint(b);
    swap_word<o>(xl, yl);
    swap_word<o>(xh, yh);
    return __hiloint2double((int)xh, (int)xl) + __hiloint2double((int)yh, (int)yl);
}

// Wavefront sum of N values per lane (N a power of two, 4 to 64) as a
// transpose butterfly: at each exchange a lane keeps half of its values and
// sends the other half to its partner, so N values cost N - 1 + 6 - log2(N)
// exchanges instead of 6 N.  Afterwards lane l holds the wavefront total of
// value l >> (6 - log2 N).  Fixed pairing: deterministic.
// (Compile-time recursion keeps every index constant, so v stays in VGPRs.)
template <int kOff, class T>
LF_DEV T sum_lanes(T v) {
    if constexpr (kOff >= 1) return sum_lanes<kOff / 2>(v + xor_lane<kOff>(v));
    else return v;
}
template <int N, int kOff, class T>
LF_DEV void transpose_halve(T *v, int lane) {
    if constexpr (N > 1) {
        constexpr int h = N / 2;
#pragma unroll
        for (int i = 0; i < h; ++i) {
            if constexpr (kOff >= 16) {  // lanes with bit kOff clear keep v[i], the others v[h + i]
                v[i] = swap_sum<kOff>(v[i], v[h + i]);
            } else {
                const bool hi = (lane & kOff) != 0;
                const T keep = hi ? v[h + i] : v[i];
                const T send = hi ? v[i] : v[h + i];
                v[i] = keep + xor_lane<kOff>(send);
            }
        }
        transpose_halve<h, kOff / 2>(v, lane);
    } else {
        v[0] = sum_lanes<kOff>(v[0]);
    }
}

template <int N, class T>
LF_DEV T transpose_reduce(T (&v)[N]) {
    static_assert(N >= 4 && N <= 64 && (N & (N - 1)) == 0, "N must be a power of two, 4 to 64");
    transpose_halve<N, 32>(v, __lane_id());
    return v[0];
}

// Partial sums of one workgroup in value order: transpose butterfly in each
// wavefront, leaving value l >> 1 in lane l, then the wavefronts meet in LDS.
// Lanes with tid < kVals return value tid (the others return 0).
LF_DEV float block_sums(FloatSums &sums, float (*s_wave)[32]) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float w = transpose_reduce<32>(sums.s);
    if ((lane & 1) == 0) s_wave[wave][lane >> 1] = w;
    __syncthreads();
    float t = 0.0f;
    if (tid < kVals) {
#pragma unroll
        for (int k = 0; k < kWaves; ++k) t += s_wave[k][tid];
    }
    return t;
}

// The sums of G <= 64 kChunks partial rows of kN <= 32 values (value v of
// workgroup g at v * G + g) in a fixed order: wavefront w takes values w, w +
// kWaves, ..., a lane adds partials l, l + 64, ... of each, then a transpose
// butterfly over the wavefront's values.  The totals land in s_sum; the caller
// synchronises before reading them.  Every load of a value comes first, then
// the sum: indices past G are clamped and their values masked to +0 with a
// bitwise AND (a select of a loaded value becomes a branch around the load with
// a wait inside it), which leaves the sum unchanged: started at +0 it is never
// -0.
LF_DEV float mask_word(float v, bool keep) { return __uint_as_float(__float_as_uint(v) & (keep ? ~0u : 0u)); }
LF_DEV double mask_word(double v, bool keep) {
    return __longlong_as_double((long long)((unsigned long long)__double_as_longlong(v) & (keep ? ~0ull : 0ull)));
}
// Stores and loads that every XCD's workgroups see (relaxed, agent scope).
template <class T>
LF_DEV void store_agent(T *p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <class T>
LF_DEV T load_agent(const T *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// This wavefront's stores have arrived where those loads look (a wait alone:
// what it orders went out past the caches).
LF_DEV void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// kAgent: rows written by this launch.
template <int kChunks, int kN, bool kAgent, class T>
LF_DEV void final_sums_chunks(const T *partials, int G, T *s_sum) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr int kPer = 4;
    static_assert(kPer * kWaves >= kN, "values per wavefront");
    T acc[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int v = wave + kWaves * j;
        const T *src = partials + (size_t)(v < kN ? v : 0) * G;
        T x[kChunks];
#pragma unroll
        for (int c = 0; c < kChunks; ++c) {
            const int g = c * 64 + lane;
            const T *q = src + (g < G ? g : G - 1);
            x[c] = mask_word(kAgent ? load_agent(q) : *q, v < kN && g < G);
        }
        T s = 0;
#pragma unroll
        for (int c = 0; c < kChunks; ++c) s += x[c];
        acc[j] = s;
    }
    const T s = transpose_reduce<kPer>(acc);
    const int v = wave + kWaves * (lane >> 4);
    if ((lane & 15) == 0 && v < kN) s_sum[v] = s;
}
// (a batch of 16 systems: 32 rows; a lone system's levels: at most 256)
template <int kN, bool kAgent = false, class T>
LF_DEV void final_sums(const T *partials, int G, T *s_sum) {
    if (G <= 64) final_sums_chunks<1, kN, kAgent>(partials, G, s_sum);
    else if (G <= 256) final_sums_chunks<4, kN, kAgent>(partials, G, s_sum);
    else final_sums_chunks<kGrid / 64, kN, kAgent>(partials, G, s_sum);
}

// The combined FP64 sums of one workgroup: transpose butterfly over the 32
// (padded) values in each wavefront, leaving value l >> 1 in lane l, then
// the wavefronts meet in LDS.  Lanes with tid < kTrackVals return value tid.
LF_DEV double block_sums_d(CombinedSums &sums, double (*s_wave)[32]) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    sums.s[28] = (double)sums.n_icp;
    sums.s[30] = (double)sums.n_rgb;
    const double w = transpose_reduce<32>(sums.s);
    if ((lane & 1) == 0) s_wave[wave][lane >> 1] = w;
    __syncthreads();
    double t = 0.0;
    if (tid < kTrackVals) {
#pragma unroll
        for (int k = 0; k < kWaves; ++k) t += s_wave[k][tid];
    }
    return t;
}

// Whether this lane's share of G <= 64 kChunks flags all hold the tag, every load in
// flight at once (a loop that ends at the first other flag takes 64 of them a memory
// round: 0.7 us more a launch at 512 workgroups).
template <int kChunks>
LF_DEV bool all_set(const unsigned long long *flags, int G, unsigned long long tag) {
    unsigned long long f[kChunks], differ = 0ull;
#pragma unroll
    for (int c = 0; c < kChunks; ++c) f[c] = load_agent(&flags[min(c * 64 + (int)threadIdx.x, G - 1)]);
#pragma unroll
    for (int c = 0; c < kChunks; ++c) differ |= f[c] ^ tag;
    return differ == 0ull;
}

// Stand-alone reductions (lf_icp_reduce, lf_rgb_step) in one launch.  kMode 1:
// ICP rows, 2: RGB rows.  Each workgroup writes its kVals partials value-major
// (value v of workgroup g at v * G + g), then its flag, and reads every flag: the
// workgroup that finds them all set sums the rows.  Nothing waits for another
// workgroup, and the scratch needs no clearing first: a flag is set when it
// holds the call's own tag, and the summing workgroup clears them all (a
// captured call has the same tag at every replay).  Rows and flags pass through
// the memory that all XCDs see (relaxed agent-scope atomics): each workgroup
// waits for its rows' stores before its flag's, and for its flag's before it
// reads the others, so the one whose flag arrives last sees them all.  Another
// may too: both store the same sums.
// A small call's time is its launches on the host, a large one's the rows.  An ICP and
// a photometric reduction, in two launches each and now, us among others (waited for
// alone): 160x120 17.6 and 13.9 (31.5 and 27.9), 320x240 17.6 and 14.2 (31.8 and 29.9),
// 640x480 20.4 and 19.6 (36.2 and 35.7), 848x480 21.9 and 22.1 (38.3 and 38.4), 1280x960
// 36.5 and 36.5 (52.6 and 52.6).
template <int kMode>
__global__ __launch_bounds__(kThreads) void k_reduce(ReduceArgs a, float *__restrict__ out29, unsigned long long *flags,
                                                     unsigned long long tag) {
    __shared__ float s_wave[kWaves][32], s_sum[32];
    __shared__ int s_all;
    constexpr bool kIcp = kMode == 1, kRgb = kMode == 2;
    const int tid = threadIdx.x, G = gridDim.x;
    float P[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) P[k] = a.pose12[k];
    const float stddev = a.stddev;
    const float th = (float)(1.345 * (double)stddev);
    FloatSums sums;
    sums.clear();
    const int n = a.lv.cols * a.lv.rows;
    for (int i = blockIdx.x * kThreads + tid; i < n; i += G * kThreads)
        pixel_rows<kIcp, kRgb, false>(a, load_own<kIcp, kRgb>(a.lv, i), P, stddev, th, sums);
    const float t = block_sums(sums, s_wave);
    if (tid < 64) {
        if (tid < kVals) store_agent(&a.partials[(size_t)tid * G + blockIdx.x], t);
        wait_stores();
        if (tid == 0) store_agent(&flags[blockIdx.x], tag);
        wait_stores();
        const bool all = G <= 64 ? all_set<1>(flags, G, tag) : G <= 256 ? all_set<4>(flags, G, tag)
                                                                        : all_set<kGrid / 64>(flags, G, tag);
        if (__ballot(all) == ~0ull && tid == 0) s_all = 1;
        else if (tid == 0) s_all = 0;
    }
    __syncthreads();
    if (!s_all) return;
    final_sums<kVals, true>(a.partials, G, s_sum);
    __syncthreads();
    if (tid < kVals) out29[tid] = s_sum[tid];
    for (int g = tid; g < G; g += kThreads) store_agent(&flags[g], 0ull);
}

// The pose as record `number` (0: none).
LF_DEV void record_pose(LfTrackState &st, const double *pose, unsigned long long number) {
    if (number == 0ull) return;
    LfPoseRecord r;
    for (int k = 0; k < 12; ++k) r.pose[k] = pose[k];
    r.number = number;
    r.check = lf_pose_check(r);
    st.record[number & 1ull] = r;
}

// End of DenseTracking::compute_transform (icp_tracker.cpp:143-155) and the
// odometry chain of DenseOdometry::trackFrame (rgbd_odometry.cpp:39): success
// test, update = est^-1 (or identity), pose = pose * update, pose24 refreshed.
// est and invalid are the frame's final estimate and flag (already in st).
LF_DEV void track_finish(LfTrackState &st, const double *est, int invalid, bool context_mode,
                         unsigned long long record) {
    double inv_est[12], D[12];
    m34_inv(est, inv_est);
    m34_mul(inv_est, st.init, D);
    // compute_transform(ctx) reports success unconditionally (icp_tracker.cpp:308-313)
    const bool ok = context_mode || (!invalid && !(se3_log_norm(D) > 0.1));
    st.success = ok ? 1 : 0;
    double upd[12];
    if (ok) for (int k = 0; k < 12; ++k) upd[k] = inv_est[k];
    else m34_identity(upd);
    double P[12];
    m34_mul(st.pose, upd, P);
    double Pi[12];
    m34_inv(P, Pi);
    for (int k = 0; k < 12; ++k) {
        st.pose[k] = P[k];
        st.pose24[k] = (float)P[k];
        st.pose24[12 + k] = (float)Pi[k];
    }
    record_pose(st, P, record);
}

// LDS of a tracking step's workgroup: the wavefronts' partial sums, and what
// the previous step's solve leaves for this one.
struct StepLds {
    double wave[kWaves][32], sum[32];
    float pose[12], stddev;
    int run;
};

// The partial rows of step k: two halves of the scratch taken in turn, as a
// step's workgroups read the previous step's rows while others write theirs.
LF_DEV double *step_partials(const ReduceArgs &a, int k) {
    return reinterpret_cast<double *>(a.partials) + (size_t)(k & 1) * (kGrid * kTrackVals);
}

// The previous step's end, at the head of every workgroup of this one: its
// partial rows summed in a fixed order, then the FP64 solve on one lane, whose
// pose is this step's.  Every workgroup computes the same; workgroup 0 stores
// the state (the two slots in turn, for the same reason as the rows).  Lane 0
// returns the state.  The rows are loaded beside the state, before it says
// whether they are wanted: after a kernel boundary each dependent round of
// loads costs about 1 us.
LF_DEV LfGnState solve_previous(const ReduceArgs &a, int wg, StepLds &s) {
    const int tid = threadIdx.x;
    LfTrackState &st = *a.st;
    LfGnState g = st.slot[(a.step - 1) & 1];
    final_sums<kTrackVals>(step_partials(a, a.step - 1), a.prev_grid, s.sum);
    __syncthreads();
    // a failed frame, or a level that broke out of its loop: no step was taken
    const bool ran = !g.invalid && (a.prev_first_iter || g.active);
    if (tid == 0) {
        double before[12];
        for (int k = 0; k < 12; ++k) before[k] = g.est[k];
        if (ran) gn_step(g, s.sum, a.prev_first_iter, a.context_mode != 0);
#pragma unroll
        for (int k = 0; k < 12; ++k) s.pose[k] = (float)g.est[k];
        s.stddev = g.stddev;
        s.run = !g.invalid && (a.first_iter || g.active);
        if (wg == 0) {
            st.slot[a.step & 1] = g;
            if (ran) {
                st.gn = g;
                for (int k = 0; k < 12; ++k) st.prev[k] = before[k];
            }
        }
    }
    __syncthreads();
    if (ran && wg == 0 && tid < kTrackVals) st.sums[tid] = s.sum[tid];
    return g;
}

// One Gauss-Newton iteration of compute_transform: the previous step's solve,
// then every workgroup sums the ICP and RGB rows of its pixels into one partial
// row.  The pose-independent loads of the first pixel are in flight during the
// solve.  One launch per step: a step's own kernel boundary is the only wait
// between the rows and their sum.  (The solve in a launch of its own, one
// workgroup, cost 3.6-4.3 us a step beside 5.3-6.6 us of rows; a
// last-workgroup ticket costs 11 ns per workgroup, as atomics on one address
// are taken in turn, and more than the launch from 128 workgroups on.)
// A coarse level's step is latency: of its 14.8k cycles (7.0-7.5 us with the
// launch, 20.5k with ds_bpermute butterflies) 3.7k load the state and the
// rows, 3.4k solve, 3.7k are two rounds of pixel loads and 2.6k the block's
// sums; a 640x480 step (11.3 us) has 13k cycles of pixels, by their
// instructions.  Re-tracking at 320x240: 246 -> 192 us a call.
// Workgroup wg of the nwg computing the step's partial rows.  kHalf: FP16 maps.
template <bool kHalf>
LF_DEV void track_step_wg(const ReduceArgs &a, int wg, int nwg, StepLds &s) {
    const int tid = threadIdx.x;
    const int n = a.lv.cols * a.lv.rows;
    const int stride = nwg * kThreads;
    int i = wg * kThreads + tid;
    Own o = {};
    if (i < n) o = load_own<true, true, kHalf>(a.lv, i);
    float P[12], stddev;
    if (a.step == 0) {
#pragma unroll
        for (int k = 0; k < 12; ++k) P[k] = a.init_f[k];
        stddev = 0.0f;
        if (wg == 0 && tid == 0) {
            LfGnState g = {};
            for (int k = 0; k < 12; ++k) a.st->init[k] = g.est[k] = a.init[k];
            a.st->slot[0] = g;
        }
    } else {
        solve_previous(a, wg, s);
        if (!s.run) return;
#pragma unroll
        for (int k = 0; k < 12; ++k) P[k] = uniform_f(s.pose[k]);
        stddev = a.first_iter ? 0.0f : uniform_f(s.stddev);
    }
    const float th = (float)(1.345 * (double)stddev);
    CombinedSums sums;
    sums.clear();
    sums.w = (double)a.icp_weight;
    while (i < n) {
        const Own cur = o;
        const int next = i + stride;
        if (next < n) o = load_own<true, true, kHalf>(a.lv, next);
        pixel_rows<true, true, kHalf>(a, cur, P, stddev, th, sums);
        i = next;
    }
    const double t = block_sums_d(sums, s.wave);
    if (tid < kTrackVals) step_partials(a, a.step)[(size_t)tid * nwg + wg] = t;
}

// Held to 128 VGPRs: 4 waves per SIMD, two 512-lane workgroups per CU.
template <bool kHalf>
__global__ __launch_bounds__(kThreads, 4) void k_track_step(ReduceArgs a) {
    __shared__ StepLds s;
    track_step_wg<kHalf>(a, blockIdx.x, gridDim.x, s);
}

// After the frame's last step (one workgroup): its solve, then the finish.  A
// frame that ended before (an error became NaN, the finest level broke out of
// its loop) left the estimate as it was then.
LF_DEV void track_end_wg(const ReduceArgs &a, StepLds &s, unsigned long long record) {
    const LfGnState g = solve_previous(a, 0, s);
    if (threadIdx.x == 0) track_finish(*a.st, g.est, g.invalid, a.context_mode != 0, record);
}

__global__ __launch_bounds__(kThreads) void k_track_end(ReduceArgs a, unsigned long long record) {
    __shared__ StepLds s;
    track_end_wg(a, s, record);
}

// Launch arguments read from a descriptor table, their pointers asserted global.
LF_DEV ReduceArgs global_args(const ReduceArgs &d) {
    ReduceArgs a = d;
    LfTrackLevel &L = a.lv;
    L.curr_vmap = global_ptr(d.lv.curr_vmap); L.curr_nmap = global_ptr(d.lv.curr_nmap);
    L.last_vmap = global_ptr(d.lv.last_vmap); L.last_nmap = global_ptr(d.lv.last_nmap);
    L.curr_I = global_ptr(d.lv.curr_I); L.last_I = global_ptr(d.lv.last_I);
    L.dIdx = global_ptr(d.lv.dIdx); L.dIdy = global_ptr(d.lv.dIdy);
    a.pose12 = global_ptr(d.pose12); a.partials = global_ptr(d.partials);
    a.st = global_ptr(d.st);
    return a;
}

// One system's step of a batch: its launch arguments and its grid (0: the
// system has nothing at this index).
struct TrackJob {
    ReduceArgs a;
    int G;
    unsigned long long record;  // number of the end's pose record (0: none)
};

// Step s of several systems (each its own tracker state, scratch and
// pyramids): a 2-D grid whose y index is the system; each system's workgroups
// run exactly the single launch's code.
template <bool kHalf>
__global__ __launch_bounds__(kThreads, 4) void k_track_step_batch(const TrackJob *__restrict__ jobs) {
    __shared__ StepLds s;
    const TrackJob &j = jobs[blockIdx.y];
    if ((int)blockIdx.x >= j.G) return;
    track_step_wg<kHalf>(global_args(j.a), blockIdx.x, j.G, s);
}

// The end of each system's frame: workgroup i, system i.
__global__ __launch_bounds__(kThreads) void k_track_end_batch(const TrackJob *__restrict__ jobs) {
    __shared__ StepLds s;
    const TrackJob &j = jobs[blockIdx.x];
    if (j.G <= 0) return;
    track_end_wg(global_args(j.a), s, j.record);
}

__global__ void k_track_finish(LfTrackState *st, unsigned long long record) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    LfTrackState &s = *st;
    double est[12];
    for (int k = 0; k < 12; ++k) est[k] = s.gn.est[k];
    track_finish(s, est, s.gn.invalid, false, record);
}

__global__ void k_track_begin(LfTrackState *st, double t0, double t1, double t2, double t3, double t4, double t5,
                              double t6, double t7, double t8, double t9, double t10, double t11) {
    const double T[12] = {t0, t1, t2, t3, t4, t5, t6, t7, t8, t9, t10, t11};
    for (int k = 0; k < 12; ++k) {
        st->gn.est[k] = T[k];
        st->prev[k] = T[k];
        st->init[k] = T[k];
    }
    st->gn.invalid = 0;
    st->gn.active = 1;
    st->gn.iterations = 0;
}

__global__ void k_track_set_pose(LfTrackState *st, unsigned long long record, double t0, double t1, double t2,
                                 double t3, double t4, double t5, double t6, double t7, double t8, double t9, double t10, double t11) {
    const double T[12] = {t0, t1, t2, t3, t4, t5, t6, t7, t8, t9, t10, t11};
    double Ti[12];
    m34_inv(T, Ti);
    for (int k = 0; k < 12; ++k) {
        st->pose[k] = T[k];
        st->pose24[k] = (float)T[k];
        st->pose24[12 + k] = (float)Ti[k];
    }
    st->success = 1;
    record_pose(*st, T, record);
}

// The state to pinned host memory: a launch and a wait take about 20 us less than a
// copy to pageable memory and a wait (a tracked 320x240 frame 169 -> 147 us,
// a System frame of 640x480 390 -> 369).
__global__ __launch_bounds__(256) void k_track_read(const LfTrackState *st, LfTrackState *host) {
    static_assert(sizeof(LfTrackState) % 8 == 0, "whole words");
    const unsigned long long *src = reinterpret_cast<const unsigned long long *>(st);
    unsigned long long *dst = reinterpret_cast<unsigned long long *>(host);
    for (unsigned int i = threadIdx.x; i < sizeof(LfTrackState) / 8; i += blockDim.x) dst[i] = src[i];
}

int check_level(const LfTrackLevel &lv) {
    if (lv.cols <= 0 || lv.rows <= 0) return lf_set_error(LF_ERR_ARG, "bad level size %dx%d", lv.cols, lv.rows);
    return LF_OK;
}

float icp_angle() { return (float)cos(30 * 3.14 / 180); }

// Workgroups of a reduction: one pixel per lane, at most kGrid workgroups.
int grid_for(const LfTrackLevel &lv) {
    const long n = (long)lv.cols * lv.rows;
    return (int)std::max(1L, std::min((long)kGrid, (n + kThreads - 1) / kThreads));
}

}  // namespace

// The stand-alone reductions' kGrid x kVals FP32 partials (a caller's scratch
// holds more than that: its size is part of the interface).
size_t lf_reduce_partials(void) { return (size_t)kGrid * 62 + 64; }
// The tracking steps' two halves of kGrid x kTrackVals FP64 partials.
size_t lf_track_scratch_floats(void) { return (size_t)kGrid * kTrackVals * 2 * 2; }

extern "C" size_t lf_reduce_scratch_floats(void) { return lf_reduce_partials(); }

int lf_track_begin(LfTrackState *st, const double *T, hipStream_t stream) {
    k_track_begin<<<1, 1, 0, stream>>>(st, T[0], T[1], T[2], T[3], T[4], T[5], T[6], T[7], T[8], T[9], T[10], T[11]);
    LF_LAUNCH_CHECK();
    return LF_OK;
}

static ReduceArgs step_args(const LfTrackLevel &lv, float *scratch, LfTrackState *st, const LfStepFlags &f,
                            float icp_weight) {
    ReduceArgs a = {};
    a.lv = lv;
    a.angle = icp_angle();
    a.dthr = 0.01f;
    a.partials = scratch;
    a.st = st;
    a.step = f.step;
    a.first_iter = f.first_of_level;
    a.prev_first_iter = f.prev_first_of_level;
    a.prev_grid = f.prev_grid;
    a.icp_weight = icp_weight;
    a.context_mode = f.context_mode;
    for (int k = 0; k < 12; ++k) {
        a.init[k] = f.init[k];
        a.init_f[k] = (float)f.init[k];
    }
    return a;
}

// Workgroups of a tracking step of one of `share` systems (wgs > 0: given):
// a lone system takes 256, one per CU.  Each of them sums all of the
// previous step's rows, and a level-0 lane then sums two pixels with the
// second one's loads in flight.  (A whole 640x480 frame on 128 or 512: 1.05x
// and 1.04x the time; one at 320x240 on 128: 1.05x.)
static int step_grid(const LfTrackLevel &lv, int share, int wgs, int end) {
    if (end) return 1;
    return std::min(grid_for(lv), wgs > 0 ? std::min(wgs, kGrid) : std::max(1, std::min(kStepGrid, kGrid / std::max(1, share))));
}

int lf_track_step(const LfTrackLevel &lv, float *scratch, LfTrackState *st, const LfStepFlags &f, float icp_weight,
                  hipStream_t stream, int *grid) {
    if (int rc = check_level(lv)) return rc;
    const ReduceArgs a = step_args(lv, scratch, st, f, icp_weight);
    const int G = step_grid(lv, 1, 0, f.end);
    if (f.end) k_track_end<<<1, kThreads, 0, stream>>>(a, f.record);
    else if (lv.half_maps) k_track_step<true><<<G, kThreads, 0, stream>>>(a);
    else k_track_step<false><<<G, kThreads, 0, stream>>>(a);
    LF_LAUNCH_CHECK();
    if (grid) *grid = G;
    return LF_OK;
}

size_t lf_track_job_bytes(void) { return sizeof(TrackJob); }

int lf_track_job_make(const LfTrackLevel &lv, float *scratch, LfTrackState *st, const LfStepFlags &f,
                      float icp_weight, int share, int wgs, void *job, int *grid) {
    if (int rc = check_level(lv)) return rc;
    TrackJob &j = *static_cast<TrackJob *>(job);
    j = TrackJob{};
    j.a = step_args(lv, scratch, st, f, icp_weight);
    // 16 systems at 640x480: 32 workgroups each instead of 512 (the step's
    // lanes sum ~19 level-0 pixels each, with the next pixel's loads in
    // flight, and do 1/16 of the block reductions): 4.1k -> 4.7k frames/s
    // aggregate in mixed precision.  16 and 64 workgroups each measured
    // slower than 32 (5.46k and 5.61k against 5.74k).
    j.G = step_grid(lv, share, wgs, f.end);
    j.record = f.record;
    if (grid) *grid = j.G;
    return LF_OK;
}

void lf_track_job_skip(void *job) {
    TrackJob &j = *static_cast<TrackJob *>(job);
    j = TrackJob{};
    j.G = 0;
}

int lf_track_batch_step(const void *jobs, int n, int gmax, int half_maps, hipStream_t stream) {
    if (!jobs || n <= 0 || n > 65535) return lf_set_error(LF_ERR_ARG, "bad tracking batch of %d", n);
    const TrackJob *J = static_cast<const TrackJob *>(jobs);
    if (gmax <= 0) return LF_OK;
    if (half_maps) k_track_step_batch<true><<<dim3(gmax, n), kThreads, 0, stream>>>(J);
    else k_track_step_batch<false><<<dim3(gmax, n), kThreads, 0, stream>>>(J);
    LF_LAUNCH_CHECK();
    return LF_OK;
}

int lf_track_batch_end(const void *jobs, int n, hipStream_t stream) {
    if (!jobs || n <= 0 || n > 65535) return lf_set_error(LF_ERR_ARG, "bad tracking batch of %d", n);
    k_track_end_batch<<<n, kThreads, 0, stream>>>(static_cast<const TrackJob *>(jobs));
    LF_LAUNCH_CHECK();
    return LF_OK;
}

int lf_track_finish(LfTrackState *st, unsigned long long record, hipStream_t stream) {
    k_track_finish<<<1, 64, 0, stream>>>(st, record);
    LF_LAUNCH_CHECK();
    return LF_OK;
}

int lf_track_set_pose(LfTrackState *st, const double *T, unsigned long long record, hipStream_t stream) {
    k_track_set_pose<<<1, 1, 0, stream>>>(st, record, T[0], T[1], T[2], T[3], T[4], T[5], T[6], T[7], T[8], T[9], T[10],
                                          T[11]);
    LF_LAUNCH_CHECK();
    return LF_OK;
}

int lf_track_read(const LfTrackState *st, LfTrackState *host, hipStream_t stream) {
    k_track_read<<<1, 256, 0, stream>>>(st, host);
    LF_LAUNCH_CHECK();
    return LF_OK;
}

// A tag that no other call of either reduction in this process has (they may share a
// scratch) and that no float pair is likely to hold.
static unsigned long long next_tag() {
    static std::atomic<unsigned long long> calls{0};
    return 0x9E3779B97F4A7C15ull * (calls.fetch_add(1, std::memory_order_relaxed) + 1);
}

// Floats of the most rows and the flags behind them on an 8-byte boundary.
constexpr size_t kRowsAndFlags = (size_t)kGrid * kVals + 2 * kGrid + 1;
// A caller's scratch holds them twice with room for the sums between.
static_assert((size_t)kGrid * 62 + 64 >= 2 * kRowsAndFlags + kVals, "sums inside the scratch overlap one place only");

// The launch of a stand-alone reduction: rows and flags share the scratch of
// `capacity` floats.  They lie at its start, or at its end where the caller has the
// sums written into the start: one workgroup may store them while another still
// reads the rows.
template <int kMode>
static int launch_reduce(ReduceArgs &a, float *scratch, size_t capacity, float *sum29, hipStream_t st) {
    const int G = grid_for(a.lv);
    const auto overlap = [](const float *x, size_t nx, const float *y, size_t ny) {
        return std::less<const float *>()(x, y + ny) && std::less<const float *>()(y, x + nx);
    };
    const size_t shift = capacity > kRowsAndFlags && overlap(sum29, kVals, scratch, kRowsAndFlags) ? capacity - kRowsAndFlags : 0;
    capacity -= shift;
    scratch += shift;
    a.partials = scratch;
    // the flags behind the most rows, on an 8-byte boundary
    const uintptr_t end = reinterpret_cast<uintptr_t>(scratch + (size_t)kGrid * kVals);
    auto *flags = reinterpret_cast<unsigned long long *>((end + 7) & ~(uintptr_t)7);
    if (reinterpret_cast<uintptr_t>(flags + G) > reinterpret_cast<uintptr_t>(scratch + capacity))
        return lf_set_error(LF_ERR_CAPACITY, "a reduction of %d workgroups does not fit %zu scratch floats", G, capacity);
    k_reduce<kMode><<<G, kThreads, 0, st>>>(a, sum29, flags, next_tag());
    LF_LAUNCH_CHECK();
    return LF_OK;
}

// icp_reduce of lf_icp_reduce and lf_icp_reduce_noalloc.
static int icp_reduce_into(const float *curr_vmap, const float *curr_nmap, const float *last_vmap,
                           const float *last_nmap, int cols, int rows, const float *pose12, const lf_intrinsics *K,
                           float *partials, size_t capacity, float *sum29, hipStream_t st) {
    ReduceArgs a = {};
    a.lv.curr_vmap = curr_vmap; a.lv.curr_nmap = curr_nmap; a.lv.last_vmap = last_vmap; a.lv.last_nmap = last_nmap;
    a.lv.cols = cols; a.lv.rows = rows; a.lv.K = *K;
    if (int rc = check_level(a.lv)) return rc;
    if ((long long)cols * rows > INT_MAX)
        return lf_set_error(LF_ERR_ARG, "icp_reduce: %dx%d is more than %d pixels", cols, rows, INT_MAX);
    a.pose12 = pose12;
    a.angle = icp_angle();
    a.dthr = 0.01f;
    return launch_reduce<1>(a, partials, capacity, sum29, st);
}

extern "C" int lf_icp_reduce(const float *curr_vmap, const float *curr_nmap, const float *last_vmap,
                             const float *last_nmap, int cols, int rows, const float *pose12,
                             const lf_intrinsics *K, float *scratch, float *sum29, void *stream) {
    if (!curr_vmap || !curr_nmap || !last_vmap || !last_nmap || !pose12 || !K || !scratch || !sum29)
        return lf_set_error(LF_ERR_ARG, "null argument to icp_reduce");
    return icp_reduce_into(curr_vmap, curr_nmap, last_vmap, last_nmap, cols, rows, pose12, K, scratch,
                           lf_reduce_partials(), sum29, lf_stream(stream));
}

// Scratch of lf_icp_reduce_noalloc: the partial rows of at most kGrid
// workgroups (116 KiB, half of it used), one copy per GPU, held until the
// process ends.  Host code never passes the array's name to a kernel or a
// copy: on the host it is only a stand-in for the symbol, so its device
// address is looked up per device (hipGetSymbolAddress, with that device
// current) and that address is used everywhere.
constexpr size_t kNoallocScratchFloats = (size_t)kGrid * 58;
static __device__ __align__(256) float scratch[kNoallocScratchFloats];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
float *g_scratch_dev[kMaxDevices] = {};

// The current device's address of `scratch`, resolved on its first use there.
int noalloc_scratch(float **out) {
    int dev = -1;
    LF_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices)
        return lf_set_error(LF_ERR_ARG, "device %d is beyond the %d devices of the fixed scratch", dev, kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_dev[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return lf_set_error(LF_ERR_HIP, "hipGetSymbolAddress of the fixed scratch failed on device %d: %s", dev,
                                hipGetErrorString(e));
        g_scratch_dev[dev] = static_cast<float *>(p);
    }
    *out = g_scratch_dev[dev];
    return LF_OK;
}
}  // namespace

extern "C" int lf_icp_reduce_noalloc(const float *curr_vmap, const float *curr_nmap, const float *last_vmap,
                                     const float *last_nmap, int cols, int rows, const float *pose12,
                                     const lf_intrinsics *K, float *sum29, void *stream) {
    if (!curr_vmap || !curr_nmap || !last_vmap || !last_nmap || !pose12 || !K || !sum29)
        return lf_set_error(LF_ERR_ARG, "null argument to icp_reduce_noalloc");
    float *partials = nullptr;
    if (int rc = noalloc_scratch(&partials)) return rc;
    // every partial that is summed is written by the call itself, and a flag
    // left from elsewhere is not its tag, so nothing in the scratch needs clearing
    return icp_reduce_into(curr_vmap, curr_nmap, last_vmap, last_nmap, cols, rows, pose12, K, partials,
                           kNoallocScratchFloats, sum29, lf_stream(stream));
}

extern "C" int lf_rgb_step(const float *curr_intensity, const float *last_intensity, const float *last_vmap,
                           const float *intensity_dx, const float *intensity_dy, int cols, int rows,
                           float stddev_estimate, const float *pose12, const lf_intrinsics *K, float *scratch,
                           float *sum29, void *stream) {
    if (!curr_intensity || !last_intensity || !last_vmap || !intensity_dx || !intensity_dy || !pose12 || !K ||
        !scratch || !sum29)
        return lf_set_error(LF_ERR_ARG, "null argument to rgb_step");
    ReduceArgs a = {};
    a.lv.last_vmap = last_vmap; a.lv.curr_I = curr_intensity; a.lv.last_I = last_intensity;
    a.lv.dIdx = intensity_dx; a.lv.dIdy = intensity_dy;
    a.lv.cols = cols; a.lv.rows = rows; a.lv.K = *K;
    if (int rc = check_level(a.lv)) return rc;
    a.pose12 = pose12;
    a.stddev = stddev_estimate;
    return launch_reduce<2>(a, scratch, lf_reduce_partials(), sum29, lf_stream(stream));
}

extern "C" void lf_unpack_jtjjtr(const float *sum29, float *jtj36, float *jtr6, float *residual2) {
    int k = 0;
    for (int i = 0; i < 6; ++i)
        for (int j = i; j < 7; ++j) {
            const float v = sum29[k++];
            if (j == 6) jtr6[i] = v;
            else jtj36[j * 6 + i] = jtj36[i * 6 + j] = v;
        }
    residual2[0] = sum29[27];
    residual2[1] = sum29[28];
}

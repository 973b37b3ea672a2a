// orient.hip -- grid lookups, OA-time docking and orientation averages.
//
// Lookup: GetAmpAtPointInPlaneJacob (Backend/GPU/CommonJacobGPUMethods.cu:69-154)
//   = cubic Hermite in phi on 4 theta rows + 4-point spline in theta, and the
//   4-plane q spline (OAJacob.cu:57-113, HybridOA.cu:78-133; GetSphr
//   Backend/Backend/Grid.cpp:487-548 for single points).
// Docking: AddAmplitudeAtPoint (HybridOA.cu:17-159): for each rotation
//   (R = Rx(a)Ry(b)Rz(c), Amplitude.h:557-573) A_leaf(R^T q) * sum_t e^{i q.t} * scale.
// MC: directions (theta = acos(2u-1), phi = 2 pi v) from a counter-based Philox
//   stream keyed by (seed; direction, shell group), so any launch shape and any
//   batch composition reproduce the same numbers (the reference draws them from
//   a clock-seeded MTGP32, GPUHybridCalc.cu:196-198), stratified per chunk
//   (mc_stratify: a wave's 64 directions share one equal-area patch, so its
//   gathers hit neighbouring grid cells).
// VEGAS: 32x32 (cos theta, phi) bins, bin-volume weighted estimate, per-bin
//   variance marginals and the damped re-binning of HybridOA.cu:181-449.
//
// Node layout: one T4 per grid node = (Re A, Im A, Re dA/dphi-spline, Im ...),
// so the two phi neighbours of a lookup are one contiguous 2*sizeof(T4) read.

#include "common.hpp"
#include "device.hpp"

namespace dplus {

template <typename T>
struct cplx {
    T x, y;
};

template <typename T>
__device__ __forceinline__ cplx<T> hermite(cplx<T> p1, cplx<T> p2, cplx<T> d1, cplx<T> d2, T t) {
    T t2 = t * t, t3 = t2 * t;
    cplx<T> r;
    r.x = p1.x + d1.x * t + ((T)3 * (p2.x - p1.x) - (T)2 * d1.x - d2.x) * t2 +
          ((T)2 * (p1.x - p2.x) + d1.x + d2.x) * t3;
    r.y = p1.y + d1.y * t + ((T)3 * (p2.y - p1.y) - (T)2 * d1.y - d2.y) * t2 +
          ((T)2 * (p1.y - p2.y) + d1.y + d2.y) * t3;
    return r;
}

// PeriodicSplineSolver.h:227-234 / CommonJacobGPUMethods.cu:34-63
template <typename T>
__device__ __forceinline__ void four_point(const cplx<T> y[4], cplx<T> &d2, cplx<T> &d3) {
    const T a = (T)(7. / 15.), b = (T)(14. / 15.), c = (T)(4. / 15.), e = (T)(2. / 15.);
    d2.x = -a * (y[1].x - y[0].x) + b * (y[2].x - y[0].x) - c * (y[3].x - y[1].x) + e * (y[3].x - y[2].x);
    d2.y = -a * (y[1].y - y[0].y) + b * (y[2].y - y[0].y) - c * (y[3].y - y[1].y) + e * (y[3].y - y[2].y);
    d3.x = e * (y[1].x - y[0].x) - c * (y[2].x - y[0].x) + b * (y[3].x - y[1].x) - a * (y[3].x - y[2].x);
    d3.y = e * (y[1].y - y[0].y) - c * (y[2].y - y[0].y) + b * (y[3].y - y[1].y) - a * (y[3].y - y[2].y);
}

constexpr double kInvPi = 0.31830988618379067153776752674503;
constexpr double kInv2Pi = 0.15915494309189533576888376337251;

// theta / pi of cos theta = 2 u - 1.  For FP32 lookups 2 asin(sqrt y) / pi, y = 1 - u, by a
// polynomial of asin(sqrt y) / sqrt y on [0, 1/2] (9e-14) and sqrt by one Newton step on the
// FP32 root (1e-14): a cell's fraction stays well below FP32's rounding of it.
template <typename T>
__device__ __forceinline__ double polar_fraction(double u) {
    if (sizeof(T) == 8) return acos(2.0 * u - 1.0) * kInvPi;
    const bool flip = u < 0.5;
    const double y = fmax(flip ? u : 1.0 - u, 1e-30);
    const float s0 = __builtin_amdgcn_sqrtf((float)y);
    double s = (double)s0;
    s = fma(fma(-s, s, y), (double)(0.5f * __builtin_amdgcn_rcpf(s0)), s);
    const double c[14] = {0.6366197723674882,   0.10610329546639952, 0.047746473800039865, 0.02842098102029294,
                          0.019329935850208507, 0.014425052426250716, 0.009232696985335458, 0.02102495864195202,
                          -0.048506457009034394, 0.18417602577157377, -0.3818597693281228,  0.5575447279642045,
                          -0.46861904441904245, 0.19281950697472416};
    double v = c[13];
#pragma unroll
    for (int i = 12; i >= 0; i--) v = fma(v, y, c[i]);
    return flip ? 1.0 - s * v : s * v;
}

// phi / 2 pi in [0, 1] of the direction (x, y).  For FP32 lookups atan(t) / 2 pi by a polynomial
// (3e-14) of t = min / max, the quotient by one Newton step on the FP32 reciprocal.
template <typename T>
__device__ __forceinline__ double azimuth_fraction(double y, double x) {
    if (sizeof(T) == 8) {
        double ph = atan2(y, x);
        if (ph < 0.0) ph += k2Pi;
        return ph * kInv2Pi;
    }
    const double ax = fabs(x), ay = fabs(y), mx = fmax(fmax(ax, ay), 1e-30), mn = fmin(ax, ay);
    double r = (double)__builtin_amdgcn_rcpf((float)mx);
    r = fma(fma(-mx, r, 1.0), r, r);
    const double t = mn * r, z = t * t;
    const double c[15] = {0.15915494309185563,   -0.05305164767892841,  0.03183098720372489,   -0.022736377200679544,
                          0.017683185381863295,  -0.014461797164107013, 0.012198398114540248,  -0.010409938335242477,
                          0.008704539505489512,  -0.006766065864383247, 0.004557582911667102,  -0.0024539396615994905,
                          0.0009607892649646508, -0.0002385112965010332, 2.785172736474061e-05};
    double v = c[14];
#pragma unroll
    for (int i = 13; i >= 0; i--) v = fma(v, z, c[i]);
    v *= t;
    v = ay > ax ? 0.25 - v : v;
    v = x < 0.0 ? 0.5 - v : v;
    return y < 0.0 ? 1.0 - v : v;
}

// sin and cos of an angle of FP32 amplitudes' phases: reduced in FP64 to an eighth of a turn
// and evaluated by polynomials (1e-15 there)
__device__ __forceinline__ void phase_poly(double angle, double &s, double &c) {
    const double t = angle * kInv2Pi, k = rint(4.0 * t), r = fma(-0.25, k, t), z = r * r;
    const double a[7] = {6.283185307179589, -41.34170224040016, 81.60524927661358, -76.70585994242144,
                         42.05872054224183, -15.096148222634003, 3.8374156880543087};
    const double b[7] = {1.0000000000000004, -19.73920880217851, 64.93939402246923, -85.45681712812244,
                         60.24462568572577, -26.424620552027367, 7.818904292222803};
    double u = a[6], v = b[6];
#pragma unroll
    for (int i = 5; i >= 0; i--) {
        u = fma(u, z, a[i]);
        v = fma(v, z, b[i]);
    }
    u *= r;
    const int q = (int)(long long)k;
    s = (q & 1) ? v : u;
    c = (q & 1) ? u : v;
    s = (q & 2) ? -s : s;
    c = ((q + 1) & 2) ? -c : c;
}
template <typename T>
__device__ __forceinline__ void phase_exact(double angle, double &s, double &c) {
    if (sizeof(T) == 8)
        sincos(angle, &s, &c);
    else
        phase_poly(angle, s, c);
}

// weights of the 4-point spline (four_point's end derivatives, then the cubic
// Hermite at t) over values y0..y3, as cubics in t: the spline at t is sum_r w[r] y[r].
// w[1] = 1 + t (-1/5 + t (-9/5 + t)) closes the sum to 1, so that rounding scales nothing.
template <typename T>
__device__ __forceinline__ void spline4_weights(T t, T w[4]) {
    w[0] = t * ((T)(-7. / 15.) + t * ((T)(4. / 5.) - (T)(1. / 3.) * t));
    w[2] = t * ((T)(4. / 5.) + t * ((T)(6. / 5.) - t));
    w[3] = t * ((T)(-2. / 15.) + t * ((T)(-1. / 5.) + (T)(1. / 3.) * t));
    w[1] = ((T)1 - w[2]) - (w[0] + w[3]);
}

// the same for a q, whose weights every direction shares: formed in FP64
template <typename T>
__device__ __forceinline__ void q_weights(double t, T w[4]) {
    double v[4];
    spline4_weights<double>(t, v);
    w[0] = (T)v[0];
    w[2] = (T)v[2];
    w[3] = (T)v[3];
    w[1] = ((T)1 - w[2]) - (w[0] + w[3]);
}

// cell and fraction of 0 <= x < 2^31 by FP64 additions (the conversions run at a quarter of
// their rate): x - 1/2 rounds to the cell in the low mantissa bits of x - 1/2 + 1.5 2^52.  At
// a node the cell may be the lower one, with fraction 1: the same interpolated value.
__device__ __forceinline__ double cell_of(double x, int &i) {
    const double magic = 6755399441055744.0, t = (x - 0.5) + magic;
    i = (int)(unsigned)__double_as_longlong(t);
    return x - (t - magic);
}

// one theta-phi plane (shell >= 1) at theta = ut pi, phi = up 2 pi; kZeroTiny
// reproduces the CPU variant's snapping of interpolation fractions below 1e-10
// (Grid.cpp:1242-1245).  The cell and fractions are the reference's
// theta / (pi / 3i) and phi / (2 pi / 6i) (CommonJacobGPUMethods.cu:69-154),
// formed as products with the direction's ut and up; the row and column
// wrap-arounds are branches instead of integer remainders.
template <typename T, typename T4, bool kZeroTiny>
__device__ cplx<T> plane_lookup(const T4 *__restrict__ plane, int shell, double ut, double up) {
    const int phiPoints = 6 * shell, thePoints = 3 * shell;
    const double xt = ut * (double)thePoints, xp = up * (double)phiPoints;
    if constexpr (sizeof(T) == 4) {
        // FP32 nodes: the cell by FP64 additions (a node may be its lower cell's upper end) and
        // the interpolation by weights, half the instructions of the forms below
        int t0, p0;
        double ft = cell_of(xt, t0), fp = cell_of(xp, p0);
        if (t0 < 0) {  // x < 2^-54 may round below the first cell
            t0 = 0;
            ft = 0.0;
        }
        if (p0 < 0) {
            p0 = 0;
            fp = 0.0;
        }
        p0 = p0 == phiPoints ? 0 : p0;
        const int p1 = p0 + 1 == phiPoints ? 0 : p0 + 1;
        const T p = (T)fp, p2 = p * p, p3 = p2 * p;
        const T h01 = (T)3 * p2 - (T)2 * p3, h00 = (T)1 - h01, h11 = p3 - p2, h10 = h11 - p2 + p;
        T w[4];
        spline4_weights<T>((T)ft, w);
        cplx<T> a = {(T)0, (T)0};
#pragma unroll
        for (int r = 0; r < 4; r++) {
            int v = t0 + r - 1, k0 = p0, k1 = p1;  // v in [-1, thePoints + 1]
            if (v < 0 || v > thePoints) {
                // past a pole: the row on the other side, half a turn away in phi
                v = v < 0 ? v + thePoints + 1 : v - (thePoints + 1);
                k0 += k0 >= thePoints ? -thePoints : thePoints;
                k1 += k1 >= thePoints ? -thePoints : thePoints;
            }
            const T4 A = plane[phiPoints * v + k0], B = plane[phiPoints * v + k1];
            const T x = h00 * A.x + h01 * B.x + h10 * A.z + h11 * B.z;
            const T y = h00 * A.y + h01 * B.y + h10 * A.w + h11 * B.w;
            a.x += w[r] * x;
            a.y += w[r] * y;
        }
        return a;
    }
    const int tI = (int)xt;
    int pI = (int)xp;
    double tphd = xp - (double)pI;
    double tthd = xt - (double)tI;
    if (kZeroTiny) {
        if (fabs(tthd) < 1.0e-10) tthd = 0.0;
        if (fabs(tphd) < 1.0e-10) tphd = 0.0;
    }
    const T tph = (T)tphd, tth = (T)tthd;
    pI = (pI == phiPoints) ? 0 : pI;
    const int pI1 = (pI + 1 == phiPoints) ? 0 : pI + 1;
    const int half = phiPoints / 2;
    cplx<T> nn[4];
#pragma unroll
    for (int rl = -1; rl < 3; rl++) {
        const int v = tI + rl;  // in [-1, thePoints + 2]
        int pos1, pos2;
        if (v < 0 || v > thePoints) {
            // past a pole: the row on the other side, half a turn away in phi
            const int theInd = v < 0 ? v + thePoints + 1 : v - (thePoints + 1);
            pos1 = phiPoints * theInd + pI + ((2 * pI >= phiPoints) ? -half : half);
            pos2 = phiPoints * theInd + pI1 + ((2 * pI1 >= phiPoints) ? -half : half);
        } else {
            pos1 = phiPoints * v + pI;
            pos2 = phiPoints * v + pI1;
        }
        const T4 a = plane[pos1], b = plane[pos2];
        nn[rl + 1] = hermite<T>({a.x, a.y}, {b.x, b.y}, {a.z, a.w}, {b.z, b.w}, tph);
    }
    cplx<T> d1, d2;
    four_point<T>(nn, d1, d2);
    return hermite<T>(nn[1], nn[2], d1, d2, tth);
}


__device__ __forceinline__ void antipode(double th, double ph, double &nth, double &nph) {
    double a = kPi - th, b = ph + kPi;
    if (b < 0) b = k2Pi + (b - (int)(b / k2Pi) * k2Pi);
    if (b >= k2Pi) b = b - (int)(b / k2Pi) * k2Pi;
    nth = fmin(fmax(a, 0.0), kPi);
    nph = b;
}

// planes layer-1 .. layer+2 and the q-spline derivatives (OAJacob.cu:57-98)
template <typename T, typename T4>
__device__ __forceinline__ void group_planes(const T4 *__restrict__ g, int layer, double th, double ph,
                                             cplx<T> amps[4], cplx<T> &d1, cplx<T> &d2) {
    const double ut = th * kInvPi, up = ph * kInv2Pi;
#pragma unroll
    for (int i = -1; i <= 2; i++) {
        const int lqi = i + layer;
        if (lqi == -1) {
            double nth, nph;
            antipode(th, ph, nth, nph);
            amps[i + 1] = plane_lookup<T, T4, false>(g + 1, 1, nth * kInvPi, nph * kInv2Pi);
        } else if (lqi == 0) {
            const T4 o = g[0];
            amps[i + 1] = {o.x, o.y};
        } else {
            amps[i + 1] = plane_lookup<T, T4, false>(g + shell_base(lqi), lqi, ut, up);
        }
    }
    four_point<T>(amps, d1, d2);
}

// one plane's lookup out of line, for the rare ones: the origin (layer 0's plane), the antipode
// on shell 1 (plane -1), directions next to a pole or a row's end, patches larger than a tile
template <typename T, typename T4>
__device__ __noinline__ cplx<T> plane_direct(const T4 *__restrict__ g, int lqi, double ut, double up) {
    if (lqi == 0) {
        const T4 o = g[0];
        return {o.x, o.y};
    }
    if (lqi < 0) {
        double nth, nph;
        antipode(ut * kPi, up * k2Pi, nth, nph);
        return plane_lookup<T, T4, false>(g + 1, 1, nth * kInvPi, nph * kInv2Pi);
    }
    return plane_lookup<T, T4, false>(g + shell_base(lqi), lqi, ut, up);
}

// the four planes layer - 1 .. layer + 2 at (pi ut, 2 pi up), FP32 nodes.  Where no lane of the
// wave is next to a pole or at a row's last column (most waves: their directions are
// neighbours), the eight nodes are four 32-bit offsets from the plane's base, each row's
// pair one load apart; else plane_lookup's wrapped addresses.
__device__ __forceinline__ void planes32(const float4 *__restrict__ g, int layer, double ut, double up,
                                         cplx<float> amps[4]) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int lqi = layer - 1 + i;
        if (lqi <= 0) {
            amps[i] = plane_direct<float, float4>(g, lqi, ut, up);
            continue;
        }
        const float4 *plane = g + shell_base(lqi);
        const int n = 6 * lqi, m = 3 * lqi;
        int t0, p0;
        const float t = (float)cell_of(ut * (double)m, t0), p = (float)cell_of(up * (double)n, p0);
        if (__ballot(t0 < 1 || t0 > m - 2 || p0 < 0 || p0 > n - 2) != 0) {
            amps[i] = plane_direct<float, float4>(g, lqi, ut, up);
            continue;
        }
        const float p2 = p * p, p3 = p2 * p;
        const float h01 = 3.f * p2 - 2.f * p3, h00 = 1.f - h01, h11 = p3 - p2, h10 = h11 - p2 + p;
        float w[4];
        spline4_weights<float>(t, w);
        unsigned off = (unsigned)((t0 - 1) * n + p0) * (unsigned)sizeof(float4);
        const unsigned row = (unsigned)n * (unsigned)sizeof(float4);
        float4 A[4], B[4];
#pragma unroll
        for (int r = 0; r < 4; r++, off += row) {
            const float4 *q = (const float4 *)((const char *)plane + off);
            A[r] = q[0];
            B[r] = q[1];
        }
        cplx<float> a = {0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; r++) {
            a.x += w[r] * (h00 * A[r].x + h01 * B[r].x + h10 * A[r].z + h11 * B[r].z);
            a.y += w[r] * (h00 * A[r].y + h01 * B[r].y + h10 * A[r].w + h11 * B[r].w);
        }
        amps[i] = a;
        // one plane's loads in flight: four planes' would hold 128 registers, and two more waves
        // per SIMD hide as much
        __builtin_amdgcn_sched_barrier(0);
    }
}

// R^T q with R = Rx(a) Ry(b) Rz(c): HybridOA.cu:60-63
__device__ __forceinline__ void rotate_t(const RotDev &r, const double q[3], double o[3]) {
#pragma unroll
    for (int i = 0; i < 3; i++) o[i] = r.m[3 * i] * q[0] + r.m[3 * i + 1] * q[1] + r.m[3 * i + 2] * q[2];
}

// phase factor e^{i q d} for the docking translations: FP64 argument, reduced
// to revolutions in FP64 and evaluated by the hardware sin/cos in mixed mode
template <typename T>
__device__ __forceinline__ void phase_sincos(double qd, T &s, T &c);
template <>
__device__ __forceinline__ void phase_sincos<float>(double qd, float &s, float &c) {
    double r = qd * (1.0 / k2Pi);
    float f = (float)(r - floor(r));
    s = __builtin_amdgcn_sinf(f);
    c = __builtin_amdgcn_cosf(f);
}
template <>
__device__ __forceinline__ void phase_sincos<double>(double qd, double &s, double &c) {
    sincos(qd, &s, &c);
}

constexpr int kMaxM = 16;  // q-values of one shell group handled per pass (one lookup serves all)


// accumulate the docked amplitude along unit direction qv for q-values qs[0..m), m <= M,
// (900 copies of two leaves in 120 rotations, 8,192 directions, grid 150: 6.58 -> 5.23 ms with
// polynomial angles, interpolation weights and the phase sums taken before the amplitudes,
// which also shortens their rounding: 4.0e-6 -> 7e-7 of I(q); 2,190 -> 1,850 VALU instructions
// a lookup, issued 0.71 of the clocks at 2 waves per SIMD beside the gathers)
// whose weights over the four planes are wq (q_weights, in LDS).
// stepq (equally spaced q, single precision): the translations of a rotation
// with several step their phases in q, e^{i q_j d} = e^{i q_0 d} (e^{i dq d})^j:
// two range-reduced sin/cos per translation and one complex rotation per further
// q instead of one sin/cos per q (a single translation keeps the direct form)
template <typename T, typename T4, int M = kMaxM>
__device__ __forceinline__ void docked_amplitude(const T4 *const *__restrict__ grids,
                                                 const RotDev *__restrict__ rots, int nrot,
                                                 const double4 *__restrict__ trans, int layer, const double qv[3],
                                                 const double *__restrict__ qs, const T (*wq)[4], int m, bool stepq,
                                                 cplx<T> acc[M]) {
    const bool rec = sizeof(T) == 4 && stepq && m > 1;
    const double q0t = qs[0] * kInv2Pi, dqt = rec ? (qs[m - 1] - qs[0]) / (double)(m - 1) * kInv2Pi : 0.0;
    for (int r = 0; r < nrot; r++) {
        const RotDev &rd = rots[r];
        double rv[3];
        rotate_t(rd, qv, rv);
        if (fabs(rv[2]) > 1.) rv[2] = (rv[2] > 0.) ? 1. : -1.;
        cplx<T> amps[4];
        if constexpr (sizeof(T) == 4) {
            planes32(grids[rd.leaf], layer, polar_fraction<T>(0.5 + 0.5 * rv[2]), azimuth_fraction<T>(rv[1], rv[0]), amps);
        } else {
            const double nth = acos(rv[2]);
            double nph = atan2(rv[1], rv[0]);
            if (nph < 0.0) nph += k2Pi;
            cplx<T> d1, d2;
            group_planes<T, T4>(grids[rd.leaf], layer, nth, nph, amps, d1, d2);
        }
        const T sc = (T)rd.scale;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            amps[p].x *= sc;
            amps[p].y *= sc;
        }
        // (the weights are read from LDS for every rotation: kept across the loop they would
        // take 4 M registers)
        int zero = 0;
        asm volatile("" : "+v"(zero));
        auto amplitude = [&](int j) {
            const T *wj = wq[j + zero];
            const T w0 = wj[0], w1 = wj[1], w2 = wj[2], w3 = wj[3];
            return cplx<T>{w0 * amps[0].x + w1 * amps[1].x + w2 * amps[2].x + w3 * amps[3].x,
                           w0 * amps[0].y + w1 * amps[1].y + w2 * amps[2].y + w3 * amps[3].y};
        };
        const int nt = rd.nt, t0 = rd.t0;
        const bool trivial = nt == 1 && trans[t0].x == 0.0 && trans[t0].y == 0.0 && trans[t0].z == 0.0;
        if (rec && nt > 1) {
            // the phases' sums over the translations first, the amplitudes times them once
            cplx<T> sum[M];
#pragma unroll
            for (int j = 0; j < M; j++) sum[j] = {(T)0, (T)0};
            for (int tr = 0; tr < nt; tr++) {
                const double4 tt = trans[t0 + tr];
                const double d = tt.x * qv[0] + tt.y * qv[1] + tt.z * qv[2];
                const float f = (float)__builtin_amdgcn_fract(q0t * d), e = (float)__builtin_amdgcn_fract(dqt * d);
                T cs = __builtin_amdgcn_cosf(f), sn = __builtin_amdgcn_sinf(f);
                const T cd = __builtin_amdgcn_cosf(e), sd = __builtin_amdgcn_sinf(e);
#pragma unroll
                for (int j = 0; j < M; j++) {
                    if (j < m) {
                        sum[j].x += cs;
                        sum[j].y += sn;
                        const T c2 = cs * cd - sn * sd;
                        sn = sn * cd + cs * sd;
                        cs = c2;
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < M; j++) {
                if (j < m) {
                    const cplx<T> a = amplitude(j);
                    acc[j].x += a.x * sum[j].x - a.y * sum[j].y;
                    acc[j].y += a.y * sum[j].x + a.x * sum[j].y;
                }
            }
            continue;
        }
#pragma unroll
        for (int j = 0; j < M; j++) {
            if (j < m) {
                const cplx<T> a = amplitude(j);
                if (trivial) {
                    acc[j].x += a.x;
                    acc[j].y += a.y;
                } else {
                    T sumc = 0, sums = 0;
                    for (int tr = 0; tr < nt; tr++) {
                        const double4 tt = trans[t0 + tr];
                        const double qd = qs[j] * (tt.x * qv[0] + tt.y * qv[1] + tt.z * qv[2]);
                        T s, c;
                        phase_sincos<T>(qd, s, c);
                        sumc += c;
                        sums += s;
                    }
                    acc[j].x += a.x * sumc - a.y * sums;
                    acc[j].y += a.y * sumc + a.x * sums;
                }
            }
        }
    }
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// ------------------------------------------------------------------ MC
// grid: x = direction block, y = active group.  mstride >= every group's m.
// partial[(gi * nblk + bx) * mstride + j] = sum over the block's directions of |A_j|^2
template <typename T, typename T4, bool kSingle, int M = kMaxM>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 1 : 2) void mc_kernel(const T4 *const *__restrict__ grids,
                                                 const RotDev *__restrict__ rots, int nrot,
                                                 const double4 *__restrict__ trans,
                                                 const GroupDev *__restrict__ groups,
                                                 const int *__restrict__ active, int mstride,
                                                 const double *__restrict__ qs, double step,
                                                 uint64_t seed, long long dir0, int nblk, int chunk, int nu,
                                                 int nv, double *__restrict__ partial) {
    const int gi = blockIdx.y;
    const GroupDev G = groups[active[gi]];
    const long long d = dir0 + (long long)blockIdx.x * blockDim.x + threadIdx.x;
    double u, v;
    uniform_pair(seed, (uint32_t)d, (uint32_t)(d >> 32), (uint32_t)G.layer, kStreamMC, u, v);
    mc_stratify(d, chunk, nu, nv, u, v);
    const double th = acos(2.0 * u - 1.0), ph = k2Pi * v;
    double qv[3] = {0.0, 0.0, 0.0};
    if (!kSingle) {
        double st, ct, sp, cp;
        sincos(th, &st, &ct);
        sincos(ph, &sp, &cp);
        qv[0] = cp * st;
        qv[1] = sp * st;
        qv[2] = ct;
    }
    __shared__ double red[4][kMaxM];
    __shared__ T wq[kMaxM][4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (kSingle) {
        // one lookup per direction serves every q of the group, each q reduced as it is formed
        cplx<T> amps[4], d1, d2;
        group_planes<T, T4>(grids[rots[0].leaf], G.layer, th, ph, amps, d1, d2);
        const T sc = (T)rots[0].scale;
        const double inv_step = 1.0 / step;
        for (int jb = 0; jb < G.m; jb += kMaxM) {
            const int m = min(kMaxM, G.m - jb);
#pragma unroll
            for (int j = 0; j < kMaxM; j++) {
                if (j < m) {
                    const T t = (T)((qs[G.q0 + jb + j] - G.layer * step) * inv_step);
                    const cplx<T> a = hermite<T>(amps[1], amps[2], d1, d2, t);
                    const T ax = a.x * sc, ay = a.y * sc;
                    double I = (double)ax * (double)ax + (double)ay * (double)ay;
                    I = wave_sum(I);
                    if (lane == 0) red[w][j] = I;
                }
            }
            __syncthreads();
            if (threadIdx.x < m) {
                const int j = threadIdx.x;
                partial[((size_t)gi * nblk + blockIdx.x) * mstride + jb + j] =
                    red[0][j] + red[1][j] + red[2][j] + red[3][j];
            }
            __syncthreads();
        }
        return;
    }
    // docked: M q per pass (8 when no group holds more: fewer accumulators)
    for (int jb = 0; jb < G.m; jb += M) {
        const int m = min(M, G.m - jb);
        __syncthreads();
        if (threadIdx.x < m) q_weights<T>((qs[G.q0 + jb + threadIdx.x] - G.layer * step) * (1.0 / step), wq[threadIdx.x]);
        __syncthreads();
        cplx<T> acc[M];
#pragma unroll
        for (int j = 0; j < M; j++) acc[j] = {(T)0, (T)0};
        docked_amplitude<T, T4, M>(grids, rots, nrot, trans, G.layer, qv, qs + G.q0 + jb, wq, m, G.uniform != 0, acc);
#pragma unroll
        for (int j = 0; j < M; j++) {
            double I = (double)acc[j].x * (double)acc[j].x + (double)acc[j].y * (double)acc[j].y;
            I = wave_sum(I);
            if (lane == 0) red[w][j] = I;
        }
        __syncthreads();
        if (threadIdx.x < m) {
            const int j = threadIdx.x;
            partial[((size_t)gi * nblk + blockIdx.x) * mstride + jb + j] =
                red[0][j] + red[1][j] + red[2][j] + red[3][j];
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------ MC, copies turned about z
// lane i's value of v, for a wave-uniform i
__device__ __forceinline__ double lane_value(double v, int i) {
    const unsigned long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, i);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), i);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// the sum over the wave's 64 lanes, in every lane: DPP exchanges within each row
// of 16 lanes (quad swaps, half-row and row mirrors), then the four row sums
__device__ __forceinline__ float wave_total(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, false));
    const int b = __float_as_int(v);
    return (__int_as_float(__builtin_amdgcn_readlane(b, 0)) + __int_as_float(__builtin_amdgcn_readlane(b, 16))) +
           (__int_as_float(__builtin_amdgcn_readlane(b, 32)) + __int_as_float(__builtin_amdgcn_readlane(b, 48)));
}
__device__ __forceinline__ double wave_total(double v) { return wave_sum(v); }

// the four planes' amplitudes (layer - 1 .. layer + 2) of one lookup at (th, ph),
// as group_planes takes them, without the q derivatives
template <typename T, typename T4>
__device__ __forceinline__ void direct_planes(const T4 *__restrict__ g, int layer, double th, double ph,
                                              cplx<T> amps[4]) {
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const int lqi = layer - 1 + p;
        if (lqi == -1) {
            double nth, nph;
            antipode(th, ph, nth, nph);
            amps[p] = plane_lookup<T, T4, false>(g + 1, 1, nth * kInvPi, nph * kInv2Pi);
        } else if (lqi == 0) {
            const T4 o = g[0];
            amps[p] = {o.x, o.y};
        } else {
            amps[p] = plane_lookup<T, T4, false>(g + shell_base(lqi), lqi, th * kInvPi, ph * kInv2Pi);
        }
    }
}

// direct_planes kept out of line, for the copy-major kernel's rare chunks whose
// segments do not fit: its registers then cost only on that path
template <typename T, typename T4>
__device__ __noinline__ void direct_planes_call(const T4 *__restrict__ g, int layer, double th, double ph,
                                                cplx<T> *amps) {
    direct_planes<T, T4>(g, layer, th, ph, amps);
}

// ------------------------------------------------------------------ patch tiles
// A patch of directions (an equal-area stratum, neighbouring VEGAS bins) touches a small
// rectangle of each shell's (theta, phi) nodes.  A workgroup copies the rectangle to LDS
// with coalesced loads, rows and columns wrapped as plane_lookup wraps them, and its
// directions look up there: 16-byte LDS reads at ~8..20 clocks a wave instead of
// divergent loads at 64, and one base address for the eight nodes.
struct Tile {
    int t0, p0, rows, cols, stride;
    __device__ int nodes() const { return rows * stride; }
};

// the rectangle of shell i for theta = pi [ut0, ut1], phi = 2 pi [up0, up1] (1e-6 of a cell
// of margin for the rounding of the ends)
__device__ __forceinline__ Tile patch_tile(int shell, double ut0, double ut1, double up0, double up1) {
    Tile t;
    const double m = 3.0 * shell, n = 6.0 * shell;
    t.t0 = (int)floor(ut0 * m - 1e-6) - 1;
    t.rows = (int)floor(ut1 * m + 1e-6) + 2 - t.t0 + 1;
    t.p0 = (int)floor(up0 * n - 1e-6);
    t.cols = (int)floor(up1 * n + 1e-6) + 1 - t.p0 + 1;
    t.stride = t.cols | 1;  // odd: the rows of one lookup start in different banks
    return t;
}

// 256 threads: a wave takes whole rows, or the power of two of them that fits its lanes,
// so that the column's place is worked out once and a node costs its load and its store
template <typename T4>
__device__ __forceinline__ void stage_tile(const T4 *__restrict__ plane, int shell, const Tile &t, T4 *tile) {
    const int n = 6 * shell, m = 3 * shell;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int lw = min(32 - __builtin_clz(t.cols - 1), 6), per = 64 >> lw;
    for (int c = lane & ((1 << lw) - 1); c < t.cols; c += 64) {
        int k = t.p0 + c;
        k += k < 0 ? n : 0;
        k -= k >= n ? n : 0;
        const int r0 = w * per + (lane >> lw);
        if (t.t0 >= 0 && t.t0 + t.rows <= m + 1) {  // no row past a pole
            const T4 *src = plane + (n * (t.t0 + r0) + k);
            T4 *dst = tile + r0 * t.stride + c;
            const int ds = 4 * per * n, dt = 4 * per * t.stride;
            int r = r0;
            for (; r + 12 * per < t.rows; r += 16 * per) {  // four loads in flight
                const T4 a = src[0], b = src[ds], d = src[2 * ds], e = src[3 * ds];
                dst[0] = a;
                dst[dt] = b;
                dst[2 * dt] = d;
                dst[3 * dt] = e;
                src += 4 * ds;
                dst += 4 * dt;
            }
            for (; r < t.rows; r += 4 * per) {
                *dst = *src;
                src += ds;
                dst += dt;
            }
        } else {
            const int half = k + m >= n ? k + m - n : k + m;  // past a pole: half a turn away in phi
#pragma unroll 2
            for (int r = r0; r < t.rows; r += 4 * per) {
                int v = t.t0 + r, q = k;
                if (v < 0 || v > m) {  // the row on the other side
                    v = v < 0 ? v + m + 1 : v - (m + 1);
                    q = half;
                }
                tile[r * t.stride + c] = plane[n * min(max(v, 0), m) + q];
            }
        }
    }
}

// plane_lookup on a staged tile, as sums over the nodes with the phi Hermite's and the
// theta spline's weights
template <typename T, typename T4>
__device__ __forceinline__ cplx<T> tile_lookup(const T4 *tile, const Tile &t, int shell, double ut, double up) {
    int tI, pI;
    const T s = (T)cell_of(ut * (double)(3 * shell), tI);
    const T p = (T)cell_of(up * (double)(6 * shell), pI), p2 = p * p, p3 = p2 * p;
    const T h01 = (T)3 * p2 - (T)2 * p3, h00 = (T)1 - h01, h11 = p3 - p2, h10 = h11 - p2 + p;
    T w[4];
    spline4_weights<T>(s, w);
    const T4 *row = tile + (tI - 1 - t.t0) * t.stride + (pI - t.p0);
    cplx<T> a = {(T)0, (T)0};
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const T4 A = row[r * t.stride], B = row[r * t.stride + 1];
        const T x = h00 * A.x + h01 * B.x + h10 * A.z + h11 * B.z;
        const T y = h00 * A.y + h01 * B.y + h10 * A.w + h11 * B.w;
        a.x += w[r] * x;
        a.y += w[r] * y;
    }
    return a;
}

// the planes' tiles of a patch: lane p of every four works out plane p's (shell0 + p), then
// each is read as wave-uniform values
__device__ __forceinline__ Tile tile_of(const Tile &mine, int p) {
    return {__builtin_amdgcn_readlane(mine.t0, p), __builtin_amdgcn_readlane(mine.p0, p),
            __builtin_amdgcn_readlane(mine.rows, p), __builtin_amdgcn_readlane(mine.cols, p),
            __builtin_amdgcn_readlane(mine.stride, p)};
}

// Sums of M values over groups of L lanes (L >= M, powers of two): at each step a lane
// passes on half of its values and adds the other lane's of the half it keeps, so M - 1
// exchanges and log2(L / M) more instead of M log2 L.  Returns the sum of value
// (lane % L) / (L / M).
template <int M>
__device__ __forceinline__ double group_sums(const double (&v)[M], int lane, int L) {
    if constexpr (M > 1) {
        const int o = L >> 1;
        const bool hi = lane & o;
        double u[M / 2];
#pragma unroll
        for (int i = 0; i < M / 2; i++) {
            const double send = hi ? v[i] : v[i + M / 2], keep = hi ? v[i + M / 2] : v[i];
            u[i] = keep + __shfl_xor(send, o, 64);
        }
        return group_sums<M / 2>(u, lane, o);
    } else {
        double t = v[0];
        for (int o = L >> 1; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
        return t;
    }
}

// LDS nodes of one plane's tile: 38 KB, four workgroups per CU
template <typename T4>
constexpr int tile_nodes() {
    return 38 * 1024 / (int)sizeof(T4);
}

// The MC average of a single leaf over several chunks: a workgroup takes one patch of
// the stratification (mc_stratify) and 4 D of its chunks, 64 directions each: per plane
// the patch's tile is staged once and serves 256 D lookups, and the q of the group share
// the lookups through per-q weights.  The same directions as mc_kernel; the sums over
// them are grouped by patch instead of by run of 256.  2,000 atoms, grid 100, 10^6
// directions, 500 q: 1.93 -> 0.94 ms (FP64, 262,144: 0.91 -> 0.45).  mc_kernel waits on 32
// divergent loads a lookup; here the VALU issues all the time (732 instructions counted per
// 64 directions and group, LDS reads 0.60 of the clocks), so fewer instructions are what is
// left.
template <typename T, typename T4, int D>
__global__ __launch_bounds__(256) void mc_patch_kernel(const T4 *const *__restrict__ grids,
                                                       const RotDev *__restrict__ rots,
                                                       const GroupDev *__restrict__ groups,
                                                       const int *__restrict__ active, int mstride,
                                                       const double *__restrict__ qs, double step, uint64_t seed,
                                                       long long dir0, int nchunks, int chunk, int nu, int nv, int nset,
                                                       double *__restrict__ partial) {
    __shared__ T4 tile[tile_nodes<T4>()];
    __shared__ T wq[kMaxM][4];
    __shared__ double red[4][kMaxM];
    const int gi = blockIdx.y;
    const GroupDev G = groups[active[gi]];
    const int patch = blockIdx.x / nset, set = blockIdx.x - patch * nset;
    const int iu = patch / nv, iv = patch - iu * nv;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int c0 = set * 4 * D + w;  // this wave's chunks: c0, c0 + 4, ...
    double ut[D], up[D];
    cplx<T> amp[4][D];
    const double inu = 1.0 / (double)nu, inv = 1.0 / (double)nv;
#pragma unroll
    for (int k = 0; k < D; k++) {
        const int c = min(c0 + 4 * k, nchunks - 1);  // (a chunk past the last is not summed)
        const long long d = dir0 + (long long)c * chunk + patch * 64 + lane;
        double u, v;
        uniform_pair(seed, (uint32_t)d, (uint32_t)(d >> 32), (uint32_t)G.layer, kStreamMC, u, v);
        u = ((double)iu + u) * inu;
        v = ((double)iv + v) * inv;
        ut[k] = polar_fraction<T>(u);
        up[k] = (k2Pi * v) * kInv2Pi;
    }
    const T4 *g = grids[rots[0].leaf];
    const Tile mine = patch_tile(max(G.layer - 1 + (lane & 3), 1), polar_fraction<float>((double)(iu + 1) * inu),
                                 polar_fraction<float>((double)iu * inu), (double)iv * inv, (double)(iv + 1) * inv);
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const int lqi = G.layer - 1 + p;
        const Tile t = tile_of(mine, p);
        if (lqi > 0 && t.nodes() <= tile_nodes<T4>()) {  // uniform over the workgroup
            if (p > 0) __syncthreads();
            stage_tile(g + shell_base(lqi), lqi, t, tile);
            __syncthreads();
#pragma unroll
            for (int k = 0; k < D; k++) amp[p][k] = tile_lookup<T, T4>(tile, t, lqi, ut[k], up[k]);
        } else {
#pragma unroll
            for (int k = 0; k < D; k++) amp[p][k] = plane_direct<T, T4>(g, lqi, ut[k], up[k]);
        }
    }
    const double sc2 = (double)(T)rots[0].scale * (double)(T)rots[0].scale;
    const double inv_step = 1.0 / step;
    for (int jb = 0; jb < G.m; jb += kMaxM) {
        const int m = min(kMaxM, G.m - jb);
        __syncthreads();
        if (threadIdx.x < m) {
            T q4[4];
            q_weights<T>((qs[G.q0 + jb + threadIdx.x] - G.layer * step) * inv_step, q4);
#pragma unroll
            for (int p = 0; p < 4; p++) wq[threadIdx.x][p] = q4[p];
        }
        __syncthreads();
        auto intensity = [&](int j) {
            const T w0 = wq[j][0], w1 = wq[j][1], w2 = wq[j][2], w3 = wq[j][3];
            double I = 0.0;
#pragma unroll
            for (int k = 0; k < D; k++) {
                const T ax = w0 * amp[0][k].x + w1 * amp[1][k].x + w2 * amp[2][k].x + w3 * amp[3][k].x;
                const T ay = w0 * amp[0][k].y + w1 * amp[1][k].y + w2 * amp[2][k].y + w3 * amp[3][k].y;
                if (c0 + 4 * k < nchunks) I += (double)ax * (double)ax + (double)ay * (double)ay;
            }
            return I;
        };
        // eight q at a time through the wave's sums
        for (int j0 = 0; j0 < m; j0 += 8) {
            double I[8];
#pragma unroll
            for (int j = 0; j < 8; j++) I[j] = j0 + j < m ? intensity(j0 + j) : 0.0;
            const double t = group_sums<8>(I, lane, 64);
            if ((lane & 7) == 0) red[w][j0 + (lane >> 3)] = t;
        }
        __syncthreads();
        if (threadIdx.x < m) {
            const int j = threadIdx.x;
            partial[((size_t)gi * gridDim.x + blockIdx.x) * mstride + jb + j] =
                sc2 * ((red[0][j] + red[1][j]) + (red[2][j] + red[3][j]));
        }
    }
}

constexpr int kRowNodes = 2560;

__device__ __forceinline__ int row_nodes(int layer) {  // four rows, each with its first node again at its end
    int n = 0;
#pragma unroll
    for (int p = 0; p < 4; p++) n += 6 * max(layer - 1 + p, 1) + 1;
    return n;
}
__device__ __forceinline__ bool whole_rows(int layer, int nz) {
    return 2 * nz >= 5 * (layer + 2) && row_nodes(layer) <= kRowNodes;
}

constexpr int kZWin = 64;  // nodes of one plane's collapsed row segment (one per lane)

// The MC average of a docking whose copies all turn about z (a helix): every
// copy of a direction looks up the direction's own theta rows, at phi - alpha.
// A block takes the same 256 directions (and writes the same partial sums) as
// mc_kernel, but a wave's lanes are copies: it walks its 64 directions one at a
// time (each broadcast from the lane that drew it) and, per direction, its
// copies 64 at a time in (leaf, alpha) order, so the copies of one chunk span a
// short segment of each theta row.  kCollapse (FP32 grids): the lookup is
// linear in the node data and theta is the same for every copy, so per plane
// the 4-row theta spline is applied once to the segment (at most kZWin nodes,
// one per lane; the row loads of two planes, 8 per lane, issued together and
// coalesced) into LDS, and
// each copy takes the phi Hermite of two collapsed nodes; a segment that does
// not fit, or a chunk spanning two leaves, takes the direct lookup, which
// every copy takes without kCollapse.  The q spline is applied with per-q
// weights.  The copies' amplitudes are summed over the lanes per direction,
// then |A_j|^2.
template <typename T, typename T4, bool kCollapse, int M>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 2 : 1) void mc_zcopy_kernel(
    const T4 *const *__restrict__ grids, const ZCopyDev *__restrict__ zc, int nz,
    const GroupDev *__restrict__ groups, const int *__restrict__ active, int mstride,
    const double *__restrict__ qs, double step, uint64_t seed, long long dir0, int nblk, int chunk, int nu, int nv,
    bool split, double *__restrict__ partial) {
    const int gi = blockIdx.y;
    const GroupDev G = groups[active[gi]];
    // split: the collapse instance takes the shell groups whose planes (up to
    // shell layer + 2) fit the window, the direct instance the others
    // (mc_zrows_kernel takes those with many copies for their rows)
    if (split && whole_rows(G.layer, nz)) return;
    const bool collapse_group = G.layer + 2 <= zc[0].aux;
    if (kCollapse ? !collapse_group : (split && collapse_group)) return;
    const long long d = dir0 + (long long)blockIdx.x * blockDim.x + threadIdx.x;
    double u, v;
    uniform_pair(seed, (uint32_t)d, (uint32_t)(d >> 32), (uint32_t)G.layer, kStreamMC, u, v);
    mc_stratify(d, chunk, nu, nv, u, v);
    // the wave's directions (theta, phi, unit vector), read back one at a time
    __shared__ double dirs[4][5][64];
    __shared__ double red[4][M];
    __shared__ T wq[M][4];
    __shared__ T wts[4][4][4];  // per wave and plane: the theta spline weights of the current direction
    __shared__ T4 win[4][4][kCollapse ? kZWin : 1];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    {
        const double th = acos(2.0 * u - 1.0), ph = k2Pi * v;
        double st, ct, sp, cp;
        sincos(th, &st, &ct);
        sincos(ph, &sp, &cp);
        dirs[w][0][lane] = th;
        dirs[w][1][lane] = ph;
        dirs[w][2][lane] = cp * st;
        dirs[w][3][lane] = sp * st;
        dirs[w][4][lane] = ct;
    }
    const double inv_step = 1.0 / step;
    for (int jb = 0; jb < G.m; jb += M) {
        const int m = min(M, G.m - jb);
        const double *q = qs + G.q0 + jb;
        if (threadIdx.x < m) q_weights<T>((q[threadIdx.x] - G.layer * step) * inv_step, wq[threadIdx.x]);
        __syncthreads();
        double mine = 0.0;  // lane j < m: the wave's sum over its directions of |A_j|^2
        for (int i = 0; i < 64; i++) {
            const double thi = dirs[w][0][i], phi = dirs[w][1][i];
            const double qv0 = dirs[w][2][i], qv1 = dirs[w][3][i], qv2 = dirs[w][4][i];
            // per plane: theta (the antipode's for layer -1), its row, and (lane p) its spline weights
            int tI[4];
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const int lqi = G.layer - 1 + p;
                const double tp = lqi == -1 ? fmin(fmax(kPi - thi, 0.0), kPi) : thi;
                const int shell = lqi <= 0 ? 1 : lqi;
                const double xt = tp * kInvPi * (double)(3 * shell);
                tI[p] = (int)xt;
                if (kCollapse && lane == p) spline4_weights<T>((T)(xt - (double)tI[p]), wts[w][p]);
            }
            if (kCollapse) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
            cplx<T> acc[M];
#pragma unroll
            for (int j = 0; j < M; j++) acc[j] = {(T)0, (T)0};
            // lanes past the last copy of a chunk repeat it with scale 0
            ZCopyDev zn = zc[min(lane, nz - 1)];
            for (int c0 = 0; c0 < nz; c0 += 64) {
                const int last = min(63, nz - 1 - c0);
                const ZCopyDev z = zn;
                if (c0 + 64 < nz) zn = zc[min(c0 + 64 + lane, nz - 1)];
                const T sc = lane <= last ? (T)z.scale : (T)0;
                double nph = phi - z.alpha;
                if (nph < 0.0) nph += k2Pi;
                cplx<T> amps[4];
                if (kCollapse) {
                    const int leaf0 = __builtin_amdgcn_readfirstlane(z.leaf);
                    bool all_fit = __builtin_amdgcn_readlane(z.leaf, last) == leaf0;
                    int off[4], kl[4], nseg[4];
                    T tph[4];
                    // each plane's segment: from the last copy's node (largest alpha)
                    // forward to the first copy's node + 1, cyclically
#pragma unroll
                    for (int p = 0; p < 4; p++) {
                        const int lqi = G.layer - 1 + p;
                        const int shell = lqi <= 0 ? 1 : lqi;
                        const int P = 6 * shell;
                        double pp = nph;
                        if (lqi < 0) {  // antipode(): phi + pi, wrapped
                            pp = nph + kPi;
                            if (pp >= k2Pi) pp = pp - (int)(pp / k2Pi) * k2Pi;
                        }
                        const double xp = (pp * kInv2Pi) * (double)P;
                        int pi = (int)xp;
                        tph[p] = (T)(xp - (double)pi);
                        pi = (pi == P) ? 0 : pi;
                        const int kf = __builtin_amdgcn_readfirstlane(pi);
                        kl[p] = __builtin_amdgcn_readlane(pi, last);
                        int span = kf - kl[p];
                        if (span < 0) span += P;
                        int o = pi - kl[p];
                        if (o < 0) o += P;
                        off[p] = o;
                        nseg[p] = lqi == 0 ? 0 : span + 2;
                        if (lqi != 0) all_fit = all_fit && span + 2 <= kZWin && __ballot(o > span) == 0;
                    }
                    if (all_fit) {
                        const T4 *g0 = grids[leaf0];
                        // two planes at a time: their 8 row loads issued together, then
                        // the theta spline of each segment node into LDS
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            T4 nd[2][4];
#pragma unroll
                            for (int e = 0; e < 2; e++) {
                                const int p = 2 * h + e;
                                const int lqi = G.layer - 1 + p;
                                const int shell = lqi <= 0 ? 1 : lqi;
                                const int P = 6 * shell, half = 3 * shell, thePoints = 3 * shell;
                                // this lane's segment node (a valid node for lanes past the segment)
                                const bool mine_node = lane < nseg[p];
                                int k = kl[p] + lane;
                                if (k >= P) k -= P;
                                const T4 *plane = g0 + shell_base(shell);
#pragma unroll
                                for (int r = 0; r < 4; r++) {
                                    const int vr = tI[p] + r - 1;
                                    int pos;
                                    if (vr < 0 || vr > thePoints) {
                                        const int theInd = vr < 0 ? vr + thePoints + 1 : vr - (thePoints + 1);
                                        pos = P * theInd + k + ((2 * k >= P) ? -half : half);
                                    } else {
                                        pos = P * vr + k;
                                    }
                                    nd[e][r] = plane[mine_node ? pos : 0];
                                }
                            }
#pragma unroll
                            for (int e = 0; e < 2; e++) {
                                const int p = 2 * h + e;
                                if (lane < nseg[p]) {
                                    T wt[4];
#pragma unroll
                                    for (int r = 0; r < 4; r++) wt[r] = wts[w][p][r];
                                    T4 cn;
                                    cn.x = wt[0] * nd[e][0].x;
                                    cn.y = wt[0] * nd[e][0].y;
                                    cn.z = wt[0] * nd[e][0].z;
                                    cn.w = wt[0] * nd[e][0].w;
#pragma unroll
                                    for (int r = 1; r < 4; r++) {
                                        cn.x += wt[r] * nd[e][r].x;
                                        cn.y += wt[r] * nd[e][r].y;
                                        cn.z += wt[r] * nd[e][r].z;
                                        cn.w += wt[r] * nd[e][r].w;
                                    }
                                    win[w][p][lane] = cn;
                                }
                            }
                            __builtin_amdgcn_wave_barrier();
                        }
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                        __builtin_amdgcn_wave_barrier();
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                        for (int p = 0; p < 4; p++) {
                            if (nseg[p] == 0) {
                                const T4 o = g0[0];
                                amps[p] = {o.x, o.y};
                            } else {
                                const T4 A = win[w][p][off[p]], B = win[w][p][off[p] + 1];
                                amps[p] = hermite<T>({A.x, A.y}, {B.x, B.y}, {A.z, A.w}, {B.z, B.w}, tph[p]);
                            }
                        }
                    } else {
                        direct_planes_call<T, T4>(grids[z.leaf], G.layer, thi, nph, amps);
                    }
                } else {
                    direct_planes<T, T4>(grids[z.leaf], G.layer, thi, nph, amps);
                }
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    amps[p].x *= sc;
                    amps[p].y *= sc;
                }
                const double dot = z.t[0] * qv0 + z.t[1] * qv1 + z.t[2] * qv2;
#pragma unroll
                for (int j = 0; j < M; j++) {
                    if (j < m) {
                        const T w0 = wq[j][0], w1 = wq[j][1], w2 = wq[j][2], w3 = wq[j][3];
                        const T ax = w0 * amps[0].x + w1 * amps[1].x + w2 * amps[2].x + w3 * amps[3].x;
                        const T ay = w0 * amps[0].y + w1 * amps[1].y + w2 * amps[2].y + w3 * amps[3].y;
                        T s, co;
                        phase_sincos<T>(q[j] * dot, s, co);
                        acc[j].x += ax * co - ay * s;
                        acc[j].y += ay * co + ax * s;
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < M; j++) {
                if (j < m) {
                    const double ax = (double)wave_total(acc[j].x), ay = (double)wave_total(acc[j].y);
                    if (lane == j) mine += ax * ax + ay * ay;
                }
            }
        }
        if (lane < m) red[w][lane] = mine;
        __syncthreads();
        if (threadIdx.x < m) {
            const int j = threadIdx.x;
            partial[((size_t)gi * nblk + blockIdx.x) * mstride + jb + j] =
                red[0][j] + red[1][j] + red[2][j] + red[3][j];
        }
        __syncthreads();
    }
}

// group_sums for FP32: the sum over the wave of value lane / (64 / M)
template <int M>
__device__ __forceinline__ float wave_sums(const float (&v)[M], int lane, int o = 32) {
    if constexpr (M > 1) {
        const bool hi = lane & o;
        float u[M / 2];
#pragma unroll
        for (int i = 0; i < M / 2; i++) {
            const float send = hi ? v[i] : v[i + M / 2], keep = hi ? v[i + M / 2] : v[i];
            u[i] = keep + __shfl_xor(send, o, 64);
        }
        return wave_sums<M / 2>(u, lane, o >> 1);
    } else {
        float t = v[0];
        for (; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
        return t;
    }
}

// The same average where the copies are many for the rows' length: every chunk of 64 copies of
// mc_zcopy_kernel collapses its own segment, and together they collapse each node several
// times.  Here a workgroup takes one direction at a time: its 256 threads apply the theta
// spline to the four planes' whole rows (coalesced, the row numbers and weights
// wave-uniform) into LDS, then a thread per copy takes two collapsed nodes per plane, the q
// weights and its translation's phases.  Both halves run without a chain from one chunk to
// the next.  Two barriers a direction; three workgroups per CU cover them.
// 1,000 copies, grid 200, 800 q, 65,536 directions: 158.9 -> 78.3 ms; VALU issue 0.86 of the
// clocks at three waves per SIMD, 381 instructions counted per 64 copies.
// Taken where the rows fit (kRowNodes) and copies >= 2.5 shells: the rows cost 4 * 6 shell
// / 64 collapses of 35 instructions (42 of the 381 here), a chunk of 64 copies 340 beside
// them and 684 there, equal near 2.4 copies per shell.
template <int M>
__global__ __launch_bounds__(256, M <= 8 ? 3 : 2) void mc_zrows_kernel(
    const float4 *const *__restrict__ grids, const ZCopyDev *__restrict__ zc, int nz,
    const GroupDev *__restrict__ groups, const int *__restrict__ active, int mstride,
    const double *__restrict__ qs, double step, uint64_t seed, long long dir0, int nblk, int chunk, int nu, int nv,
    double *__restrict__ partial) {
    const int gi = blockIdx.y;
    const GroupDev G = groups[active[gi]];
    if (!whole_rows(G.layer, nz)) return;
    __shared__ float4 rows[kRowNodes];
    __shared__ double dirs[5][256];
    __shared__ float wq[M][4];
    __shared__ double qt[M];
    __shared__ float red[4][2 * M];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    {
        const long long d = dir0 + (long long)blockIdx.x * blockDim.x + threadIdx.x;
        double u, v;
        uniform_pair(seed, (uint32_t)d, (uint32_t)(d >> 32), (uint32_t)G.layer, kStreamMC, u, v);
        mc_stratify(d, chunk, nu, nv, u, v);
        const double th = acos(2.0 * u - 1.0), ph = k2Pi * v;
        double st, ct, sp, cp;
        sincos(th, &st, &ct);
        sincos(ph, &sp, &cp);
        dirs[0][threadIdx.x] = th * kInvPi;
        dirs[1][threadIdx.x] = ph;
        dirs[2][threadIdx.x] = cp * st;
        dirs[3][threadIdx.x] = sp * st;
        dirs[4][threadIdx.x] = ct;
    }
    int n[4], base[4];
    {
        int b = 0;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            n[p] = 6 * max(G.layer - 1 + p, 1);
            base[p] = b;
            b += n[p] + 1;
        }
    }
    for (int jb = 0; jb < G.m; jb += M) {
        const int m = min(M, G.m - jb);
        const double *q = qs + G.q0 + jb;
        __syncthreads();
        if (threadIdx.x < M) {
            if (threadIdx.x < m) q_weights<float>((q[threadIdx.x] - G.layer * step) * (1.0 / step), wq[threadIdx.x]);
            qt[threadIdx.x] = threadIdx.x < m ? q[threadIdx.x] * kInv2Pi : 0.0;
        }
        __syncthreads();
        double mine = 0.0;  // thread j < m: the sum over the directions of |A_j|^2
        for (int i = 0; i < 256; i++) {
            const double phi = dirs[1][i];
            // lane p of every four: plane p's row and theta weights (the antipode's for plane -1)
            int t0;
            float wt[4];
            {
                const int p = lane & 3, lqi = G.layer - 1 + p;
                const double ut = lqi < 0 ? 1.0 - dirs[0][i] : dirs[0][i];
                spline4_weights<float>((float)cell_of(ut * (double)(3 * max(lqi, 1)), t0), wt);
                t0 = max(t0, 0);
            }
            float acc[2 * M];
#pragma unroll
            for (int j = 0; j < 2 * M; j++) acc[j] = 0.f;
            for (int k0 = 0, k1; k0 < nz; k0 = k1) {
                k1 = zc[k0].run;
                const float4 *g0 = grids[zc[k0].leaf];
                if (k0 > 0) __syncthreads();  // the previous leaf's copies are done with the rows
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    const int lqi = G.layer - 1 + p;
                    if (lqi == 0) continue;
                    const int half = n[p] >> 1, tp = __builtin_amdgcn_readlane(t0, p);
                    float wp[4];
                    const float4 *row[4];
                    bool past[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        wp[r] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wt[r]), p));
                        int v = tp + r - 1;
                        past[r] = v < 0 || v > half;  // past a pole: the other side's row, half a turn away
                        if (past[r]) v = v < 0 ? v + half + 1 : v - (half + 1);
                        row[r] = g0 + shell_base(max(lqi, 1)) + v * n[p];
                    }
                    for (int k = threadIdx.x; k < n[p]; k += 256) {
                        const int kh = k >= half ? k - half : k + half;
                        float4 a[4];
#pragma unroll
                        for (int r = 0; r < 4; r++) a[r] = row[r][past[r] ? kh : k];
                        float4 c;
                        c.x = wp[0] * a[0].x + wp[1] * a[1].x + wp[2] * a[2].x + wp[3] * a[3].x;
                        c.y = wp[0] * a[0].y + wp[1] * a[1].y + wp[2] * a[2].y + wp[3] * a[3].y;
                        c.z = wp[0] * a[0].z + wp[1] * a[1].z + wp[2] * a[2].z + wp[3] * a[3].z;
                        c.w = wp[0] * a[0].w + wp[1] * a[1].w + wp[2] * a[2].w + wp[3] * a[3].w;
                        rows[base[p] + k] = c;
                        if (k == 0) rows[base[p] + n[p]] = c;
                    }
                }
                __syncthreads();
                for (int k = k0 + threadIdx.x; k < k1; k += 256) {
                    const ZCopyDev z = zc[k];
                    double up = (phi - z.alpha) * kInv2Pi;
                    up += up < 0.0 ? 1.0 : 0.0;
                    // below a whole turn by less than FP32 sees, so that no cell lies past the row's end
                    constexpr double kTurn = 1.0 - 1e-11;
                    up = fmin(up, kTurn);
                    const float sc = (float)z.scale;
                    cplx<float> amps[4];
#pragma unroll
                    for (int p = 0; p < 4; p++) {
                        const int lqi = G.layer - 1 + p;
                        if (lqi == 0) {
                            const float4 o = g0[0];
                            amps[p] = {o.x * sc, o.y * sc};
                            continue;
                        }
                        const double u = lqi < 0 ? (up >= 0.5 ? up - 0.5 : fmin(up + 0.5, kTurn)) : up;
                        int c;
                        const float t = (float)cell_of(u * (double)n[p], c);
                        const float4 A = rows[base[p] + c], B = rows[base[p] + c + 1];
                        const float t2 = t * t, t3 = t2 * t;
                        const float h01 = 3.f * t2 - 2.f * t3, h00 = 1.f - h01, h11 = t3 - t2, h10 = h11 - t2 + t;
                        amps[p] = {sc * (h00 * A.x + h01 * B.x + h10 * A.z + h11 * B.z),
                                   sc * (h00 * A.y + h01 * B.y + h10 * A.w + h11 * B.w)};
                    }
                    const double dot = z.t[0] * dirs[2][i] + z.t[1] * dirs[3][i] + z.t[2] * dirs[4][i];
#pragma unroll
                    for (int j = 0; j < M; j++) {
                        if (j < m) {
                            const float ax = wq[j][0] * amps[0].x + wq[j][1] * amps[1].x + wq[j][2] * amps[2].x + wq[j][3] * amps[3].x;
                            const float ay = wq[j][0] * amps[0].y + wq[j][1] * amps[1].y + wq[j][2] * amps[2].y + wq[j][3] * amps[3].y;
                            const float f = (float)__builtin_amdgcn_fract(qt[j] * dot);
                            const float s = __builtin_amdgcn_sinf(f), co = __builtin_amdgcn_cosf(f);
                            acc[j] += ax * co - ay * s;
                            acc[M + j] += ay * co + ax * s;
                        }
                    }
                }
            }
            const float t = wave_sums<2 * M>(acc, lane);
            if (lane % (64 / (2 * M)) == 0) red[w][lane / (64 / (2 * M))] = t;
            __syncthreads();
            if (threadIdx.x < m) {
                const int j = threadIdx.x;
                const double ax = ((double)red[0][j] + (double)red[1][j]) + ((double)red[2][j] + (double)red[3][j]);
                const double ay = ((double)red[0][M + j] + (double)red[1][M + j]) + ((double)red[2][M + j] + (double)red[3][M + j]);
                mine += ax * ax + ay * ay;
            }
        }
        if (threadIdx.x < m) partial[((size_t)gi * nblk + blockIdx.x) * mstride + jb + threadIdx.x] = mine;
    }
}

// ------------------------------------------------------------------ gather ceiling
// The node reads of the mixed MC average without its arithmetic: for every
// (direction, layer) of an MC launch (the same stratified Philox directions) and
// every rotation, the 4 planes x 4 theta rows x 2 phi nodes of the lookup
// (plane_lookup's cells; the antipode / origin planes of layers 0 and 1 read
// shell 1) are loaded and summed, and each wave writes one float.  The rotated
// directions' angles are formed in FP32.  With few registers it runs at full
// occupancy, so its rate is the ceiling of these gathers on the device.
__device__ __forceinline__ void plane_gather(const float4 *__restrict__ plane, int shell, float ut, float up,
                                             float4 &acc) {
    const int phiPoints = 6 * shell, thePoints = 3 * shell;
    const int tI = (int)(ut * (float)thePoints);
    int pI = (int)(up * (float)phiPoints);
    pI = (pI >= phiPoints) ? 0 : pI;
    const int pI1 = (pI + 1 == phiPoints) ? 0 : pI + 1;
    const int half = phiPoints / 2;
#pragma unroll
    for (int rl = -1; rl < 3; rl++) {
        const int v = tI + rl;
        int pos1, pos2;
        if (v < 0 || v > thePoints) {
            const int theInd = v < 0 ? v + thePoints + 1 : v - (thePoints + 1);
            pos1 = phiPoints * theInd + pI + ((2 * pI >= phiPoints) ? -half : half);
            pos2 = phiPoints * theInd + pI1 + ((2 * pI1 >= phiPoints) ? -half : half);
        } else {
            pos1 = phiPoints * v + pI;
            pos2 = phiPoints * v + pI1;
        }
        const float4 a = plane[pos1], b = plane[pos2];
        acc.x += a.x + b.x;
        acc.y += a.y + b.y;
        acc.z += a.z + b.z;
        acc.w += a.w + b.w;
    }
}

template <bool kRot>
__global__ __launch_bounds__(256) void gather_probe(const float4 *__restrict__ g, int N,
                                                    const RotDev *__restrict__ rots, int nrot, int layer0,
                                                    uint64_t seed, int chunk, int nu, int nv,
                                                    float *__restrict__ sink) {
    const int layer = layer0 + blockIdx.y;
    const long long d = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    double u, v;
    uniform_pair(seed, (uint32_t)d, (uint32_t)(d >> 32), (uint32_t)layer, kStreamMC, u, v);
    mc_stratify(d, chunk, nu, nv, u, v);
    const float th = acosf((float)(2.0 * u - 1.0)), ph = (float)(k2Pi * v);
    float st, ct, sp, cp;
    sincosf(th, &st, &ct);
    sincosf(ph, &sp, &cp);
    const float qv[3] = {cp * st, sp * st, ct};
    float4 acc = {0.f, 0.f, 0.f, 0.f};
    const int nr = kRot ? nrot : 1;
    for (int r = 0; r < nr; r++) {
        float ut, up;
        if (kRot) {
            const double *m = rots[r].m;
            float rv[3];
#pragma unroll
            for (int i = 0; i < 3; i++)
                rv[i] = (float)m[3 * i] * qv[0] + (float)m[3 * i + 1] * qv[1] + (float)m[3 * i + 2] * qv[2];
            rv[2] = fminf(fmaxf(rv[2], -1.f), 1.f);
            float a = atan2f(rv[1], rv[0]);
            if (a < 0.f) a += (float)k2Pi;
            ut = acosf(rv[2]) * (float)kInvPi;
            up = fminf(a * (float)kInv2Pi, 1.f);
        } else {
            ut = fminf(th * (float)kInvPi, 1.f);
            up = (float)v;
        }
#pragma unroll
        for (int i = -1; i <= 2; i++) {
            const int lq = min(max(layer + i, 1), N);
            plane_gather(g + shell_base(lq), lq, ut, up, acc);
        }
    }
    float t = acc.x + acc.y + acc.z + acc.w;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    if ((threadIdx.x & 63) == 0)
        sink[((size_t)blockIdx.y * gridDim.x + blockIdx.x) * (blockDim.x / 64) + (threadIdx.x >> 6)] = t;
}

// sum the block partials of every active group in a fixed order:
// out[gi * mstride + j]; one wave per q (lane l adds blocks l, l + 64, ... in
// turn, then the wave's fixed shuffle tree), four waves per group
__global__ __launch_bounds__(256) void mc_reduce(const GroupDev *__restrict__ groups, const int *__restrict__ active,
                                                 const double *__restrict__ partial, int nblk, int mstride,
                                                 double *__restrict__ out) {
    const int gi = blockIdx.x;
    const int m = groups[active[gi]].m;
    const int lane = threadIdx.x & 63;
    for (int j = threadIdx.x >> 6; j < m; j += blockDim.x >> 6) {
        double s = 0.0;
        for (int b = lane; b < nblk; b += 64) s += partial[((size_t)gi * nblk + b) * mstride + j];
        s = wave_sum(s);
        if (lane == 0) out[(size_t)gi * mstride + j] = s;
    }
}

// intensity of every q from the group sums of a fixed-count MC average:
// I[q0 + j] = out[gi * mstride + j] / total (one block per group)
__global__ void mc_finish(const GroupDev *__restrict__ groups, int mstride, const double *__restrict__ out,
                          double total, double *__restrict__ I) {
    const GroupDev g = groups[blockIdx.x];
    for (int j = threadIdx.x; j < g.m; j += blockDim.x) I[g.q0 + j] = out[(size_t)blockIdx.x * mstride + j] / total;
}

// chi^2 = sum_q ((scale * I_q + constant - y_q) / sigma_q)^2 in one block, in a
// fixed summation order; q with sigma <= 0 are skipped
__global__ __launch_bounds__(1024) void chi2_kernel(const double *__restrict__ I, const double *__restrict__ y,
                                                    const double *__restrict__ sig, int n, double scale,
                                                    double constant, double *__restrict__ chi2) {
    __shared__ double part[1024];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const double sg = sig[i];
        if (sg > 0.0) {
            const double r = (scale * I[i] + constant - y[i]) / sg;
            acc = fma(r, r, acc);
        }
    }
    part[threadIdx.x] = acc;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *chi2 = part[0];
}

void launch_mc_finish(const GroupDev *groups, int ngroups, int mstride, const double *out, double total, double *I,
                      hipStream_t s) {
    mc_finish<<<ngroups, 64, 0, s>>>(groups, mstride, out, total, I);
}

void launch_chi2(const double *I, const double *y, const double *sig, int n, double scale, double constant,
                 double *chi2, hipStream_t s) {
    chi2_kernel<<<1, 1024, 0, s>>>(I, y, sig, n, scale, constant, chi2);
}

// the same with (scale, constant) read from device memory, for captured graphs
// whose fit parameters change between replays
__global__ __launch_bounds__(1024) void chi2_param_kernel(const double *__restrict__ I, const double *__restrict__ y,
                                                          const double *__restrict__ sig, int n,
                                                          const double *__restrict__ sc, double *__restrict__ chi2) {
    __shared__ double part[1024];
    const double scale = sc[0], constant = sc[1];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const double sg = sig[i];
        if (sg > 0.0) {
            const double r = (scale * I[i] + constant - y[i]) / sg;
            acc = fma(r, r, acc);
        }
    }
    part[threadIdx.x] = acc;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *chi2 = part[0];
}

void launch_chi2_param(const double *I, const double *y, const double *sig, int n, const double *scale_constant,
                       double *chi2, hipStream_t s) {
    chi2_param_kernel<<<1, 1024, 0, s>>>(I, y, sig, n, scale_constant, chi2);
}

// ------------------------------------------------------------------ VEGAS
constexpr int kVM = 8;         // q-values per pass in the VEGAS kernels
constexpr int kVPts = 4;       // points per lane and bin: points per bin <= 256

// bounds[g*66 + 0..32] theta-axis boundaries in u = (1-cos)/2, [33..65] phi-axis in phi/2pi.
// A bin is served by L lanes (L a power of two, ppb <= kVPts L), a wave by 64 / L
// bins: lane l of the wave takes the points l % L + L k of bin slot l / L.  It
// writes binsum[(gi * mstride + j) * 1024 + bin] = sum over the bin's points of
// I_j and binvar[gi * 1024 + bin] = ppb * sum_p (vol * S_p - mean)^2 with
// S_p = sum_j I_j(p) (HybridVEGASBinReduceToIKernel / HybridVEGASBinReduceKernel,
// HybridOA.cu:300-449).
__device__ __forceinline__ double lanes_sum(double v, int L) {
    for (int o = L >> 1; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// kL: lanes per bin fixed at compile time, or 0 for L; kTiled: a single leaf with L >= 8
template <typename T, typename T4, int kL, bool kSingle, int kP, bool kTiled>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 2 : 1) void vegas_sample(const T4 *const *__restrict__ grids,
                                                    const RotDev *__restrict__ rots, int nrot,
                                                    const double4 *__restrict__ trans,
                                                    const GroupDev *__restrict__ groups,
                                                    const int *__restrict__ active, int mstride,
                                                    const double *__restrict__ qs, double step,
                                                    uint64_t seed, int iter, int ppb, int Lrt,
                                                    const double *__restrict__ bounds,
                                                    double *__restrict__ binsum,
                                                    double *__restrict__ binvar) {
    const int L = kL > 0 ? kL : Lrt;
    const int gi = blockIdx.y;
    const int g = active[gi];
    const GroupDev G = groups[g];
    const int lane = threadIdx.x & 63, pl = lane & (L - 1);
    // every bin of the launch exists: 1024 is a multiple of the 4 (64 / L) bins of a block
    const int bin = (blockIdx.x * 4 + (threadIdx.x >> 6)) * (64 / L) + lane / L;
    const int ti = bin / kVB, pj = bin % kVB;
    const double *bt = bounds + (size_t)g * 66, *bp = bt + 33;
    const double vol = (bt[ti + 1] - bt[ti]) * (bp[pj + 1] - bp[pj]);
    double qv[kP][3];
    double so[kP];
#pragma unroll
    for (int k = 0; k < kP; k++) {
        so[k] = 0.0;
        const int p = pl + L * k;
        double u = 0.5, v = 0.5;
        if (p < ppb) uniform_pair(seed, (uint32_t)(bin * ppb + p), (uint32_t)iter, (uint32_t)G.layer, kStreamVegas, u, v);
        u = u * (bt[ti + 1] - bt[ti]) + bt[ti];
        const double ph = (v * (bp[pj + 1] - bp[pj]) + bp[pj]) * 2. * kPi;
        if (kSingle) {  // the lookup takes theta / pi and phi / 2 pi (u runs from the other pole than MC's)
            qv[k][0] = polar_fraction<T>(1. - u);
            qv[k][1] = ph * kInv2Pi;
            qv[k][2] = 0.0;
        } else {
            const double th = acos(1. - 2. * u);
            double st, ct, sp, cp;
            sincos(th, &st, &ct);
            sincos(ph, &sp, &cp);
            qv[k][0] = cp * st;
            qv[k][1] = sp * st;
            qv[k][2] = ct;
        }
    }
    // single leaf: each point's lookup (four planes) once, held for every q chunk of the
    // group.  A workgroup's bins are neighbours in phi on one theta row of bins (L >= 8), so
    // where that patch's nodes are fewer than half the points' node reads they are staged
    // as a tile (grid 250, 98 points a bin: 556 -> 403 us an iteration; FP64, grid 120, 24
    // points: 143 -> 118; fewer than 8 lanes a bin, or tiles of more nodes, gained nothing);
    // else the points look up in the grid, in a rolled loop, one lookup in flight
    // (unrolled, their gathers would be interleaved past the register budget), their
    // results kept by selection.
    cplx<T> hold[kP][4];
    __shared__ T4 tile[kTiled ? tile_nodes<T4>() : 1];
    __shared__ T wq[kVM][4];
    if (kSingle) {
        const T4 *grid = grids[rots[0].leaf];
        const int nb = 256 / L, b0 = blockIdx.x * nb, r0 = b0 / kVB, q0 = b0 % kVB;
        Tile mine{};
        if (kTiled)
            mine = patch_tile(max(G.layer - 1 + (lane & 3), 1), polar_fraction<float>(1. - bt[r0]),
                              polar_fraction<float>(1. - bt[r0 + 1]), bp[q0], bp[q0 + nb]);
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const int lqi = G.layer - 1 + p;
            const Tile t = tile_of(mine, p);
            if (kTiled && lqi > 0 && t.nodes() <= tile_nodes<T4>() && t.nodes() < 4 * ppb * nb) {  // uniform
                if (p > 0) __syncthreads();
                stage_tile(grid + shell_base(lqi), lqi, t, tile);
                __syncthreads();
#pragma unroll
                for (int k = 0; k < kP; k++)
                    if (pl + L * k < ppb) hold[k][p] = tile_lookup<T, T4>(tile, t, lqi, qv[k][0], qv[k][1]);
            } else {
#pragma unroll 1
                for (int k = 0; k < kP; k++) {
                    if (pl + L * k >= ppb) break;
                    double ut = qv[0][0], up = qv[0][1];
#pragma unroll
                    for (int kk = 1; kk < kP; kk++)
                        if (kk == k) {
                            ut = qv[kk][0];
                            up = qv[kk][1];
                        }
                    const cplx<T> a = plane_direct<T, T4>(grid, lqi, ut, up);
#pragma unroll
                    for (int kk = 0; kk < kP; kk++)
                        if (kk == k) hold[kk][p] = a;
                }
            }
        }
    }
    for (int jb = 0; jb < G.m; jb += kVM) {
        const int m = min(kVM, G.m - jb);
        double e[kVM];
#pragma unroll
        for (int j = 0; j < kVM; j++) e[j] = 0.0;
        // the q's weights over the planes, shared by every point
        __syncthreads();
        if (threadIdx.x < m) q_weights<T>((qs[G.q0 + jb + threadIdx.x] - G.layer * step) * (1.0 / step), wq[threadIdx.x]);
        __syncthreads();
        if (kSingle) {
            const double sc2 = (double)(T)rots[0].scale * (double)(T)rots[0].scale;
#pragma unroll
            for (int j = 0; j < kVM; j++) {
                if (j >= m) continue;
                const T w0 = wq[j][0], w1 = wq[j][1], w2 = wq[j][2], w3 = wq[j][3];
#pragma unroll
                for (int k = 0; k < kP; k++) {
                    if (pl + L * k >= ppb) continue;
                    const T ax = w0 * hold[k][0].x + w1 * hold[k][1].x + w2 * hold[k][2].x + w3 * hold[k][3].x;
                    const T ay = w0 * hold[k][0].y + w1 * hold[k][1].y + w2 * hold[k][2].y + w3 * hold[k][3].y;
                    const double I = sc2 * ((double)ax * (double)ax + (double)ay * (double)ay);
                    e[j] += I;
                    so[k] += I;
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < kP; k++) {
                if (pl + L * k >= ppb) continue;
                cplx<T> acc[kVM];
#pragma unroll
                for (int j = 0; j < kVM; j++) acc[j] = {(T)0, (T)0};
                docked_amplitude<T, T4, kVM>(grids, rots, nrot, trans, G.layer, qv[k], qs + G.q0 + jb, wq, m,
                                             G.uniform != 0, acc);
#pragma unroll
                for (int j = 0; j < kVM; j++) {
                    const double I = (double)acc[j].x * (double)acc[j].x + (double)acc[j].y * (double)acc[j].y;
                    if (j < m) {
                        e[j] += I;
                        so[k] += I;
                    }
                }
            }
        }
        if (kTiled || kL == 64) {  // L >= 8
            const double t = group_sums<kVM>(e, lane, L);
            const int lj = L / kVM, j = pl / lj;
            if (pl % lj == 0 && j < m) binsum[((size_t)gi * mstride + jb + j) * (kVB * kVB) + bin] = t;
        } else {
#pragma unroll
            for (int j = 0; j < kVM; j++) {
                const double t = lanes_sum(e[j], L);
                if (pl == 0 && j < m) binsum[((size_t)gi * mstride + jb + j) * (kVB * kVB) + bin] = t;
            }
        }
    }
    // variance of vol * S over the bin's points, two-pass (equal to the reference's Welford sum)
    double sx = 0.0;
#pragma unroll
    for (int k = 0; k < kP; k++)
        if (pl + L * k < ppb) sx += vol * so[k];
    const double mean = lanes_sum(sx, L) / (double)ppb;
    double sq = 0.0;
#pragma unroll
    for (int k = 0; k < kP; k++)
        if (pl + L * k < ppb) sq += (vol * so[k] - mean) * (vol * so[k] - mean);
    sq = lanes_sum(sq, L);
    if (pl == 0) binvar[(size_t)gi * (kVB * kVB) + bin] = sq * ppb;
}

// damped re-binning weight (HybridOA.cu:181-263) of x = total / (local mean of the
// variances): ((x - 1) / (x ln x))^1.5, 0 where that is no number
__device__ __forceinline__ double vegas_weight(double x) {
    const double y = (x - 1.) / (x * log(x));
    const double w = y * sqrt(y);
    return w != w ? 0. : w;
}

// The re-binning of one axis by a half wave (lane i of 32 holds weight w_i and the bin
// [b_i, b_i+1]): new interior boundaries at equal shares of the weights (vegas_boundary);
// boundaries that no sum reaches keep their value.  lane i returns boundary i + 1 (of 32; the
// last stays).  Every lane adds the weights in bin order, from LDS: a scan across the lanes adds
// each running sum in another order, and a bin of weight 0 then starts or ends above its
// neighbour's sum.
__device__ __forceinline__ double vegas_rebin(double w, double lo, double hi, int i, double *cum, double *wt, double *edge) {
    const double first = __shfl(lo, 0, kVB);
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    wt[i] = w;
    edge[i] = hi;
    wave_sync();
    double c = 0.0, mine = 0.0;
#pragma unroll
    for (int k = 0; k < kVB; k++) {
        c += wt[k];
        if (k == i) mine = c;
    }
    cum[i] = mine;
    wave_sync();
    return i == kVB - 1 ? hi : vegas_boundary(wt, cum, edge, first, i + 1, hi);
}

// one block (1024 threads = the 32x32 bins) per active group: the iteration's
// integral sum_bins vol * mean_bin(I_j) (q dealt over waves 1 to 15 first), the
// theta/phi marginals of the bin variances, re-binning, and the running mean over iterations
// (HybridVEGASResizeGridKernel; GPUHybridCalc.cu:654-701).  The re-binning runs on one wave,
// an axis per half wave, by running sums and a binary search: 16.5 -> 5.8 us an iteration (its 64
// serial steps waited on LDS).
// hist[iter * nq + q] holds the running mean after iteration iter.
__global__ __launch_bounds__(1024) void vegas_reduce(const GroupDev *__restrict__ groups,
                                                     const int *__restrict__ active, int mstride,
                                                     int ppb, int iter, const double *__restrict__ binsum,
                                                     const double *__restrict__ binvar,
                                                     double *__restrict__ bounds,
                                                     double *__restrict__ hist, int nq) {
    const int gi = blockIdx.x;
    const int g = active[gi];
    const GroupDev G = groups[g];
    const int bin = threadIdx.x, ti = bin / kVB, pj = bin % kVB;
    double *bt = bounds + (size_t)g * 66, *bp = bt + 33;
    __shared__ double sv[kVB][kVB + 1];
    __shared__ double svol[1024];
    __shared__ double cum[2][kVB], wt[2][kVB], edge[2][kVB];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    sv[ti][pj] = binvar[(size_t)gi * 1024 + bin];
    svol[bin] = (bt[ti + 1] - bt[ti]) * (bp[pj + 1] - bp[pj]) / (double)ppb;
    // wave 0, half wave ax: axis ax, lane i its bin i
    const int ax = lane / kVB, i = lane % kVB;
    const double *b = ax == 0 ? bt : bp;
    double lo = 0.0, hi = 0.0;
    if (w == 0) {
        lo = b[i];
        hi = b[i + 1];
    }
    __syncthreads();  // every boundary is read above before any is rewritten below
    if (w == 0) {
        double a = 0.0;
#pragma unroll 8
        for (int k = 0; k < kVB; k++) a += ax == 0 ? sv[i][k] : sv[k][i];
        double total = a;
#pragma unroll
        for (int d = kVB / 2; d > 0; d >>= 1) total += __shfl_xor(total, d, kVB);
        const double before = __shfl_up(a, 1, kVB), after = __shfl_down(a, 1, kVB);
        const double local = i == 0 ? (a + after) / 2. : i == kVB - 1 ? (a + before) / 2. : (before + a + after) / 3.;
        const double wgt = total == 0. ? 0. : vegas_weight(total / local);
        const double nb = vegas_rebin(wgt, lo, hi, i, cum[ax], wt[ax], edge[ax]);
        if (total != 0.) (ax == 0 ? bt : bp)[i + 1] = nb;
    }
    // the integrals: wave w takes q = w - 1, w + 15, ... (wave 0 re-bins meanwhile, and joins
    // where it is done first)
    for (int j = w == 0 ? 15 : w - 1; j < G.m; j += 16) {
        const double *bs = binsum + ((size_t)gi * mstride + j) * 1024;
        double c = 0.0;
#pragma unroll
        for (int k = 0; k < 16; k++) c += bs[lane + 64 * k] * svol[lane + 64 * k];
        c = wave_sum(c);
        if (lane == 0) {
            const int q = G.q0 + j;
            double e = c;
            if (iter > 0) e = (hist[(size_t)(iter - 1) * nq + q] * (double)iter + e) / (double)(iter + 1);
            hist[(size_t)iter * nq + q] = e;
        }
    }
}

// ------------------------------------------------------------------ single points
// GetSphr (Grid.cpp:487-548): the CPU-path lookup used by getAmplitude and GK
template <typename T, typename T4>
__device__ __forceinline__ cplx<T> get_sphr(const T4 *__restrict__ g, int N, double step, double rr, double ut,
                                            double up) {  // theta = pi ut, phi = 2 pi up
    const T4 o = g[0];
    if (rr == 0.0) return {o.x, o.y};
    double frc = rr / step;
    frc = __longlong_as_double(__double_as_longlong(frc) + 8);
    const int fInd = (int)frc;
    const double frac = frc - (double)fInd;
    cplx<T> p[4];
    p[1] = fInd > 0 ? plane_lookup<T, T4, true>(g + shell_base(fInd), fInd, ut, up) : cplx<T>{o.x, o.y};
    if (frac < 1.e-9) return p[1];
    p[2] = plane_lookup<T, T4, true>(g + shell_base(fInd + 1), fInd + 1, ut, up);
    if (fInd == 0) {
        double nth, nph;
        antipode(ut * kPi, up * k2Pi, nth, nph);
        p[0] = plane_lookup<T, T4, true>(g + 1, 1, nth * kInvPi, nph * kInv2Pi);
    } else if (fInd == 1) {
        p[0] = {o.x, o.y};
    } else {
        p[0] = plane_lookup<T, T4, true>(g + shell_base(fInd - 1), fInd - 1, ut, up);
    }
    p[3] = (fInd + 2 < N) ? plane_lookup<T, T4, true>(g + shell_base(fInd + 2), fInd + 2, ut, up) : p[2];
    cplx<T> d1, d2;
    four_point<T>(p, d1, d2);
    return hermite<T>(p[1], p[2], d1, d2, (T)frac);
}

// GetCart (Grid.cpp:384-392)
template <typename T, typename T4>
__device__ __forceinline__ cplx<T> get_cart(const T4 *__restrict__ g, int N, double step, double x,
                                            double y, double z) {
    double r = sqrt(x * x + y * y + z * z);
    if (fabs(z) > r) r = fabs(z);
    if (r == 0.0) return get_sphr<T, T4>(g, N, step, 0.0, 0.0, 0.0);
    if constexpr (sizeof(T) == 4)
        return get_sphr<T, T4>(g, N, step, r, polar_fraction<T>(0.5 + 0.5 * (z / r)), azimuth_fraction<T>(y, x));
    const double th = acos(z / r);
    double ph = atan2(y, x);
    if (ph < 0.0) ph += k2Pi;
    return get_sphr<T, T4>(g, N, step, r, th * kInvPi, ph * kInv2Pi);
}

// the same for a point of known norm r > 0 (a rotated node or sample), rinv = 1 / r
template <typename T, typename T4>
__device__ __forceinline__ cplx<T> get_turned(const T4 *__restrict__ g, int N, double step, const double v[3], double r,
                                              double rinv) {
    if constexpr (sizeof(T) == 4)
        return get_sphr<T, T4>(g, N, step, r, polar_fraction<T>(0.5 + 0.5 * (v[2] * rinv)),
                               azimuth_fraction<T>(v[1], v[0]));
    return get_cart<T, T4>(g, N, step, v[0], v[1], v[2]);
}

// batch GetSphr at (q, theta, phi) triples
template <typename T, typename T4>
__global__ __launch_bounds__(256) void sphr_batch(const T4 *__restrict__ g, int N, double step, int n,
                           const double *__restrict__ q, const double *__restrict__ th,
                           const double *__restrict__ ph, double2 *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    cplx<T> a = get_sphr<T, T4>(g, N, step, q[i], th[i] * kInvPi, ph[i] * kInv2Pi);
    out[i] = make_double2((double)a.x, (double)a.y);
}

// batch InterpolateThetaPhiPlane (Grid.cpp:61-134): shell ri[i] >= 1 at
// (theta, phi) with the CPU variant's snapping of tiny fractions
template <typename T, typename T4>
__global__ __launch_bounds__(256) void plane_batch(const T4 *__restrict__ g, int n, const int *__restrict__ ri,
                                                   const double *__restrict__ th, const double *__restrict__ ph,
                                                   double2 *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int r = ri[i];
    cplx<T> a = plane_lookup<T, T4, true>(g + shell_base(r), r, th[i] * kInvPi, ph[i] * kInv2Pi);
    out[i] = make_double2((double)a.x, (double)a.y);
}

// |A|^2 of JacobianSphereGrid::CalculateIntensity's samples (Grid.cpp:421-466):
// phi[i] and v2[i] in [0,2), theta = acos(v2-1), lookup through GetCart
template <typename T, typename T4>
__global__ __launch_bounds__(256) void seeded_samples(const T4 *__restrict__ g, int N, double step, double q, long long n,
                               const double *__restrict__ phi, const double *__restrict__ v2,
                               double *__restrict__ out) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double theta = acos(v2[i] - 1.0);
    double st, ct, sp, cp;
    sincos(theta, &st, &ct);
    sincos(phi[i], &sp, &cp);
    cplx<T> a = get_cart<T, T4>(g, N, step, q * st * cp, q * st * sp, q * ct);
    out[i] = (double)a.x * (double)a.x + (double)a.y * (double)a.y;
}

// |A(q)|^2 of docked leaves at cartesian q (Amplitude.cpp:3035-3056 composed
// with Symmetries.cpp:697-716): the integrand of Gauss-Kronrod

template <typename T, typename T4>
__device__ double docked_intensity(const T4 *const *__restrict__ grids, const LeafGeo *__restrict__ geo,
                                   const RotDev *__restrict__ rots, int nrot, const double4 *__restrict__ trans,
                                   const double q[3]) {
    double ax = 0.0, ay = 0.0;
    const double n = sqrt(q[0] * q[0] + q[1] * q[1] + q[2] * q[2]), ninv = 1.0 / n;
    for (int r = 0; r < nrot; r++) {
        const RotDev rd = rots[r];
        double rv[3];
        rotate_t(rd, q, rv);
        const LeafGeo G = geo[rd.leaf];
        const cplx<T> a = n > 0.0 ? get_turned<T, T4>(grids[rd.leaf], G.N, G.step, rv, n, ninv)
                                  : get_sphr<T, T4>(grids[rd.leaf], G.N, G.step, 0.0, 0.0, 0.0);
        double sc = 0.0, ss = 0.0;
        for (int tr = 0; tr < rd.nt; tr++) {
            const double4 t = trans[rd.t0 + tr];
            double s = 0.0, c = 1.0;
            if (t.x != 0.0 || t.y != 0.0 || t.z != 0.0) phase_exact<T>(q[0] * t.x + q[1] * t.y + q[2] * t.z, s, c);
            sc += c;
            ss += s;
        }
        ax += ((double)a.x * sc - (double)a.y * ss) * rd.scale;
        ay += ((double)a.y * sc + (double)a.x * ss) * rd.scale;
    }
    return ax * ax + ay * ay;
}

template <typename T, typename T4>
__global__ __launch_bounds__(256) void docked_cart_batch(const T4 *const *__restrict__ grids, const LeafGeo *__restrict__ geo,
                                  const RotDev *__restrict__ rots, int nrot,
                                  const double4 *__restrict__ trans, int n,
                                  const double *__restrict__ qxyz, double *__restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double q[3] = {qxyz[3 * i], qxyz[3 * i + 1], qxyz[3 * i + 2]};
    out[i] = docked_intensity<T, T4>(grids, geo, rots, nrot, trans, q);
}

// Azimuthal average of the 2-D generate path (DomainModel::CalculateIntensity2DMatrix,
// Amplitude.cpp:843-993): point p = (q sin(theta), q cos(theta)) of the (q_z, q_perp)
// plane; I_p = (1 / nphi) sum_k |A(q, theta, phi_k)|^2 over stratified azimuths
// phi_k = 2 pi (k + u_k) / nphi, u_k from the Philox stream keyed by (seed, k, p).
// The reference draws phi uniformly per (q, theta) point with a per-layer
// mt19937 (AverageIntensitiesBetweenLayers2D, :2825-2897); one stratum per
// sample gives the same expectation with a fraction of the variance.  One block
// per point; the block's sum is formed in a fixed order.
template <typename T, typename T4>
__global__ __launch_bounds__(256) void azimuthal_kernel(const T4 *const *__restrict__ grids,
                                                        const LeafGeo *__restrict__ geo,
                                                        const RotDev *__restrict__ rots, int nrot,
                                                        const double4 *__restrict__ trans,
                                                        const double2 *__restrict__ pts, int nphi, uint64_t seed,
                                                        double *__restrict__ out) {
    __shared__ double red[4];
    const int p = blockIdx.x;
    const double2 pt = pts[p];
    double sum = 0.0;
    for (int k = threadIdx.x; k < nphi; k += blockDim.x) {
        double u, v;
        uniform_pair(seed, (uint32_t)k, (uint32_t)p, 0u, kStreamAzimuth, u, v);
        const double ph = k2Pi * ((double)k + u) / (double)nphi;
        double sp, cp;
        sincos(ph, &sp, &cp);
        const double q[3] = {pt.x * cp, pt.x * sp, pt.y};
        sum += docked_intensity<T, T4>(grids, geo, rots, nrot, trans, q);
    }
    sum = wave_sum(sum);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) out[p] = (red[0] + red[1] + red[2] + red[3]) / (double)nphi;
}

// Gauss-Kronrod phi intervals.  A workgroup of 240 threads evaluates the 15
// points phi = a + b x_k of 16 intervals, then one thread per interval forms
// the Kronrod and Gauss sums
//   kv = sum_k I_k b kw_k,  gv = sum_{k odd} I_k b gw_{k/2}
// in k order with every product and sum rounded as written (no fused
// multiply-add), the arithmetic of DomainModel::GaussLegPhi
// (Amplitude.cpp:1443-1467), so that accept/split decisions follow it.
constexpr int kGkTasksPerBlock = 16;

template <typename T, typename T4>
__device__ __forceinline__ double gk_point(const T4 *const *__restrict__ grids, const LeafGeo *__restrict__ geo,
                                           const RotDev *__restrict__ rots, int nrot,
                                           const double4 *__restrict__ trans, const double4 &tk, double x) {
    const double xi = fma(tk.w, x, tk.z);  // one rounding, whatever the caller forms a and b from
    const double q[3] = {tk.x * cos(xi), tk.x * sin(xi), tk.y};
    return docked_intensity<T, T4>(grids, geo, rots, nrot, trans, q);
}
__device__ __forceinline__ void gk_sums(const double *v, double hw, const GkNodes *__restrict__ nodes, double &kv,
                                        double &gv) {
    kv = gv = 0.0;
    for (int k = 0; k < 15; k++) {
        const double p = __dmul_rn(v[k], hw);
        kv = __dadd_rn(kv, __dmul_rn(p, nodes->kw[k]));
        if (k % 2 == 1) gv = __dadd_rn(gv, __dmul_rn(p, nodes->gw[k / 2]));
    }
}

// the sums of a list of tasks (q sin(theta), q cos(theta), a, b): out[2t] = kv, out[2t + 1] = gv
template <typename T, typename T4>
__global__ __launch_bounds__(15 * kGkTasksPerBlock) void docked_gk_batch(
    const T4 *const *__restrict__ grids, const LeafGeo *__restrict__ geo, const RotDev *__restrict__ rots,
    int nrot, const double4 *__restrict__ trans, long long ntasks, const double4 *__restrict__ tasks,
    const GkNodes *__restrict__ nodes, double *__restrict__ out) {
    __shared__ double val[15 * kGkTasksPerBlock];
    const long long t0 = (long long)blockIdx.x * kGkTasksPerBlock;
    const long long t = t0 + threadIdx.x / 15;
    double I = 0.0;
    if (t < ntasks)
        I = gk_point<T, T4>(grids, geo, rots, nrot, trans, tasks[t], nodes->x[threadIdx.x % 15]);
    val[threadIdx.x] = I;
    __syncthreads();
    const long long ts = t0 + threadIdx.x;
    if (threadIdx.x < kGkTasksPerBlock && ts < ntasks) {
        double kv, gv;
        gk_sums(val + 15 * threadIdx.x, tasks[ts].w, nodes, kv, gv);
        out[2 * ts] = kv;
        out[2 * ts + 1] = gv;
    }
}

// One level of the phi recursion in one launch: a workgroup evaluates 16 open
// intervals, and its first 16 threads accept each or split it at its midpoint
// (two new intervals, their slots from one atomic per workgroup, and a node).
// The accept rule and the midpoint are GaussLegPhi's (Amplitude.cpp:1449-1467).
// An accepted value climbs: the first half of a split leaves its value at the
// node, the second takes it, adds and goes on to the node above; left + right
// either way round is the same sum, and a root's value is its phi integral.  So
// no pass over the trees follows.  The level's length is read from the device
// (the grid covers at most 16 times 4,096 intervals, larger levels go round), so
// several levels are launched without the host waiting for each.  With a launch
// of its own to decide, one more to add up a level and a wait for each count, a
// level of up to 1,000 intervals took 25 us, of which the evaluation is 9: 501
// q at tolerance 1e-3 (36 levels of 60 to 30,000 intervals) 2.28 -> 1.32 ms.
template <typename T, typename T4>
__global__ __launch_bounds__(15 * kGkTasksPerBlock, 2) void docked_gk_level(
    const T4 *const *__restrict__ grids, const LeafGeo *__restrict__ geo, const RotDev *__restrict__ rots,
    int nrot, const double4 *__restrict__ trans, const GkNodes *__restrict__ nodes, GkLevel L) {
    __shared__ double val[15 * kGkTasksPerBlock];
    const int n = L.first ? L.nroots : L.counts[L.level];
    int below = L.before;  // intervals below the roots, this level's among them
    for (int l = 1; l <= L.level; l++) below += L.counts[l];
    if (n > L.cap_int || L.nroots + below > L.cap_nodes) return;  // the host sees the same counts
    for (int t0 = (int)blockIdx.x * kGkTasksPerBlock; t0 < n; t0 += (int)gridDim.x * kGkTasksPerBlock) {
        auto interval = [&](int t) {
            return L.first ? GkInterval{0.0, k2Pi, -1, t} : L.cur[t];
        };
        const int t = t0 + (int)threadIdx.x / 15;
        double I = 0.0;
        if (t < n) {
            const GkInterval iv = interval(t);
            const double2 r = L.roots[iv.root];
            const double4 tk = make_double4(r.x, r.y, __dmul_rn(__dadd_rn(iv.pmax, iv.pmin), 0.5),
                                            __dmul_rn(__dsub_rn(iv.pmax, iv.pmin), 0.5));
            I = gk_point<T, T4>(grids, geo, rots, nrot, trans, tk, nodes->x[threadIdx.x % 15]);
        }
        val[threadIdx.x] = I;
        __syncthreads();
        if (threadIdx.x < 64) {
            const int lane = threadIdx.x, ts = t0 + lane;
            const bool live = lane < kGkTasksPerBlock && ts < n;
            GkInterval iv{0.0, 0.0, -1, 0};
            double kv = 0.0;
            bool accept = false;
            if (live) {
                double gv;
                iv = interval(ts);
                gk_sums(val + 15 * lane, __dmul_rn(__dsub_rn(iv.pmax, iv.pmin), 0.5), nodes, kv, gv);
                accept = L.last || fabs(1.0 - (gv / kv)) <= L.eps || gv == kv;
            }
            const bool split = live && !accept;
            const unsigned long long mask = __ballot(split);
            int w = 0;
            if (mask) {
                if (lane == 0) w = atomicAdd(&L.counts[L.level + 1], 2 * __popcll(mask));
                w = __shfl(w, 0, 64) + 2 * __popcll(mask & ((1ull << lane) - 1ull));
            }
            if (split && w + 2 <= L.cap_int && L.nroots + below + w + 2 <= L.cap_nodes) {
                const int c = (below + w) / 2;
                const double mid = (iv.pmax + iv.pmin) * 0.5;
                L.nodes[c] = GkNode{kGkEmpty, iv.parent, iv.root};
                L.next[w] = GkInterval{iv.pmin, mid, c, iv.root};
                L.next[w + 1] = GkInterval{mid, iv.pmax, c, iv.root};
            }
            if (live && accept) {
                double v = kv;
                int p = iv.parent;
                while (p >= 0) {
                    unsigned long long mine = (unsigned long long)__double_as_longlong(v);
                    if (mine == kGkEmpty) mine = 0x7ff8000000000000ull;
                    const unsigned long long other = atomicExch(&L.nodes[p].mail, mine);
                    if (other == kGkEmpty) break;
                    v = __dadd_rn(v, __longlong_as_double((long long)other));
                    p = L.nodes[p].parent;
                }
                if (p < 0) L.phival[iv.root] = v;
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------ launchers
void launch_mc(bool fp64, bool single, const void *const *grids, const RotDev *rots, int nrot,
               const double4 *trans, const ZCopyDev *zc, int nz, const GroupDev *groups, const int *active,
               int nactive, int mstride, const double *qs, double step, uint64_t seed, long long dir0, int nblk,
               int chunk, double *partial, double *out, hipStream_t s) {
    dim3 grid(nblk, nactive);
    int nu, nv;
    mc_strata(chunk, nu, nv);
    if (!single && zc && nz >= kZCopyMin) {
        // 8 q per pass when no shell group holds more (fewer accumulators);
        // FP32 grids: the whole-row kernel, the collapse instance and the direct one over the
        // same grid, each block running in one of them
#define DPLUS_MCZ(T, T4, C, M, SPLIT)                                                                             \
    mc_zcopy_kernel<T, T4, C, M><<<grid, 256, 0, s>>>((const T4 *const *)grids, zc, nz, groups, active, mstride, \
                                                      qs, step, seed, dir0, nblk, chunk, nu, nv, SPLIT, partial)
        if (fp64 && mstride <= 8) {
            DPLUS_MCZ(double, double4, false, 8, false);
        } else if (fp64) {
            DPLUS_MCZ(double, double4, false, kMaxM, false);
        } else if (mstride <= 8) {
            mc_zrows_kernel<8><<<grid, 256, 0, s>>>((const float4 *const *)grids, zc, nz, groups, active, mstride, qs,
                                                    step, seed, dir0, nblk, chunk, nu, nv, partial);
            DPLUS_MCZ(float, float4, true, 8, true);
            DPLUS_MCZ(float, float4, false, 8, true);
        } else {
            mc_zrows_kernel<kMaxM><<<grid, 256, 0, s>>>((const float4 *const *)grids, zc, nz, groups, active, mstride,
                                                        qs, step, seed, dir0, nblk, chunk, nu, nv, partial);
            DPLUS_MCZ(float, float4, true, kMaxM, true);
            DPLUS_MCZ(float, float4, false, kMaxM, true);
        }
#undef DPLUS_MCZ
        mc_reduce<<<nactive, 256, 0, s>>>(groups, active, partial, nblk, mstride, out);
        return;
    }
    // a single leaf over four chunks or more: by patch (its tile serves every chunk)
    const long long nchunks = (long long)nblk * 256 / chunk;
    if (single && nchunks >= 4) {
        int D, nset;
        mc_patch_sets(nchunks, D, nset);
        const int nb = chunk / 64 * nset;
        if (nb > nblk) throw Error(kErrGeneral, "more workgroups than blocks of partial sums");
        const dim3 pg(nb, nactive);
#define DPLUS_MCP(T, T4, D)                                                                                        \
    mc_patch_kernel<T, T4, D><<<pg, 256, 0, s>>>((const T4 *const *)grids, rots, groups, active, mstride, qs, step, \
                                                 seed, dir0, (int)nchunks, chunk, nu, nv, nset, partial)
        if (fp64) {
            D == 4 ? (void)DPLUS_MCP(double, double4, 4) : D == 2 ? (void)DPLUS_MCP(double, double4, 2) : (void)DPLUS_MCP(double, double4, 1);
        } else {
            D == 4 ? (void)DPLUS_MCP(float, float4, 4) : D == 2 ? (void)DPLUS_MCP(float, float4, 2) : (void)DPLUS_MCP(float, float4, 1);
        }
#undef DPLUS_MCP
        mc_reduce<<<nactive, 256, 0, s>>>(groups, active, partial, nb, mstride, out);
        return;
    }
#define DPLUS_MC(T, T4, S, M)                                                                                      \
    mc_kernel<T, T4, S, M><<<grid, 256, 0, s>>>((const T4 *const *)grids, rots, nrot, trans, groups, active, mstride, \
                                                qs, step, seed, dir0, nblk, chunk, nu, nv, partial)
    if (fp64 && single)
        DPLUS_MC(double, double4, true, kMaxM);
    else if (fp64 && mstride <= 8)
        DPLUS_MC(double, double4, false, 8);
    else if (fp64)
        DPLUS_MC(double, double4, false, kMaxM);
    else if (single)
        DPLUS_MC(float, float4, true, kMaxM);
    else if (mstride <= 8)
        DPLUS_MC(float, float4, false, 8);
    else
        DPLUS_MC(float, float4, false, kMaxM);
#undef DPLUS_MC
    mc_reduce<<<nactive, 256, 0, s>>>(groups, active, partial, nblk, mstride, out);
}

// the gather-ceiling probe over layers [layer0, layer0 + nlayers) of a mixed grid
// with N shells: nblk blocks of 256 directions per layer; sink holds
// nblk * nlayers * 4 floats
void launch_gather_probe(const void *grid, int N, const RotDev *rots, int nrot, int layer0, int nlayers, int nblk,
                         uint64_t seed, int chunk, float *sink, hipStream_t s) {
    int nu, nv;
    mc_strata(chunk, nu, nv);
    dim3 gr(nblk, nlayers);
    if (rots)
        gather_probe<true><<<gr, 256, 0, s>>>((const float4 *)grid, N, rots, nrot, layer0, seed, chunk, nu, nv, sink);
    else
        gather_probe<false><<<gr, 256, 0, s>>>((const float4 *)grid, N, nullptr, 1, layer0, seed, chunk, nu, nv,
                                               sink);
}

void launch_vegas_iter(bool fp64, bool single, const void *const *grids, const RotDev *rots, int nrot,
                       const double4 *trans, const GroupDev *groups, const int *active, int nactive,
                       int mstride, const double *qs, double step, uint64_t seed, int iter, int ppb,
                       double *bounds, double *binsum, double *binvar, double *hist, int nq, hipStream_t s) {
    // lanes per bin: the least power of two >= ppb, at most a wave (ppb <= kVPts * 64)
    int L = 1;
    while (L < ppb && L < 64) L <<= 1;
    dim3 grid(kVB * kVB / (4 * (64 / L)), nactive);
#define DPLUS_VEGAS(T, T4, KL, S, P, TILED)                                                                   \
    vegas_sample<T, T4, KL, S, P, TILED><<<grid, 256, 0, s>>>((const T4 *const *)grids, rots, nrot, trans,       \
                                                              groups, active, mstride, qs, step, seed, iter,    \
                                                              ppb, L, bounds, binsum, binvar)
    // points per lane: the single-leaf instances are sized to the bin's points
    // (fewer registers), the docked ones take up to kVPts
    const int per_lane = (ppb + L - 1) / L;
#define DPLUS_VEGAS_P(T, T4)                             \
    if (!single && L == 64)                              \
        DPLUS_VEGAS(T, T4, 64, false, kVPts, false);     \
    else if (!single)                                    \
        DPLUS_VEGAS(T, T4, 0, false, kVPts, false);      \
    else if (L < 8)                                      \
        DPLUS_VEGAS(T, T4, 0, true, 1, false);           \
    else if (L < 64)                                     \
        DPLUS_VEGAS(T, T4, 0, true, 1, true);            \
    else if (per_lane <= 1)                              \
        DPLUS_VEGAS(T, T4, 64, true, 1, true);           \
    else if (per_lane <= 2)                              \
        DPLUS_VEGAS(T, T4, 64, true, 2, true);           \
    else                                                 \
        DPLUS_VEGAS(T, T4, 64, true, kVPts, true);
    if (fp64) {
        DPLUS_VEGAS_P(double, double4)
    } else {
        DPLUS_VEGAS_P(float, float4)
    }
#undef DPLUS_VEGAS_P
#undef DPLUS_VEGAS
    vegas_reduce<<<nactive, 1024, 0, s>>>(groups, active, mstride, ppb, iter, binsum, binvar, bounds, hist, nq);
}

void launch_sphr_batch(bool fp64, const void *g, int N, double step, int n, const double *q,
                       const double *th, const double *ph, double2 *out, hipStream_t s) {
    unsigned nb = (n + 255) / 256;
    if (fp64)
        sphr_batch<double, double4><<<nb, 256, 0, s>>>((const double4 *)g, N, step, n, q, th, ph, out);
    else
        sphr_batch<float, float4><<<nb, 256, 0, s>>>((const float4 *)g, N, step, n, q, th, ph, out);
}

void launch_plane_batch(bool fp64, const void *g, int n, const int *ri, const double *th, const double *ph,
                        double2 *out, hipStream_t s) {
    unsigned nb = (n + 255) / 256;
    if (fp64)
        plane_batch<double, double4><<<nb, 256, 0, s>>>((const double4 *)g, n, ri, th, ph, out);
    else
        plane_batch<float, float4><<<nb, 256, 0, s>>>((const float4 *)g, n, ri, th, ph, out);
}

void launch_seeded_samples(bool fp64, const void *g, int N, double step, double q, long long n,
                           const double *phi, const double *v2, double *out, hipStream_t s) {
    unsigned nb = (unsigned)((n + 255) / 256);
    if (fp64)
        seeded_samples<double, double4><<<nb, 256, 0, s>>>((const double4 *)g, N, step, q, n, phi, v2, out);
    else
        seeded_samples<float, float4><<<nb, 256, 0, s>>>((const float4 *)g, N, step, q, n, phi, v2, out);
}

void launch_docked_gk(bool fp64, const void *const *grids, const LeafGeo *geo, const RotDev *rots, int nrot,
                      const double4 *trans, long long ntasks, const double4 *tasks, const GkNodes *nodes,
                      double *out, hipStream_t s) {
    const unsigned nb = (unsigned)((ntasks + kGkTasksPerBlock - 1) / kGkTasksPerBlock);
    const int bs = 15 * kGkTasksPerBlock;
    if (fp64)
        docked_gk_batch<double, double4><<<nb, bs, 0, s>>>((const double4 *const *)grids, geo, rots, nrot, trans,
                                                            ntasks, tasks, nodes, out);
    else
        docked_gk_batch<float, float4><<<nb, bs, 0, s>>>((const float4 *const *)grids, geo, rots, nrot, trans,
                                                          ntasks, tasks, nodes, out);
}

// one level of at most bound open intervals
void launch_docked_gk_level(bool fp64, const void *const *grids, const LeafGeo *geo, const RotDev *rots, int nrot,
                            const double4 *trans, const GkNodes *nodes, const GkLevel &L, long long bound,
                            hipStream_t s) {
    const unsigned nb = (unsigned)std::min<long long>((bound + kGkTasksPerBlock - 1) / kGkTasksPerBlock, 4096);
    const int bs = 15 * kGkTasksPerBlock;
    if (fp64)
        docked_gk_level<double, double4><<<nb, bs, 0, s>>>((const double4 *const *)grids, geo, rots, nrot, trans,
                                                            nodes, L);
    else
        docked_gk_level<float, float4><<<nb, bs, 0, s>>>((const float4 *const *)grids, geo, rots, nrot, trans,
                                                          nodes, L);
}

void launch_azimuthal(bool fp64, const void *const *grids, const LeafGeo *geo, const RotDev *rots, int nrot,
                      const double4 *trans, int npts, const double2 *pts, int nphi, uint64_t seed, double *out,
                      hipStream_t s) {
    if (npts <= 0) return;
    if (fp64)
        azimuthal_kernel<double, double4><<<npts, 256, 0, s>>>((const double4 *const *)grids, geo, rots, nrot, trans,
                                                               pts, nphi, seed, out);
    else
        azimuthal_kernel<float, float4><<<npts, 256, 0, s>>>((const float4 *const *)grids, geo, rots, nrot, trans,
                                                             pts, nphi, seed, out);
}

void launch_docked_cart(bool fp64, const void *const *grids, const LeafGeo *geo, const RotDev *rots,
                        int nrot, const double4 *trans, int n, const double *qxyz, double *out,
                        hipStream_t s) {
    unsigned nb = (n + 255) / 256;
    if (fp64)
        docked_cart_batch<double, double4><<<nb, 256, 0, s>>>((const double4 *const *)grids, geo, rots,
                                                               nrot, trans, n, qxyz, out);
    else
        docked_cart_batch<float, float4><<<nb, 256, 0, s>>>((const float4 *const *)grids, geo, rots, nrot,
                                                             trans, n, qxyz, out);
}

}  // namespace dplus

namespace dplus {

// ------------------------------------------------------------------ grid-level docking
__device__ __forceinline__ void node_indices(long long index, int &qi, long long &ti, long long &pi) {
    if (index <= 0) {
        qi = 0;
        ti = pi = 0;
        return;
    }
    long long q = (long long)cbrt((double)index / 6.0);
    if (q < 1) q = 1;
    while (q > 1 && shell_base(q) > index) q--;
    while (shell_base(q + 1) <= index) q++;
    const long long rem = index - shell_base(q);
    qi = (int)q;
    ti = rem / (6 * q);
    pi = rem % (6 * q);
}

// (13 copies, grid 150: 700 -> 500 us with the polynomial angles and phases of FP32 grids and
// the node's norm known; VALU-bound at 385 instructions a lookup)
// ManualSymmetry::calcAmplitude (Symmetries.cpp:697-716) at every node of the
// output grid (Grid.cpp:760-826 node vectors), sub-amplitudes through GetCart
// Space-filling lattice sum sum_{n<N} e^{i n d} = e^{i(N-1)d/2} sin(Nd/2)/sin(d/2)
// (GridSymmetry::calcAmplitude, DefaultModels/Symmetries.cpp:97-136; GPU
// CalcSpaceFillingKernelJcb, GPU/SymmetryGenJacob.cu:32-132).  N at d = 0 as the
// reference does; at the other zeros of sin(d/2) (d = 2 pi k) the limit
// N (-1)^{(N-1)k}, where the reference's expression is 0/0.
__device__ inline void lattice_mul(double d, double n, double &re, double &im) {
    if (fabs(d) < 100.0 * 2.220446049250313e-16 || n == 1.0) {
        re *= n;
        im *= n;
        return;
    }
    const double h = 0.5 * d;
    const double sh = sin(h);
    double f;
    if (fabs(sh) < 1e-12) {
        const double k = rint(d / k2Pi);
        f = (fmod(fabs((n - 1.0) * k), 2.0) == 1.0) ? -n : n;
    } else {
        f = sin(n * h) / sh;
    }
    double sp, cp;
    sincos((n - 1.0) * h, &sp, &cp);
    const double r = re * cp - im * sp, i = im * cp + re * sp;
    re = r * f;
    im = i * f;
}

template <typename T, typename T4>
__global__ __launch_bounds__(256) void dock_grid_kernel(const T4 *const *__restrict__ grids, const LeafGeo *__restrict__ geo,
                                 const RotDev *__restrict__ rots, int nrot, const double4 *__restrict__ trans,
                                 T4 *__restrict__ out, double step_out, long long P, double scale,
                                 LatticeDev lat) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= P) return;
    int qi;
    long long ti, pi;
    node_indices(idx, qi, ti, pi);
    double q[3] = {0.0, 0.0, 0.0};
    if (qi > 0) {
        const double qI = (double)qi * step_out;
        const double tI = kPi * (double)ti / (double)(3 * qi);
        const double pI = k2Pi * (double)pi / (double)(6 * qi);
        double st, ct, sp, cp;
        sincos(tI, &st, &ct);
        sincos(pI, &sp, &cp);
        q[0] = qI * st * cp;
        q[1] = qI * st * sp;
        q[2] = qI * ct;
    }
    double ax = 0.0, ay = 0.0;
    const double n = (double)qi * step_out, ninv = 1.0 / n;  // a node's norm, turned or not
    for (int r = 0; r < nrot; r++) {
        const RotDev rd = rots[r];
        double rv[3];
        rotate_t(rd, q, rv);
        const LeafGeo G = geo[rd.leaf];
        const cplx<T> a = n > 0.0 ? get_turned<T, T4>(grids[rd.leaf], G.N, G.step, rv, n, ninv)
                                  : get_sphr<T, T4>(grids[rd.leaf], G.N, G.step, 0.0, 0.0, 0.0);
        double sc = 0.0, ss = 0.0;
        for (int tr = 0; tr < rd.nt; tr++) {
            const double4 t = trans[rd.t0 + tr];
            double s = 0.0, c = 1.0;
            if (t.x != 0.0 || t.y != 0.0 || t.z != 0.0) phase_exact<T>(q[0] * t.x + q[1] * t.y + q[2] * t.z, s, c);
            sc += c;
            ss += s;
        }
        ax += ((double)a.x * sc - (double)a.y * ss) * rd.scale;
        ay += ((double)a.y * sc + (double)a.x * ss) * rd.scale;
    }
    if (lat.on)
        for (int k = 0; k < 3; k++)
            lattice_mul(q[0] * lat.v[3 * k] + q[1] * lat.v[3 * k + 1] + q[2] * lat.v[3 * k + 2], lat.n[k], ax, ay);
    T4 o;
    o.x = (T)(ax * scale);
    o.y = (T)(ay * scale);
    o.z = (T)0;
    o.w = (T)0;
    out[idx] = o;
}

void dock_grid(const DockSet &D, Grid &out, double scale, hipStream_t s, const LatticeDev *lattice) {
    const unsigned nb = (unsigned)((out.P + 255) / 256);
    LatticeDev lat{};
    if (lattice) lat = *lattice;
    KTimer kt("dock", s);
    if (D.fp64)
        dock_grid_kernel<double, double4><<<nb, 256, 0, s>>>((const double4 *const *)D.grids.p,
                                                              (const LeafGeo *)D.geos.p, (const RotDev *)D.rotb.p,
                                                              D.nrot, (const double4 *)D.trb.p,
                                                              (double4 *)out.dev.p, out.step, out.P, scale, lat);
    else
        dock_grid_kernel<float, float4><<<nb, 256, 0, s>>>((const float4 *const *)D.grids.p,
                                                            (const LeafGeo *)D.geos.p, (const RotDev *)D.rotb.p,
                                                            D.nrot, (const double4 *)D.trb.p, (float4 *)out.dev.p,
                                                            out.step, out.P, scale, lat);
    check_hip(hipGetLastError(), "dock_grid launch");
    out.splines(s);
    check_hip(hipStreamSynchronize(s), "dock_grid");
}

}  // namespace dplus

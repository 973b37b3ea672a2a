// amp_mesh.hip -- amplitude grids through a frequency mesh, for gfx950.
//
// The direct builder (amp_build.hip) sums every source at every canonical node:
// nodes x sources terms, at the VALU's issue limit.  For structures of more than
// a few thousand sources this file evaluates the same sums as a non-uniform
// Fourier transform between two irregular point sets (a "type 3" transform:
// Dutt and Rokhlin 1993; Lee and Greengard 2005; with the Kaiser-Bessel window):
//
//   F_f(q) = sum_a w_a e^{i q.r_a}   for every class f of sources (an ion; the boxes)
//   A(q)   = scale * sum_f ff_f(|q|) F_f(q)
//
//  1. mesh_weights  the window values of every box piece on a Cartesian mesh of
//                   spacing h, per axis, divided by the second window's transform.
//  2. mesh_spread   the mesh densities: for a brick of 8 x 8 x 16 mesh points, the
//                   sum over its sources of wx(x) wy(y) wz(z) -- a contraction over
//                   the sources on the FP64 matrix unit (an atom's window values,
//                   one polynomial each, are formed on the way into LDS).
//  3. mesh_dft      the densities' transform at the points of a frequency mesh of
//                   spacing dk, one axis at a time, as products with the axis's
//                   exponentials (divided by the first window's transform) on the
//                   FP64 matrix unit: the meshes have ~30..250 points per axis, where
//                   dense products beat a fast transform's passes.
//  4. mesh_interp   the nodes: a workgroup takes a patch of one shell, adds the classes'
//                   frequency meshes with the shell's form factors while it sums the
//                   z window points of every row, and then every node's W^2 points
//                   in (x, y); the antipode takes the conjugate.
//
// Solvent boxes are cut into pieces of at most kMeshPiece nm; a piece is spread as
// the Gauss-Legendre quadrature of its volume, axis by axis, which gives the box
// transform prod_a L_a sinc(q_a L_a / 2) to the window's accuracy.
//
// Measured (MI355X, GPU time of a build): 50,000 atoms and 136,000 boxes at grid 250,
// mixed: 119.7 ms direct -> 1.23 ms (spread 0.62, interpolation 0.34, transforms 0.19,
// weights 0.07); 200,000 atoms at grid 110, mixed: 13.9 -> 0.78 ms; 5,000 atoms and
// 22,000 boxes at grid 120, FP64: 19.5 -> 0.81 ms.  Error against direct sums in 64 bits,
// median over the shells of |dA| / |A| (2-norms, against 80-bit sums; 2,000 to 20,000 atoms, a
// protein, a cube, a slab, off the origin): mixed 6e-8 .. 1.6e-7 where the direct builder has
// 1.1e-7 .. 4.3e-7; FP64 1.5e-16 .. 2.6e-15 where the direct one has 2.3e-16 .. 2.5e-15.
//
// Everything up to the frequency mesh is FP64.  A mixed grid's nodes are
// interpolated in FP32 with W = 8 and an FP64 grid's in FP64 with W = 16.
// No step depends on the order of concurrent work: a build always gives the same bits.

#include <cmath>
#include <mutex>
#include <vector>

#include "device.hpp"

namespace dplus {

using d4 = __attribute__((__vector_size__(4 * sizeof(double)))) double;

// ------------------------------------------------------------------ windows (host)
// phi(t) = I0(beta sqrt(1 - (2 t / W)^2)) / I0(beta), |t| <= W / 2, beta = 0.985
// (1 - 1 / (2 sigma)) pi W for oversampling sigma (|xi| <= pi / sigma is used),
// represented per unit interval l by a polynomial of degree W + 1 in z = 2 s - 1,
// phi(l - W/2 + s); the transform phihat(xi) is that polynomial's (Gauss quadrature),
// and 1 / phihat a polynomial in xi^2 on |xi| <= pi / 2.  At sigma = 2, W = 8 represents
// e^{i u xi} to 6e-8 (rms) and W = 10 to 7e-10; W = 16 to 1e-15 at sigma = 2 and to
// 1e-16 at 2.5, where the window's transform falls 3.5 times over the range instead of
// 8 and so amplifies rounding less.
namespace {

constexpr int kInvDeg = 16;  // 1 / phihat: coefficients of xi^0, xi^2, ...

struct Window {
    int W = 0;
    std::vector<double> coef;  // [W][W + 2], ascending powers of z
    double inv[kInvDeg];
};

long double bessel_i0(long double x) {
    long double t = 1.0L, s = 1.0L;
    for (int k = 1; k < 200; k++) {
        t *= (x / (2.0L * k)) * (x / (2.0L * k));
        s += t;
        if (t < 1e-21L * s) break;
    }
    return s;
}

// Gauss-Legendre nodes and weights on [-1, 1].  In long double: a weight carries the
// polynomials' rounding divided by 1 - z^2, 6e-15 of a double one, and every transform 1e-15
void gauss_legendre(int n, std::vector<long double> &x, std::vector<long double> &w) {
    x.assign(n, 0.0L);
    w.assign(n, 0.0L);
    for (int i = 0; i < n; i++) {
        long double z = std::cos(kPi * (i + 0.75) / (n + 0.5)), dp = 1.0L;
        for (int it = 0; it < 6; it++) {  // (doubles its digits each time, from four)
            long double p0 = 1.0L, p1 = z;
            for (int k = 2; k <= n; k++) {
                const long double p2 = ((2.0L * k - 1.0L) * z * p1 - (k - 1.0L) * p0) / k;
                p0 = p1;
                p1 = p2;
            }
            dp = n * (z * p1 - p0) / (z * z - 1.0L);
            z -= p1 / dp;
        }
        x[i] = z;
        w[i] = 2.0L / ((1.0L - z * z) * dp * dp);
    }
}

// Chebyshev interpolation of f on [-1, 1] at n nodes, as ascending powers (long double throughout)
template <typename F>
void power_fit(int n, F f, long double *c) {
    std::vector<long double> a(n, 0.0L), p(n, 0.0L), t0(n, 0.0L), t1(n, 0.0L), t2(n, 0.0L);
    const long double pi = 3.141592653589793238462643383279502884L;
    std::vector<long double> y(n);
    for (int k = 0; k < n; k++) y[k] = f(cosl(pi * (k + 0.5L) / n));
    for (int m = 0; m < n; m++) {
        for (int k = 0; k < n; k++) a[m] += y[k] * cosl(pi * m * (k + 0.5L) / n);
        a[m] *= (m == 0 ? 1.0L : 2.0L) / n;
    }
    t0[0] = 1.0L;
    if (n > 1) t1[1] = 1.0L;
    for (int i = 0; i < n; i++) p[i] = a[0] * t0[i] + (n > 1 ? a[1] * t1[i] : 0.0L);
    for (int m = 2; m < n; m++) {
        for (int i = 0; i < n; i++) t2[i] = (i > 0 ? 2.0L * t1[i - 1] : 0.0L) - t0[i];
        for (int i = 0; i < n; i++) p[i] += a[m] * t2[i];
        t0.swap(t1);
        t1.swap(t2);
    }
    for (int i = 0; i < n; i++) c[i] = p[i];
}

// single: coefficients for FP32 evaluation, whose transform is that of the rounded ones
const Window &window(int W, double sigma, bool single) {
    static std::mutex mu;
    static Window tab[32];  // one oversampling and one precision per width
    std::lock_guard<std::mutex> lk(mu);
    Window &k = tab[W];
    if (k.W) return k;
    const int nc = W + 2;
    const long double beta = 0.985 * (1.0 - 0.5 / sigma) * kPi * W, i0b = bessel_i0(beta);
    k.coef.assign((size_t)W * nc, 0.0);
    std::vector<long double> fit(std::max(nc, kInvDeg)), phi((size_t)W * nc), gx, gw;
    gauss_legendre(32, gx, gw);
    long double area = 0.0L;
    for (int l = 0; l < W; l++) {
        power_fit(nc, [&](long double z) {
            const long double t = l - 0.5L * W + 0.5L * (z + 1.0L);
            return bessel_i0(beta * sqrtl(std::max(0.0L, 1.0L - 4.0L * t * t / ((long double)W * W)))) / i0b;
        }, fit.data());
        for (int g = 0; g < 32; g++) {
            long double v = 0.0L;
            for (int d = nc - 1; d >= 0; d--) v = v * gx[g] + fit[d];
            area += 0.5L * gw[g] * v;
        }
        for (int d = 0; d < nc; d++) phi[(size_t)l * nc + d] = fit[d];
    }
    // of unit area: 1 / phihat starts at 1, which no rounding of its constant term scales
    for (size_t i = 0; i < phi.size(); i++) {
        k.coef[i] = (double)(phi[i] / area);
        if (single) k.coef[i] = (double)(float)k.coef[i];
    }
    auto phihat = [&](long double xi) {
        long double s = 0.0L;
        for (int l = 0; l < W; l++)
            for (int g = 0; g < 32; g++) {
                long double v = 0.0L;
                for (int d = nc - 1; d >= 0; d--) v = v * gx[g] + (long double)k.coef[(size_t)l * nc + d];
                s += 0.5L * gw[g] * v * cosl(xi * (l - 0.5L * W + 0.5L * (gx[g] + 1.0L)));
            }
        return s;
    };
    // in x = (xi / (pi / 2))^2 on [0, 1]: fitted in z = 2 x - 1 and expanded in powers of
    // x, whose coefficients are positive (no cancellation where the value is small)
    const long double half = 0.5L * 3.141592653589793238462643383279502884L;
    power_fit(kInvDeg, [&](long double z) {
        const long double x = 0.5L * (z + 1.0L);
        return 1.0L / phihat(half * sqrtl(x > 0 ? x : 0.0L));
    }, fit.data());
    std::vector<long double> p(kInvDeg, 0.0L), t(kInvDeg, 0.0L);
    for (int d = kInvDeg - 1; d >= 0; d--) {  // p <- p (2 x - 1) + fit[d]
        for (int i = 0; i < kInvDeg; i++) t[i] = -p[i] + (i > 0 ? 2.0L * p[i - 1] : 0.0L);
        t[0] += fit[d];
        p.swap(t);
    }
    for (int i = 0; i < kInvDeg; i++) k.inv[i] = (double)p[i];
    k.W = W;
    return k;
}

}  // namespace

// ------------------------------------------------------------------ device helpers
// 1 / phihat at xi (|xi| <= pi / 2), in powers of (2 xi / pi)^2
__device__ __forceinline__ double inv_transform(const double *__restrict__ inv, double xi) {
    const double y = xi * (2.0 / kPi), z = y * y;
    double v = inv[kInvDeg - 1];
#pragma unroll
    for (int i = kInvDeg - 2; i >= 0; i--) v = fma(v, z, inv[i]);
    return v;
}

// the window's values at its W points: z -> y[0..W), c = [W][W + 2] ascending powers.
// phi is even: the values at l and W - 1 - l are E(z^2) + z O(z^2) and E - z O.
template <typename T, int W, typename F>
__device__ __forceinline__ void window_values(const T *c, T z, F put) {
    constexpr int nc = W + 2;
    static_assert(W % 2 == 0, "even and odd parts pair up");
    const T zz = z * z;
#pragma unroll
    for (int l = 0; l < W / 2; l++) {
        T e = c[l * nc + nc - 2], o = c[l * nc + nc - 1];
#pragma unroll
        for (int d = nc - 4; d >= 0; d -= 2) {
            e = fma(e, zz, c[l * nc + d]);
            o = fma(o, zz, c[l * nc + d + 1]);
        }
        put(l, fma(z, o, e));
        put(W - 1 - l, fma(-z, o, e));
    }
}

// The place of coordinate x = r * scale + off / 2 (off whole) on a mesh of unit spacing for a
// window of W points (W even): its first point, and z in (-1, 1] of the window's
// polynomials.  The fraction comes from one fused product, so it keeps the full
// precision of r * scale whatever the mesh's size.
template <int W>
__device__ __forceinline__ int window_place(double r, double scale, int off, double &z) {
    const double i = ceil(fma(r, scale, 0.5 * (double)off));  // the first point + W / 2
    z = -2.0 * fma(r, scale, 0.5 * (double)off - i) - 1.0;
    return (int)i - W / 2;
}

// ------------------------------------------------------------------ 1. weights
// One (box piece, axis) per thread: the piece's Gauss-Legendre nodes one after the
// other, each adding its window times weight / phihat_interp(r dk) to the thread's row
// in LDS; the rows leave in order.  wgt[(s * 3 + axis) * WP + p] is the value at mesh
// point base[s].axis + p.
constexpr int kMaxGl = 16, kMaxWp = 31;

template <int WS>
__global__ __launch_bounds__(192) void mesh_weights(MeshPlan P, const double4 *__restrict__ src,
                                                    const double4 *__restrict__ len, long long nsrc, int gl, int WP,
                                                    const double *__restrict__ tab, double *__restrict__ wgt,
                                                    int4 *__restrict__ base) {
    extern __shared__ double rows[];  // 192 rows of WP | 1
    const int S = WP | 1;
    const long long s0 = (long long)blockIdx.x * 64;
    const int ns = (int)min(64LL, nsrc - s0);
    const int t = threadIdx.x, s = t / 3, a = t - 3 * s;
    double *row = rows + t * S;
    for (int p = 0; p < WP; p++) row[p] = 0.0;
    if (s < ns) {
        const double4 p = src[s0 + s], L = len[s0 + s];
        const double l = 0.5 * (a == 0 ? L.x : a == 1 ? L.y : L.z), c = (a == 0 ? p.x : a == 1 ? p.y : p.z) - P.ax[a].c;
        const double w = l * (a == 0 ? p.w : 1.0), hinv = P.ax[a].hinv, dk = P.ax[a].dk;
        const double *gx = tab + P.t_gl;  // nodes, falling, then weights
        const int off = P.ax[a].m - 1;
        double z;
        const int b = window_place<WS>(c + l * gx[gl - 1], hinv, off, z);
        ((int *)base)[(s0 + s) * 4 + a] = b;
        for (int g = 0; g < gl; g++) {
            const double r = c + l * gx[g];
            const int o = window_place<WS>(r, hinv, off, z) - b;
            const double f = w * gx[gl + g] * inv_transform(tab + P.t_iinv, r * dk);
            // o + WS <= WP: a piece spans at most WP - WS - 1 mesh steps
            window_values<double, WS>(tab + P.t_spread, z, [&](int k, double y) { row[o + k] = fma(f, y, row[o + k]); });
        }
    }
    __syncthreads();
    const int n = ns * 3 * WP;
    for (int e = t; e < n; e += 192) {
        const int r = e / WP;
        wgt[s0 * 3 * WP + e] = rows[r * S + e - r * WP];
    }
}

// ------------------------------------------------------------------ 2. spread
// One workgroup per (brick, class): mesh points [8 bx, +8) x [8 by, +8) x [16 bz, +16).
// The sources of a class are sorted by cell (z fastest), so those whose windows can
// reach the brick are one contiguous run per (x, y) cell column.  256 at a time, their
// window values at the brick's points go to LDS, then each of four wave groups sums 64
// of them: wave w of a group rows (x = 2 w + r / 8, y = r % 8) by 16 z points,
// D[row][z] += (wx wy)[row][s] wz[z][s], in 16x16x4 FP64 MFMA steps; the groups' sums
// are added at the end.  Every point of the mesh is written.  A mesh has a few hundred
// bricks and the fullest holds many times the mean, so the time is the fullest brick's
// chain of batches (run -> source -> window -> LDS -> MFMA): 16 waves and 256 sources per
// batch, the next batch's loads under this one's MFMA steps, and nslice slices of a
// brick's batches (each with a mesh of its own; the transform adds them).
constexpr int kRuns = kMeshCells * kMeshCells;
constexpr int kBatch = 256;

template <int WS>
__global__ __launch_bounds__(1024) void mesh_spread(MeshPlan P, int f0, int nslice, const double4 *__restrict__ atoms,
                                                    const int *__restrict__ cell_start, const double *__restrict__ tab,
                                                    const double *__restrict__ wb, const int4 *__restrict__ bb,
                                                    double *__restrict__ mesh) {
    __shared__ double wt[32][kBatch + 2];  // point (8 x, 8 y, 16 z) x source; + 2: the MFMA operand reads spread over the banks
    __shared__ int run0[kRuns], runp[kRuns + 1], sidx[kBatch];
    __shared__ int wsum[16];
    const int f = f0 + blockIdx.y / nslice, slice = blockIdx.y % nslice;
    const bool boxes = P.boxes && f == P.nfield - 1;
    const int nbz = P.ax[2].m / 16, nby = P.ax[1].m / 8;
    const int b = blockIdx.x, bz = b % nbz, by = (b / nbz) % nby, bx = b / (nbz * nby);
    const int o[3] = {8 * bx, 8 * by, 16 * bz}, n[3] = {8, 8, 16};
    int lo[3], hi[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const double reach = (0.5 * WS + 1e-6) * P.ax[a].h + (boxes ? P.box_half[a] : 0.0);
        const double x = P.ax[a].x0 + o[a] * P.ax[a].h;
        const double l = (x - reach - P.cell0[a]) * P.cell_inv[a], h = (x + (n[a] - 1) * P.ax[a].h + reach - P.cell0[a]) * P.cell_inv[a];
        lo[a] = (int)fmin(fmax(floor(l), 0.0), (double)P.ncell[a]);
        hi[a] = (int)fmin(fmax(floor(h), -1.0), (double)(P.ncell[a] - 1));
    }
    const int nx = max(0, hi[0] - lo[0] + 1), ny = max(0, hi[1] - lo[1] + 1);
    const int nrun = hi[2] >= lo[2] ? nx * ny : 0;  // at most kRuns
    const int *cs = cell_start + (size_t)f * (P.ncell[0] * P.ncell[1] * P.ncell[2] + 1);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int total = 0;
    {
        const int r = threadIdx.x;
        int cnt = 0, st = 0;
        if (r < nrun) {
            const int cell = ((lo[0] + r / ny) * P.ncell[1] + lo[1] + r % ny) * P.ncell[2];
            st = cs[cell + lo[2]];
            cnt = cs[cell + hi[2] + 1] - st;
        }
        int inc = cnt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int t = __shfl_up(inc, d, 64);
            if (lane >= d) inc += t;
        }
        if (lane == 63) wsum[w] = inc;
        __syncthreads();
        int before = 0;
        for (int k = 0; k < 16; k++) {
            if (k < w) before += wsum[k];
            total += wsum[k];
        }
        if (r < nrun) {
            run0[r] = st;
            runp[r] = before + inc - cnt;
        }
        __syncthreads();
    }
    auto source = [&](int e) {  // the e-th source of the runs
        int l = 0, h = nrun - 1;  // the last run that starts at or before e
        while (l < h) {
            const int m = (l + h + 1) >> 1;
            if (runp[m] <= e)
                l = m;
            else
                h = m - 1;
        }
        return run0[l] + (e - runp[l]);
    };
    // a batch's sum, added to the brick's when it is complete (the density is a sum of
    // thousands of like-signed terms: two levels keep its rounding at FP64's)
    d4 acc = {0.0, 0.0, 0.0, 0.0}, sum = {0.0, 0.0, 0.0, 0.0};
    const int wg = w >> 2, wq = w & 3, mrow = lane & 15, mk = lane >> 4;
    const int px = 2 * wq + (mrow >> 3), py = 8 + (mrow & 7), pz = 16 + mrow;
    auto multiply = [&](int k0) {  // half of the batch's MFMA steps
#pragma unroll
        for (int k = k0; k < k0 + 8; k++) {
            const int s = 64 * wg + 4 * k + mk;
            const double a = wt[px][s] * wt[py][s], c = wt[pz][s];
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, c, acc, 0, 0, 0);
        }
    };
    const int stride = kBatch * nslice;  // this slice's batches: b0, b0 + stride, ...
    int b0 = kBatch * slice;
    if (boxes && b0 < total) {
        // thread: point pt of the pieces tid / 32 + 32 k; the next batch's positions and
        // values are loaded around this batch's MFMA steps
        const int pt = threadIdx.x & 31, a = pt < 8 ? 0 : pt < 16 ? 1 : 2, sl = threadIdx.x >> 5;
        const int at = a == 0 ? o[0] + pt : a == 1 ? o[1] + pt - 8 : o[2] + pt - 16;
        int i[8];
        double v[8];
        auto places = [&]() {
#pragma unroll
            for (int k = 0; k < 8; k++) i[k] = at - ((const int *)bb)[(size_t)sidx[sl + 32 * k] * 4 + a];
        };
        auto values = [&]() {
#pragma unroll
            for (int k = 0; k < 8; k++)
                v[k] = wb[((size_t)sidx[sl + 32 * k] * 3 + a) * P.wp_box + min(max(i[k], 0), P.wp_box - 1)];
        };
        if (threadIdx.x < kBatch) sidx[threadIdx.x] = source(min(b0 + (int)threadIdx.x, total - 1));
        __syncthreads();
        places();
        values();
        for (; b0 < total; b0 += stride) {
#pragma unroll
            for (int k = 0; k < 8; k++)
                wt[pt][sl + 32 * k] = i[k] >= 0 && i[k] < P.wp_box && b0 + sl + 32 * k < total ? v[k] : 0.0;
            __syncthreads();
            const bool more = b0 + stride < total;
            if (more && threadIdx.x < kBatch) sidx[threadIdx.x] = source(min(b0 + stride + (int)threadIdx.x, total - 1));
            multiply(0);
            __syncthreads();  // the next batch's sources stand
            if (more) places();
            multiply(8);
            sum += acc;
            acc = d4{0.0, 0.0, 0.0, 0.0};
            if (more) values();
            __syncthreads();
        }
    } else if (b0 < total) {
        // an atom's window: waves 4 a .. 4 a + 3 serve axis a < 3, one lane per source; the
        // next batch's atoms are loaded before this batch's MFMA steps
        const int ax = min(wg, 2), first = 8 * ax, npt = ax == 2 ? 16 : 8;
        const MeshAxis A = P.ax[ax];
        const int oax = ax == 0 ? o[0] : ax == 1 ? o[1] : o[2], col = wq * 64 + lane;
        double pos = 0.0;
        auto fetch = [&](int e) {
            if (wg < 3) pos = ((const double *)(atoms + source(min(e, total - 1))))[ax];
        };
        fetch(b0 + col);
        for (; b0 < total; b0 += stride) {
            if (wg < 3) {
#pragma unroll
                for (int k = 0; k < 16; k++)
                    if (k < npt) wt[first + k][col] = 0.0;
                const double r = pos - A.c;
                double z;
                const int at = window_place<WS>(r, A.hinv, A.m - 1, z) - oax;
                const double g = b0 + col < total ? inv_transform(tab + P.t_iinv, r * A.dk) : 0.0;
                window_values<double, WS>(tab + P.t_spread, z, [&](int l, double y) {
                    if (at + l >= 0 && at + l < npt) wt[first + at + l][col] = g * y;
                });
            }
            __syncthreads();
            if (b0 + stride < total) fetch(b0 + stride + col);
            multiply(0);
            multiply(8);
            sum += acc;
            acc = d4{0.0, 0.0, 0.0, 0.0};
            __syncthreads();
        }
    }
    // the four groups' sums, in order (16 waves x 4 values x 64 lanes of LDS)
    double *part = &wt[0][0];
#pragma unroll
    for (int r = 0; r < 4; r++) part[(w * 4 + r) * 64 + lane] = sum[r];
    __syncthreads();
    if (wg > 0) return;
    double *out = mesh + (size_t)blockIdx.y * P.ax[0].m * P.ax[1].m * P.ax[2].m;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        double v = sum[r];
#pragma unroll
        for (int g = 1; g < 4; g++) v += part[((4 * g + w) * 4 + r) * 64 + lane];
        const int row = 4 * r + mk;  // the FP64 MFMA's D: row 4 r + lane / 16, column lane % 16
        const int x = o[0] + 2 * w + (row >> 3), y = o[1] + (row & 7), z = o[2] + mrow;
        out[((size_t)x * P.ax[1].m + y) * P.ax[2].m + z] = v;
    }
}

// ------------------------------------------------------------------ 3. transform
// E[n][j] = e^{i k_n x_j} / psihat(k_n h) of one axis, real and imaginary parts apart
__global__ __launch_bounds__(256) void mesh_twiddles(MeshPlan P, const double *__restrict__ tab, double *__restrict__ E0,
                                                     double *__restrict__ E1, double *__restrict__ E2) {
    const int a = blockIdx.y;
    const MeshAxis X = P.ax[a];
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= X.k * X.m) return;
    const int n = e / X.m, j = e % X.m;
    // k x in revolutions: a whole number times turn = 1 / (4 pi hinv dkinv), the product
    // with turn's leading part split exactly, so the angle keeps its absolute precision
    const double p = (double)(n - X.n0) * (double)(2 * j - (X.m - 1));
    const double r = p * X.turn, e0 = fma(p, X.turn, -r) + p * X.turn_lo;
    double s, c;
    sincospi(2.0 * ((r - rint(r)) + e0), &s, &c);
    const double g = inv_transform(tab + P.t_sinv, (double)(n - X.n0) * X.dk * X.h);
    double *E = a == 0 ? E0 : a == 1 ? E1 : E2;
    E[e] = c * g;
    E[(size_t)X.k * X.m + e] = s * g;
}

// out[f][n][row] (kLast: out[f][row][n]) = sum_j E[n][j] in[f][row][j]: a workgroup
// takes 32 n x 64 rows, its four waves 16 x 32 each (1 x 2 tiles, real and imaginary
// accumulators; two workgroups or more per CU hide each other's barriers), 16 j at a time through LDS (stride 17: the MFMA operand reads hit
// distinct banks), the next 16 j loaded while these are multiplied.  TI: double (real
// input: the sum of nslice arrays, `rows * J` apart) or double2, TO: double2 or float2.
constexpr int kDftJ = 16, kDftS = 17;

template <typename TI, typename TO, bool kLast>
__global__ __launch_bounds__(256, 2) void mesh_dft(const TI *__restrict__ in, TO *__restrict__ out,
                                                   const double *__restrict__ E, int J, int nk, int rows, int nslice) {
    constexpr bool kReal = sizeof(TI) == sizeof(double);
    __shared__ double er[32 * kDftS], ei[32 * kDftS], xr[64 * kDftS], xi[kReal ? 1 : 64 * kDftS];
    const int f = blockIdx.z, n0 = blockIdx.y * 32, r0 = blockIdx.x * 64;
    in += (size_t)f * nslice * rows * J;
    out += (size_t)f * rows * nk;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int wn = (w & 1) * 16, wr = (w >> 1) * 32, mr = lane & 15, mk = lane >> 4;
    d4 re[2], im[2];
    const d4 zero = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int b = 0; b < 2; b++) re[b] = im[b] = zero;
    // this thread's share of a chunk: column j = tid % 16 of rows tid / 16 + 16 t
    const int lj = threadIdx.x & 15, lr = threadIdx.x >> 4;
    double ga[2], gb[2];
    TI gx[4];
    auto fetch = [&](int j0) {
        const int j = min(j0 + lj, J - 1);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int n = min(n0 + lr + 16 * t, nk - 1);
            ga[t] = E[(size_t)n * J + j];
            gb[t] = E[(size_t)(nk + n) * J + j];
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const size_t at = (size_t)min(r0 + lr + 16 * t, rows - 1) * J + j;
            gx[t] = in[at];
            if constexpr (kReal)
                for (int y = 1; y < nslice; y++) gx[t] += in[(size_t)y * rows * J + at];
        }
    };
    fetch(0);
    for (int j0 = 0; j0 < J; j0 += kDftJ) {
        const bool inj = j0 + lj < J;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int e = (lr + 16 * t) * kDftS + lj;
            if (t < 2) {
                er[e] = inj ? ga[t & 1] : 0.0;
                ei[e] = inj ? gb[t & 1] : 0.0;
            }
            if constexpr (kReal) {
                xr[e] = inj ? gx[t] : 0.0;
            } else {
                xr[e] = inj ? gx[t].x : 0.0;
                xi[e] = inj ? gx[t].y : 0.0;
            }
        }
        __syncthreads();
        if (j0 + kDftJ < J) fetch(j0 + kDftJ);
        d4 sr[2] = {zero, zero}, si[2] = {zero, zero};  // this chunk's sums
#pragma unroll
        for (int k = 0; k < kDftJ; k += 4) {
            double X[2], Y[2];
            const double Er = er[(wn + mr) * kDftS + k + mk], Ei = ei[(wn + mr) * kDftS + k + mk];
#pragma unroll
            for (int b = 0; b < 2; b++) {
                X[b] = xr[(wr + 16 * b + mr) * kDftS + k + mk];
                Y[b] = kReal ? 0.0 : xi[(wr + 16 * b + mr) * kDftS + k + mk];
            }
            auto mma = [](double e, double x, d4 c) {
                return kLast ? __builtin_amdgcn_mfma_f64_16x16x4f64(x, e, c, 0, 0, 0)
                             : __builtin_amdgcn_mfma_f64_16x16x4f64(e, x, c, 0, 0, 0);
            };
#pragma unroll
            for (int b = 0; b < 2; b++) {
                sr[b] = mma(Er, X[b], sr[b]);
                si[b] = mma(Ei, X[b], si[b]);
                if (!kReal) {
                    sr[b] = mma(-Ei, Y[b], sr[b]);
                    si[b] = mma(Er, Y[b], si[b]);
                }
            }
        }
#pragma unroll
        for (int b = 0; b < 2; b++) {
            re[b] += sr[b];
            im[b] += si[b];
        }
        __syncthreads();
    }
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 4 * r + mk;
            const int n = n0 + wn + (kLast ? mr : i), row = r0 + wr + 16 * b + (kLast ? i : mr);
            if (n < nk && row < rows) {
                TO v;
                v.x = re[b][r];
                v.y = im[b][r];
                out[kLast ? (size_t)row * nk + n : (size_t)n * rows + row] = v;
            }
        }
}

// ------------------------------------------------------------------ 4. interpolation
// One workgroup: a patch of rows j0.. and columns k0.. of one shell's canonical half
// (rows j <= 3 i / 2; of the equator row's nodes the first half turn), sized by the
// host in frequency steps.  The patch's window points span a small box of the
// frequency mesh.  A row's nodes share q_z, so the z sum is taken once per row: each
// thread walks the z points of one (x, y) column of the box, adds the classes there
// with the shell's form factors, and accumulates the column into every row with the
// row's z window (zero outside it); the rows' (x, y) planes go to LDS, and each node
// sums its W x W points there -- per node W^2 taps and its share of the columns
// instead of W^3 taps.
constexpr int kPatchCols = 256, kPatchZ = 40;

template <typename T, typename T2, typename T4, int W, int kRows, int kThreads>
__global__ __launch_bounds__(kThreads, 2) void mesh_interp(MeshPlan P, const MeshBand *__restrict__ bands, int nbands,
                                                   const double *__restrict__ ff, const int *__restrict__ fion,
                                                   const double *__restrict__ tab, const T2 *__restrict__ G,
                                                   T4 *__restrict__ grid, double scale) {
    constexpr int nc = W + 2, kYUnroll = sizeof(T) == 8 ? 1 : W / 2, kZ = sizeof(T) == 8 ? 4 : 8;
    extern __shared__ unsigned char raw[];
    T2 *planes = reinterpret_cast<T2 *>(raw);
    __shared__ T coef[W * nc];
    __shared__ T wzt[kPatchZ][kRows];
    __shared__ double rz[kRows], rs[kRows], cc[kPatchCols], cn[kPatchCols];
    __shared__ double wf[kMeshFields];
    constexpr int kWaves = kThreads / 64;
    __shared__ int red[kWaves][4];
    int lo = 0, hi = nbands - 1;
    const int tile = blockIdx.x;
    while (lo < hi) {
        const int m = (lo + hi + 1) >> 1;
        if (bands[m].tile0 <= tile)
            lo = m;
        else
            hi = m - 1;
    }
    const MeshBand B = bands[lo];
    const int shell = B.shell, n6 = 6 * shell, half = 3 * shell;
    const int k0 = (tile - B.tile0) * B.cols, ncol = min(B.cols, n6 - k0), nrow = B.rows, nn = nrow * ncol;
    const double q = (double)shell * P.step;
    for (int e = threadIdx.x; e < W * nc; e += kThreads) coef[e] = (T)tab[P.t_interp + e];
    if (threadIdx.x < P.nfield)
        wf[threadIdx.x] = fion[threadIdx.x] < 0 ? 1.0 : ff[(size_t)shell * P.nion + fion[threadIdx.x]];
    if (threadIdx.x >= 64 && threadIdx.x < 64 + nrow) {
        const int r = threadIdx.x - 64;
        double s, c;
        sincospi((double)(B.j0 + r) / (double)half, &s, &c);
        rz[r] = q * c;
        rs[r] = q * s;
    }
    for (int e = threadIdx.x; e < ncol; e += kThreads) {
        double s, c;  // (of whole fractions of a half turn: an angle in radians carries two more roundings)
        sincospi((double)(k0 + e) / (double)half, &s, &c);
        cc[e] = c;
        cn[e] = s;
    }
    __syncthreads();
    // window of node (r, c): first frequency point on each axis, and z of the polynomials
    auto place_x = [&](int r, int c, double &z) { return window_place<W>(rs[r] * cc[c], P.ax[0].dkinv, 0, z) + P.ax[0].n0; };
    auto place_y = [&](int r, int c, double &z) { return window_place<W>(rs[r] * cn[c], P.ax[1].dkinv, 0, z) + P.ax[1].n0; };
    auto place_z = [&](int r, double &z) { return window_place<W>(rz[r], P.ax[2].dkinv, 0, z) + P.ax[2].n0; };
    // the box: q_z falls with the row; x and y over the patch's nodes
    double zz;
    const int z0 = place_z(nrow - 1, zz), nz = place_z(0, zz) - z0 + W, nz8 = (nz + kZ - 1) / kZ * kZ;
    int mnx = 1 << 30, mxx = -(1 << 30), mny = 1 << 30, mxy = -(1 << 30);
    for (int e = threadIdx.x; e < nn; e += kThreads) {
        const int ix = place_x(e / ncol, e % ncol, zz), iy = place_y(e / ncol, e % ncol, zz);
        mnx = min(mnx, ix);
        mxx = max(mxx, ix);
        mny = min(mny, iy);
        mxy = max(mxy, iy);
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
        mnx = min(mnx, __shfl_xor(mnx, d, 64));
        mxx = max(mxx, __shfl_xor(mxx, d, 64));
        mny = min(mny, __shfl_xor(mny, d, 64));
        mxy = max(mxy, __shfl_xor(mxy, d, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        int *r = red[threadIdx.x >> 6];
        r[0] = mnx;
        r[1] = mxx;
        r[2] = mny;
        r[3] = mxy;
    }
    for (int e = threadIdx.x; e < nz8 * kRows; e += kThreads) {  // the rows' z windows (nz8 <= kPatchZ by the patch's size)
        const int r = e % kRows, z = e / kRows;
        T v = (T)0;
        if (r < nrow) {
            const int l = z0 + z - place_z(r, zz);
            if (l >= 0 && l < W) {
                const T t = (T)zz;
                v = coef[l * nc + nc - 1];
#pragma unroll
                for (int d = nc - 2; d >= 0; d--) v = fma(v, t, coef[l * nc + d]);
            }
        }
        wzt[z][r] = v;
    }
    __syncthreads();
    int x0 = red[0][0], x1 = red[0][1], y0 = red[0][2], y1 = red[0][3];
#pragma unroll
    for (int k = 1; k < kWaves; k++) {
        x0 = min(x0, red[k][0]);
        x1 = max(x1, red[k][1]);
        y0 = min(y0, red[k][2]);
        y1 = max(y1, red[k][3]);
    }
    const int nx = x1 - x0 + W, ny = y1 - y0 + W;
    const int sx = nx | 1, plane = ny * sx;  // odd row stride: rows start in different banks
    const int Kx = P.ax[0].k, Ky = P.ax[1].k, Kz = P.ax[2].k;
    const size_t fstride = (size_t)Kx * Ky * Kz;
    for (int e = threadIdx.x; e < nx * ny; e += kThreads) {
        const int y = e / nx, x = e - y * nx;
        // every window point lies on the mesh by the plan's reach; the clamp only guards the address
        const int gx = min(max(x0 + x, 0), Kx - 1), gy = min(max(y0 + y, 0), Ky - 1);
        const T2 *col = G + (size_t)gy * Kz * Kx + gx;
        T ar[kRows], ai[kRows];
#pragma unroll
        for (int r = 0; r < kRows; r++) ar[r] = ai[r] = (T)0;
        for (int zb = 0; zb < nz8; zb += kZ) {  // kZ loads of a class in flight
            T vr[kZ], vi[kZ];
#pragma unroll
            for (int z = 0; z < kZ; z++) vr[z] = vi[z] = (T)0;
            for (int f = 0; f < P.nfield; f++) {
                const T2 *g = col + f * fstride;
                const T c = (T)wf[f];
                T2 v[kZ];
#pragma unroll
                for (int z = 0; z < kZ; z++) v[z] = g[(size_t)min(max(z0 + zb + z, 0), Kz - 1) * Kx];
#pragma unroll
                for (int z = 0; z < kZ; z++) {
                    vr[z] = fma(c, v[z].x, vr[z]);
                    vi[z] = fma(c, v[z].y, vi[z]);
                }
            }
#pragma unroll
            for (int z = 0; z < kZ; z++)
#pragma unroll
                for (int r = 0; r < kRows; r++) {
                    ar[r] = fma(wzt[zb + z][r], vr[z], ar[r]);
                    ai[r] = fma(wzt[zb + z][r], vi[z], ai[r]);
                }
        }
#pragma unroll
        for (int r = 0; r < kRows; r++)
            if (r < nrow) {
                T2 v;
                v.x = ar[r];
                v.y = ai[r];
                planes[r * plane + y * sx + x] = v;
            }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < nn; e += kThreads) {
        const int r = e / ncol, c = e - r * ncol, j = B.j0 + r, k = k0 + c;
        if (2 * j == half && k >= half) continue;  // the equator's second half turn: antipodes of the first
        // the window's coefficients are read from LDS for every node: kept in registers
        // across the loop, FP64's 144 would spill
        int zero = 0;
        asm volatile("" : "+v"(zero));
        const T *cf = coef + zero;
        double zx, zy;
        const int ix = place_x(r, c, zx) - x0, iy = place_y(r, c, zy) - y0;
        T wx[W];
        window_values<T, W>(cf, (T)zx, [&](int l, T v) { wx[l] = v; });
        const T ty = (T)zy, tt = ty * ty;
        const T2 *p = planes + r * plane + iy * sx + ix;
        T ax = (T)0, ay = (T)0;
        // the rows l and W - 1 - l of the window together (window_values' even and odd parts)
#pragma unroll kYUnroll
        for (int l = 0; l < W / 2; l++) {
            T we = cf[l * nc + nc - 2], wo = cf[l * nc + nc - 1];
#pragma unroll
            for (int d = nc - 4; d >= 0; d -= 2) {
                we = fma(we, tt, cf[l * nc + d]);
                wo = fma(wo, tt, cf[l * nc + d + 1]);
            }
            T ux0 = (T)0, uy0 = (T)0, ux1 = (T)0, uy1 = (T)0;
#pragma unroll
            for (int lx = 0; lx < W; lx++) {
                const T2 v = p[l * sx + lx], u = p[(W - 1 - l) * sx + lx];
                ux0 = fma(wx[lx], v.x, ux0);
                uy0 = fma(wx[lx], v.y, uy0);
                ux1 = fma(wx[lx], u.x, ux1);
                uy1 = fma(wx[lx], u.y, uy1);
            }
            const T w0 = fma(ty, wo, we), w1 = fma(-ty, wo, we);
            ax = fma(w0, ux0, fma(w1, ux1, ax));
            ay = fma(w0, uy0, fma(w1, uy1, ay));
        }
        double re = (double)ax * scale, im = (double)ay * scale;
        if (P.shifted) {  // sources placed about the mesh's centre: e^{i q.c}
            double s, co;
            sincos(rs[r] * cc[c] * P.ax[0].c + rs[r] * cn[c] * P.ax[1].c + rz[r] * P.ax[2].c, &s, &co);
            const double t0 = re * co - im * s;
            im = im * co + re * s;
            re = t0;
        }
        T4 v;
        v.x = (T)re;
        v.y = (T)im;
        v.z = (T)0;
        v.w = (T)0;
        grid[index_from_indices(shell, j, k)] = v;
        v.y = -v.y;
        grid[index_from_indices(shell, half - j, k + half >= n6 ? k - half : k + half)] = v;
    }
}

// ------------------------------------------------------------------ plan (host)
namespace {

constexpr int kSpreadMixed = 10, kInterpMixed = 8, kSpread64 = 16, kInterp64 = 16;
constexpr double kSigmaMixed = 2.0, kSigma64 = 2.5;
// interpolation patches: rows at most, and the sides down the rows and along them in
// frequency steps (mesh_lds bounds the (x, y) planes they need, kPatchZ the z points)
constexpr int kRowsMixed = 16, kRows64 = 12, kThreadsMixed = 256, kThreads64 = 512;
constexpr double kDownMixed = 6.0, kAlongMixed = 10.0, kDown64 = 3.0, kAlong64 = 6.0;
// (a column's z points are rounded up to the 8 or 4 that mesh_interp loads at a time)
static_assert((int)kDownMixed + 1 + kInterpMixed + 7 <= kPatchZ && (int)kDown64 + 1 + kInterp64 + 3 <= kPatchZ,
              "the rows' z windows fit wzt");

int round_up(int v, int m) { return (v + m - 1) / m * m; }

// nodes of the Gauss-Legendre rule that integrates e^{i q t} over |t| <= len / 2 to
// tol (its error term, a = q len / 2), or 0
int gl_nodes(double a, double tol) {
    for (int m = 2; m <= kMaxGl; m++) {
        // 2^(2m+1) (m!)^4 / ((2m+1) ((2m)!)^3) a^(2m)
        const double e = (2.0 * m + 1.0) * std::log(2.0) + 4.0 * std::lgamma(m + 1.0) - std::log(2.0 * m + 1.0) -
                         3.0 * std::lgamma(2.0 * m + 1.0) + 2.0 * m * std::log(std::max(a, 1e-30));
        if (e < std::log(tol)) return m + 1;
    }
    return 0;
}

}  // namespace

bool mesh_plan(const MeshSources &S, int N, double step, bool fp64, int nion, size_t room, MeshPlan &P, MeshSizes &Z) {
    if (!S.ok || S.nfield < 1 || S.nfield > kMeshFields) return false;
    const int WS = fp64 ? kSpread64 : kSpreadMixed, WI = fp64 ? kInterp64 : kInterpMixed;
    P = MeshPlan{};
    P.nfield = S.nfield;
    P.boxes = S.npieces > 0;
    P.nion = nion;
    P.step = step;
    const double Q = (double)N * step, sigma = fp64 ? kSigma64 : kSigmaMixed;
    P.shifted = 0;
    double points = 1.0;
    for (int a = 0; a < 3; a++) {
        MeshAxis &A = P.ax[a];
        // about the origin where that costs little (no shift phase at the nodes), else about the middle
        const double far = std::max(std::fabs(S.lo[a]), std::fabs(S.hi[a])), mid = 0.5 * (S.lo[a] + S.hi[a]);
        const double half = 0.5 * (S.hi[a] - S.lo[a]);
        const bool centred = far <= 1.15 * half + 0.05;
        A.c = centred ? 0.0 : mid;
        if (!centred) P.shifted = 1;
        // frequency step: |r| dk <= pi / sigma for every source (a small structure's mesh
        // keeps at least two steps per Q)
        const double X = std::max(centred ? far : half, kPi / (4.0 * Q)) * (1.0 + 1e-9);
        A.dk = kPi / (sigma * X);
        A.dkinv = 1.0 / A.dk;
        A.dk = 1.0 / A.dkinv;
        const double steps = std::ceil(Q / A.dk + 0.5 * WI) + 1.0;
        if (!(steps > 0.0 && steps < 65536.0)) return false;  // (also extents that are no sizes of a structure)
        const int reach = (int)steps;
        const double K = reach * A.dk;
        A.h = kPi / (sigma * K) * (1.0 - 1e-9);
        A.hinv = 1.0 / A.h;
        // the windows' places come from hinv and dkinv; the exponentials follow them exactly
        const long double turn = 1.0L / (4.0L * 3.141592653589793238462643383279502884L * A.hinv * A.dkinv);
        A.turn = (double)turn;
        A.turn_lo = (double)(turn - A.turn);
        const double span = 2.0 * X / A.h + WS + 2.0;
        if (!(span < 4096.0)) return false;
        A.m = round_up((int)std::ceil(span), a == 2 ? 16 : 8);
        A.x0 = -0.5 * (A.m - 1) * A.h;
        // the canonical half has q_z >= 0
        A.n0 = a == 2 ? WI / 2 + 1 : reach;
        A.k = A.n0 + reach + 1;
        points *= A.m;
        P.cell0[a] = S.cell0[a] - A.c;
        P.ncell[a] = S.ncell[a];
        P.cell_inv[a] = S.cell_inv[a];
        P.box_half[a] = S.piece_half[a];
    }
    P.wp_box = 0;
    P.gl = 1;
    if (P.boxes) {
        double ext = 0.0, phase = 0.0;
        for (int a = 0; a < 3; a++) {
            ext = std::max(ext, 2.0 * S.piece_half[a] * P.ax[a].hinv);
            phase = std::max(phase, Q * S.piece_half[a]);
        }
        P.gl = gl_nodes(phase, fp64 ? 1e-16 : 1e-10);
        if (P.gl == 0 || P.gl > kMaxGl || !(ext < 64.0)) return false;
        P.wp_box = WS + (int)std::ceil(ext) + 1;
    }
    // tables: [spread window | 1/phihat spread | interpolation window | 1/phihat interpolation | quadrature]
    if (P.wp_box > kMaxWp) return false;
    P.t_spread = 0;
    P.t_sinv = WS * (WS + 2);
    P.t_interp = P.t_sinv + kInvDeg;
    P.t_iinv = P.t_interp + WI * (WI + 2);
    P.t_gl = P.t_iinv + kInvDeg;
    Z.tab = P.t_gl + 2 * P.gl;
    const size_t nf = S.nfield, mx = P.ax[0].m, my = P.ax[1].m, mz = P.ax[2].m, fx = P.ax[0].k, fy = P.ax[1].k,
                 fz = P.ax[2].k;
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    size_t o = 0;
    auto take = [&](size_t b) {
        const size_t at = o;
        o += al(b);
        return at;
    };
    Z.wb = take((size_t)S.npieces * 3 * P.wp_box * 8);
    Z.bb = take((size_t)S.npieces * 16);
    Z.e0 = take(2 * fx * mx * 8);
    Z.e1 = take(2 * fy * my * 8);
    Z.e2 = take(2 * fz * mz * 8);
    Z.g = take(nf * fx * fy * fz * (fp64 ? 16 : 8));
    // two buffers used in turn by as many classes at a time as fit `room`
    // (and slices of a brick's sources, two batches or more each on average)
    // bricks that read a source: those its window reaches, and those that only its cell reaches
    // (cells of kMeshCell are in the fit of mesh_pays; a long axis has larger ones)
    double reach = 1.0;
    for (int a = 0; a < 3; a++) {
        const double brick = a == 2 ? 16.0 : 8.0, cell = std::max(0.0, 1.0 / S.cell_inv[a] - kMeshCell) * P.ax[a].hinv;
        reach *= std::min((WS + brick + cell) / brick, P.ax[a].m / brick);
    }
    const double batches = (double)std::max(S.natoms, S.npieces) * reach / (points / 1024.0) / 256.0;
    Z.slices = (int)std::max(1.0, std::min(4.0, batches / 2.0));
    size_t b0, b1 = al(fz * mx * my * 16);
    for (;; Z.slices--) {
        b0 = al(std::max(Z.slices * mx * my * mz * 8, fy * fz * mx * 16));
        if (o + b0 + b1 <= room) break;
        if (Z.slices == 1) return false;
    }
    Z.group = (int)std::min(nf, (room - o) / (b0 + b1));
    Z.b0 = take(Z.group * b0);
    Z.b1 = take(Z.group * b1);
    Z.bytes = o;
    const double dk = std::min(P.ax[0].dk, std::min(P.ax[1].dk, P.ax[2].dk));
    Z.s = step * (kPi / 3.0) / dk;
    // the kernels' work, for mesh_pays
    Z.nodes = (double)half_base(N + 1);
    Z.pairs = (double)(S.natoms + S.npieces) * reach;
    Z.dft = (double)nf * ((double)mx * my * mz * fz * 4.0 + (double)mx * my * fz * fy * 8.0 + (double)mx * fy * fz * fx * 8.0);
    // interpolation patches: mesh_bands cuts rows x columns of about these sides
    const double down = fp64 ? kDown64 : kDownMixed, along = fp64 ? kAlong64 : kAlongMixed;
    const double rows = std::min((double)(fp64 ? kRows64 : kRowsMixed), std::floor(down / Z.s) + 1.0);
    const double cols = std::min((double)kPatchCols, std::floor(along / (0.7 * Z.s)) + 1.0);
    Z.tiles = Z.nodes / (rows * cols) + 4.0 * N;
    return true;
}

// LDS of the interpolation's (x, y) planes.  A patch's rows span at most (rows - 1) s steps of
// q sin(theta) and its widest row an arc of at most `along` steps, so two of its nodes are at
// most hypot of the two apart in any direction of the plane (the chord between radii a and b at
// an angle d is (a - b)^2 + 4 a b sin^2(d / 2) squared), and their windows' first points one
// more than the whole steps of that.
size_t mesh_lds(const MeshSizes &Z, bool fp64) {
    const int W = fp64 ? kInterp64 : kInterpMixed, most = fp64 ? kRows64 : kRowsMixed;
    const double down = fp64 ? kDown64 : kDownMixed, along = fp64 ? kAlong64 : kAlongMixed;
    const int rows = (int)std::min((double)most, std::floor(down / Z.s) + 1.0);
    const int n = (int)std::floor(std::hypot((rows - 1) * Z.s, along)) + 2 + W;
    return (size_t)rows * n * (n | 1) * (fp64 ? 16 : 8);
}

void mesh_bands(const MeshPlan &P, const MeshSizes &Z, int N, bool fp64, std::vector<MeshBand> &bands, int &ntiles) {
    const double down = fp64 ? kDown64 : kDownMixed, along = fp64 ? kAlong64 : kAlongMixed;
    const int most = fp64 ? kRows64 : kRowsMixed;
    bands.clear();
    ntiles = 0;
    for (int i = 1; i <= N; i++) {
        const int rows = 3 * i / 2 + 1, n6 = 6 * i;
        int nr = (int)std::min((double)most, std::floor(down / Z.s) + 1.0);
        const int nb = (rows + nr - 1) / nr;
        nr = (rows + nb - 1) / nb;
        for (int j0 = 0; j0 < rows; j0 += nr) {
            MeshBand b;
            b.shell = i;
            b.j0 = j0;
            b.rows = std::min(nr, rows - j0);
            // columns at the band's widest row, Z.s sin(theta) apart
            const double w = Z.s * std::sin(kPi * (j0 + b.rows - 1) / (3.0 * i));
            int nc = w > 0.0 ? (int)std::min((double)n6, std::floor(along / w) + 1.0) : n6;
            nc = std::max(1, std::min(nc, kPatchCols));
            const int nt = (n6 + nc - 1) / nc;
            b.cols = (n6 + nt - 1) / nt;
            b.tile0 = ntiles;
            ntiles += (n6 + b.cols - 1) / b.cols;
            bands.push_back(b);
        }
    }
}

void mesh_tables(const MeshPlan &P, bool fp64, double *tab) {
    const double sigma = fp64 ? kSigma64 : kSigmaMixed;
    const Window &s = window(fp64 ? kSpread64 : kSpreadMixed, sigma, false), &i = window(fp64 ? kInterp64 : kInterpMixed, sigma, !fp64);
    std::copy(s.coef.begin(), s.coef.end(), tab + P.t_spread);
    std::copy(s.inv, s.inv + kInvDeg, tab + P.t_sinv);
    std::copy(i.coef.begin(), i.coef.end(), tab + P.t_interp);
    std::copy(i.inv, i.inv + kInvDeg, tab + P.t_iinv);
    std::vector<long double> x, w;
    gauss_legendre(P.gl, x, w);
    std::copy(x.begin(), x.end(), tab + P.t_gl);
    std::copy(w.begin(), w.end(), tab + P.t_gl + P.gl);
}

// GPU time of the builders in us, fitted to 77 builds of 500..200,000 atoms (with and
// without a hydration layer) at grids 20..250 on MI355X, each within 20 % of its
// measurement near the line: mixed 2,000 atoms at grid 60 86 us direct, 66 through the
// mesh; 500 atoms at grid 40 47 and 50; 40,000 atoms at grid 250 25,249 and 406; FP64
// 2,000 atoms at grid 100 874 and 190.  The mesh builder takes a build it shortens by 50 us
// or more: below that its ten small launches leave less of the device to other work.
bool mesh_pays(const MeshPlan &P, const MeshSizes &Z, int N, double sources, bool fp64) {
    const double terms = (double)half_base(N + 1) * sources;
    const double passes = std::ceil((double)P.nfield / Z.group), tiles = (double)Z.tiles * P.nfield;
    const double direct = fp64 ? 150.0 + 7.0e-7 * terms : 46.0 + 1.1e-7 * terms;
    const double mesh = fp64 ? 49.0 + 24.0 * passes + 6.3e-5 * Z.nodes + 3.6e-4 * Z.pairs + 1.2e-8 * Z.dft + 1.7e-2 * tiles
                             : 32.0 + 25.0 * passes + 4.4e-6 * Z.nodes + 3.3e-4 * Z.pairs + 1.2e-8 * Z.dft + 9.4e-3 * tiles;
    return mesh + 50.0 < direct;
}

template <typename T, typename T2, typename T4, int WS, int WI, int kRows, int kThreads>
static void launch_mesh_t(const MeshJob &J, hipStream_t s) {
    const MeshPlan &P = J.plan;
    char *w = (char *)J.work;
    double *wb = (double *)(w + J.z.wb);
    int4 *bb = (int4 *)(w + J.z.bb);
    double *E0 = (double *)(w + J.z.e0), *E1 = (double *)(w + J.z.e1), *E2 = (double *)(w + J.z.e2);
    if (J.npieces > 0)
        mesh_weights<WS><<<(unsigned)((J.npieces + 63) / 64), 192, 192 * (size_t)(P.wp_box | 1) * 8, s>>>(
            P, J.pieces, J.lens, J.npieces, P.gl, P.wp_box, J.tab, wb, bb);
    const int mx = P.ax[0].m, my = P.ax[1].m, mz = P.ax[2].m, fx = P.ax[0].k, fy = P.ax[1].k, fz = P.ax[2].k;
    int most = 0;
    for (int a = 0; a < 3; a++) most = std::max(most, P.ax[a].m * P.ax[a].k);
    mesh_twiddles<<<dim3((most + 255) / 256, 3), 256, 0, s>>>(P, J.tab, E0, E1, E2);
    double *mesh = (double *)(w + J.z.b0);
    double2 *b0 = (double2 *)(w + J.z.b0), *b1 = (double2 *)(w + J.z.b1);
    for (int f = 0; f < P.nfield; f += J.z.group) {
        const int nf = std::min(J.z.group, P.nfield - f);
        T2 *G = (T2 *)(w + J.z.g) + (size_t)f * fx * fy * fz;
        auto grid = [&](int rows, int nk) { return dim3((rows + 63) / 64, (nk + 31) / 32, nf); };
        mesh_spread<WS><<<dim3((mx / 8) * (my / 8) * (mz / 16), nf * J.z.slices), 1024, 0, s>>>(P, f, J.z.slices, J.atoms, J.cells, J.tab, wb, bb, mesh);
        mesh_dft<double, double2, false><<<grid(mx * my, fz), 256, 0, s>>>(mesh, b1, E2, mz, fz, mx * my, J.z.slices);
        mesh_dft<double2, double2, false><<<grid(fz * mx, fy), 256, 0, s>>>(b1, b0, E1, my, fy, fz * mx, 1);
        mesh_dft<double2, T2, true><<<grid(fy * fz, fx), 256, 0, s>>>(b0, G, E0, mx, fx, fy * fz, 1);
    }
    mesh_interp<T, T2, T4, WI, kRows, kThreads><<<J.ntiles, kThreads, mesh_lds(J.z, sizeof(T) == 8), s>>>(P, J.bands, J.nbands, J.ff, J.fion, J.tab,
                                                                       (const T2 *)(w + J.z.g), (T4 *)J.grid, J.scale);
}

void launch_mesh(const MeshJob &J, bool fp64, hipStream_t s) {
    if (fp64)
        launch_mesh_t<double, double2, double4, kSpread64, kInterp64, kRows64, kThreads64>(J, s);
    else
        launch_mesh_t<float, float2, float4, kSpreadMixed, kInterpMixed, kRowsMixed, kThreadsMixed>(J, s);
}

}  // namespace dplus

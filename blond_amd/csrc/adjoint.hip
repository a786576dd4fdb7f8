// Differentiable tracking on the MI355X: forward turns, checkpoints and the
// hand-written reverse (adjoint) pass.
//
// The map per turn t (the intensity map of the fused engine with a smooth
// profile), in one of two forms chosen at compile time (MAP):
//
// MAP = kMapReference, the reference's own functions:
//   p_t     = smooth_histogram(dt_t)   histogram.cpp:75-132 with its quirk:
//                            f = (dt - cut_left) inv_bw, k = (int) f,
//                            d = f - k; bin k gets 0.5 - d, bin
//                            k2 = (int)(f + 1) (d > 1/2) or (int)(f - 1)
//                            gets 0.5 + d; particles outside
//                            [cut_left + bw/2, cut_right - bw/2] dropped
//   e1      = linear_interp_kick(dt, dE, V_t, bin_centers, q, 0)
//                            (linear_interp_kick.cpp:21-71: slope and
//                            intercept of each bin, formed per workgroup in
//                            LDS from V_t in the reference's order)
//   The weights are piecewise linear in dt, with jumps where a particle
//   crosses a bin centre or edge; the reverse pass uses their derivatives on
//   the pieces: d p[k]/d dt = -inv_bw, d p[k2]/d dt = +inv_bw, d kick/d dt =
//   the bin's slope, d kick/d V[k], V[k+1] = q (1 - s), q s with
//   s = (dt - bc[k]) inv_bw_bc.
//
// MAP = kMapSpline, a variant with continuous first derivatives:
//   p_t     = D(dt_t)        quadratic B-spline deposit on bin centres: a
//                            particle at bin-centre coordinate
//                            u = (dt - cut_left) inv_bw - 1/2 = k + d,
//                            k = round(u), adds (1/2 - d)^2 / 2, 3/4 - d^2,
//                            (1/2 + d)^2 / 2 to bins k-1, k, k+1
//   e1      = dE + q sum_b V_t[b] w_b(dt)   the same spline weights
//
// Both:
//   V_t     = -scale * (g conv p_t)[:ns],  g = irfft(Z, n_fft) (circular,
//                            as the FFT route of impedance.py:457-489)
//   e2      = e1 + q sum_j V_j sin(w_j dt + phi_j) + acc   (kick.cpp:16-35)
//   dt_{t+1} = dt + coeff_{t+1} e2,  dE_{t+1} = e2          (drift.cpp "simple")
// and the loss depends on p_T.
//
// Reverse turn t, per particle (state at t recomputed from a checkpoint):
//   lx <- lx + sum_b lp_{t+1}[b] dp_b/d dt                    deposit of p_{t+1}
//   le2 = le + coeff lx
//   lx <- lx + le2 (q sum_j V_j w_j cos(.) + d kick / d dt)   RF + induced kick
//   lV_t[b] += le2 d kick / d V_t[b]                           induced kick
//   dL/dV_j += le2 q sin(.),  dL/dphi_j += le2 q V_j cos(.)
//   le <- le2
// then, once per turn: lp_t = -scale * (g corr lV_t); and once per pass
// corr[m] = sum_t sum_i lV_t[i] p_t[(i - m) mod n_fft], from which the host
// forms dL/dZ-parameters as -scale * sum_m irfft(dZ/dtheta)[m] corr[m].
//
// Traffic per macroparticle-turn: 32 B forward, 8 B recompute (the dt of a
// segment's states are written; the particles stay in registers), 48 B reverse
// (dt_t and dt_{t+1} read, two adjoints read and written).
//
// One launch a turn in each direction up to kAdjFuseSlices slices: every
// particle workgroup forms the turn's slice-axis product (V_t from p_t, or
// lp_{t+1} from lV_{t+1}) for itself on the matrix cores in its prologue,
// while its first particles are on their way, and the first workgroup
// publishes it.  The accumulators a turn's particles add into are used in
// rotation (three): turn t reads one, adds into the next and clears the one
// the launch before it read.
#include <math.h>
#include <string.h>

#include <vector>

#include "adjoint.h"
#include "blmi_common.h"
#include "particles.h"

namespace blmi {

int smooth_scale_bits(int64_t n);

constexpr int kAdjMaxRf = 4;
constexpr int kAdjBlock = 1024;

struct AdjArgs {
    int n_rf;
    double charge;
    const double *rf;  // [turn][3][n_rf]
    const double *acc;
    const DriftCoeffs<double> *drift;
    int ns;
    double cut_left, inv_bw_cut, fix_scale;
    double *vt;          // [turn][ns] induced voltage V_t
    unsigned long long *dep;  // [kAdjRing][copies][ns] deposit of p_t: slot t % kAdjRing
    double *lv;               // [kAdjRing][copies][ns] lV_t: slot t % kAdjRing
    double *lp;               // [ns]
    double *gpart;            // [grid][2 n_rf], added to by every reverse turn
    double *prof;             // [turn][ns] p_t
    double *lvh;              // [turn][ns] lV_t
    const double *g;          // [n_fft] wake
    int n_fft;
    double scale;
    // the reference map: smooth_histogram's range and the interpolation's
    // bin centres (histogram.cpp:82-85, linear_interp_kick.cpp:33)
    double lo, hi;
    const double *bc;  // [ns]
    double bc0, inv_bw_bc;
};

constexpr int kMapSpline = 0;
constexpr int kMapReference = 1;

// Quadratic B-spline: u = (x - cut_left) inv_bw - 1/2 = k + d, k = round(u),
// d in [-1/2, 1/2); weights of bins k-1, k, k+1 and their u-derivatives.
// k = kNoBin when none of the three bins is inside [0, ns).
constexpr int kNoBin = -1000000;
__device__ __forceinline__ int spline(double x, const AdjArgs &a, double w[3], double dw[3]) {
    const double u = (x - a.cut_left) * a.inv_bw_cut - 0.5;
    const double kf = floor(u + 0.5);
    if (!(kf >= -1.0 && kf <= (double)a.ns)) return kNoBin;  // also NaN
    const double d = u - kf;
    const double l = 0.5 - d, r = 0.5 + d;
    w[0] = 0.5 * l * l;
    w[1] = 0.75 - d * d;
    w[2] = 0.5 * r * r;
    dw[0] = -l;
    dw[1] = -2.0 * d;
    dw[2] = r;
    return (int)kf;
}

// A weight in fixed point, |w * scale| < 2^51: adding 1.5 * 2^52 leaves the
// nearest integer (ties to even, as __double2ll_rn) in the low mantissa bits.
// Two additions in place of the ten instructions of a double to 64-bit
// integer conversion.
__device__ __forceinline__ unsigned long long to_fixed(double w, double scale) {
    constexpr double kMagic = 6755399441055744.0;  // 1.5 * 2^52
    const double m = w * scale + kMagic;
    return (unsigned long long)(__double_as_longlong(m) - __double_as_longlong(kMagic));
}

__device__ __forceinline__ void deposit_lds(unsigned long long *h, double x, const AdjArgs &a) {
    double w[3], dw[3];
    const int k = spline(x, a, w, dw);
    if (k == kNoBin) return;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int b = k - 1 + q;
        if (b >= 0 && b < a.ns)
            atomicAdd(&h[b], to_fixed(w[q], a.fix_scale));
    }
}

// smooth_histogram's two bins of a particle (histogram.cpp:100-113): bin k
// gets 0.5 - d, bin k2 gets 0.5 + d.  False outside [lo, hi] (NaN
// included); a bin outside [0, ns) (a rounding corner at hi) is skipped by
// the callers.
__device__ __forceinline__ bool smooth_bins(double x, const AdjArgs &a, int &k, int &k2,
                                            double &d) {
    if (!(x >= a.lo && x <= a.hi)) return false;
    const double f = (x - a.cut_left) * a.inv_bw_cut;
    k = (int)f;
    d = f - (double)k;
    k2 = d > 0.5 ? (int)(f + 1.0) : (int)(f - 1.0);
    return true;
}

__device__ __forceinline__ void deposit_smooth(unsigned long long *h, double x, const AdjArgs &a) {
    int k, k2;
    double d;
    if (!smooth_bins(x, a, k, k2, d)) return;
    if (k >= 0 && k < a.ns)
        atomicAdd(&h[k], to_fixed(0.5 - d, a.fix_scale));
    if (k2 >= 0 && k2 < a.ns)
        atomicAdd(&h[k2], to_fixed(0.5 + d, a.fix_scale));
}

template <int MAP>
__device__ __forceinline__ void deposit(unsigned long long *h, double x, const AdjArgs &a) {
    if (MAP == kMapReference) deposit_smooth(h, x, a);
    else deposit_lds(h, x, a);
}

// linear_interp_kick.cpp:44-48 on V_t (acceleration 0, as
// TotalInducedVoltage.track passes it): (slope, intercept) of bin b, in the
// reference's order of operations.
__device__ __forceinline__ double2 interp_pair(double v0, double v1, double bcb,
                                               const AdjArgs &a) {
    const double k = a.charge * (v1 - v0) * a.inv_bw_bc;
    return make_double2(k, (a.charge * v0 - bcb * k) + 0.0);
}

// linear_interp_kick.cpp:56-63: the bin a particle is kicked by, or -1 (a
// signed range test in place of the reference's unsigned cast: negative,
// NaN and last-bin positions get no kick).
__device__ __forceinline__ int interp_bin(double x, const AdjArgs &a) {
    const double f = floor((x - a.bc0) * a.inv_bw_bc);
    return (f >= 0.0 && f < (double)(a.ns - 1)) ? (int)f : -1;
}

// into the deposit of turn t's profile
__device__ __forceinline__ void deposit_flush(unsigned long long *h, const AdjArgs &a, int t) {
    __syncthreads();
    unsigned long long *out =
        a.dep + ((size_t)(t % kAdjRing) * kAdjCopies + blockIdx.x % kAdjCopies) * a.ns;
    for (int b = threadIdx.x; b < a.ns; b += blockDim.x)
        if (h[b]) atomic_add_agent(&out[b], h[b]);
}

template <int MAP>
__global__ void __launch_bounds__(kAdjBlock) adj_deposit_kernel(const double *__restrict__ x,
                                                                int64_t n, AdjArgs a) {
    extern __shared__ unsigned long long hdep[];
    for (int b = threadIdx.x; b < a.ns; b += blockDim.x) hdep[b] = 0ull;
    __syncthreads();
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        deposit<MAP>(hdep, x[i], a);
    deposit_flush(hdep, a, 0);
}

// q sum_b V[b] w_b(x) and (with D) its u-derivative, V in LDS
__device__ __forceinline__ double induced_kick(const double *V, double x, const AdjArgs &a,
                                               double *dkick, double w[3], int &k) {
    double dw[3];
    k = spline(x, a, w, dw);
    double s = 0.0, ds = 0.0;
    if (k != kNoBin) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int b = k - 1 + q;
            if (b >= 0 && b < a.ns) {
                s = s + V[b] * w[q];
                ds = ds + V[b] * dw[q];
            }
        }
    }
    if (dkick) *dkick = a.charge * ds * a.inv_bw_cut;
    return a.charge * s;
}

// ---------------------------------------------------------------------------
// Slice-axis products in a particle workgroup's prologue
// ---------------------------------------------------------------------------
// out[i] = sum_j g[(DIR (i - j)) mod n_fft] x[j], i, j < ns, as a matrix
// product for the FP64 matrix cores: with i = 16 a + b and j = 16 c + d,
//   out[b, a] = sum over (m, d) of G[16 m + b - d] X[16 (a - m) + d],
// a 16-row matrix of G (rows b, columns (m, d)) times one of shifted X
// (columns a), 16 x 16 outputs a tile.  A tile's rows of m are split over the
// wavefronts that share it and their sums added through LDS.  X is padded
// with zeros (15 chunks of 16 on either side, 17 words a chunk: the lanes of
// a column read at stride 17, on distinct banks), G is zero beyond +-(ns - 1),
// so half the products of 256 slices are zeros, and still the product takes
// under a microsecond: read from LDS by vector code, every multiply would need
// two LDS reads.
typedef double MfmaD4 __attribute__((ext_vector_type(4)));
__host__ __device__ __forceinline__ int prod_chunks(int ns) { return (ns + 15) / 16; }
__host__ __device__ __forceinline__ int prod_tiles(int ns) { return (prod_chunks(ns) + 15) / 16; }
__host__ __device__ __forceinline__ int prod_g_words(int ns) {
    return 256 * prod_tiles(ns) + 16 * prod_chunks(ns);
}
__host__ __device__ __forceinline__ int prod_x_words(int ns) {
    return 17 * (prod_chunks(ns) + 30);
}
constexpr int kAdjWaves = kAdjBlock / 64;
// words of a tile of sums, stored by columns of 16 + 1: the lanes of a row
// write at stride 17 and consecutive outputs are consecutive words (at stride
// 16 the bank conflicts of these sums took 4 us of a launch)
constexpr int kProdTile = 17 * 16;
__host__ __device__ __forceinline__ int prod_words(int ns) {
    return prod_g_words(ns) + prod_x_words(ns) + kProdTile * kAdjWaves;
}
// a chunk's 17th word is never read
__device__ __forceinline__ int prod_x_at(int j) { return 17 * ((j >> 4) + 15) + (j & 15); }

// Largest slice count a prologue forms the product for (one G word and one
// slice a thread, at most two tiles); above it the slice axis has launches of
// its own.  1e6 macroparticles, 256 slices: forward 12.9 us a turn against 10.3
// and 5.2 for the particle and the slice launch, reverse 17.3 (15.6 since it
// reads dt_{t+1}) against 13.7 and 5.8, and a launch gap of about 1.4 us less in each; of the prologue about 2 us
// are the product.  It grows with the square of the slices on every CU: four
// times the matrix work at 512, and at 1024 more (8 us) than the slice launch.
constexpr int kAdjFuseSlices = 512;

// This thread's word of G (read early: nothing here waits for it).
template <int DIR>
__device__ __forceinline__ double prod_load_g(const AdjArgs &a) {
    const int k = (int)threadIdx.x - 16 * prod_chunks(a.ns);
    const int ka = DIR > 0 ? k : -k;
    const bool in = k > -a.ns && k < a.ns;
    const int m = ka < 0 ? ka + a.n_fft : ka;  // ns <= n_fft
    const double v = a.g[in ? m : 0];
    return in ? v : 0.0;
}

// G (a word a thread) and X (slice threadIdx.x's x, zeros around) into LDS.
__device__ __forceinline__ void prod_put(double *lds, double g, double x, const AdjArgs &a) {
    const int gw = prod_g_words(a.ns), xw = prod_x_words(a.ns);
    double *X = lds + gw;
    if ((int)threadIdx.x < gw) lds[threadIdx.x] = g;
    const int lo = prod_x_at(0), hi = prod_x_at(a.ns);
    for (int w = threadIdx.x; w < xw; w += kAdjBlock)
        if (w < lo || w >= hi) X[w] = 0.0;
    if ((int)threadIdx.x < a.ns) X[prod_x_at(threadIdx.x)] = x;
}

// After a barrier: this wavefront's share of the product, into LDS.
__device__ __forceinline__ void prod_run(double *lds, const AdjArgs &a) {
    const int A = prod_chunks(a.ns), Q = prod_tiles(a.ns);
    const double *G = lds + 16 * A;
    const double *X = lds + prod_g_words(a.ns);
    double *part = lds + prod_g_words(a.ns) + prod_x_words(a.ns);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int per = kAdjWaves / Q;  // wavefronts a tile
    const int q = wid / per, r0 = wid % per;
    MfmaD4 c = {0.0, 0.0, 0.0, 0.0};
    const int l16 = lane & 15, k4 = lane >> 4;
    const double *gp = G + l16 - k4;                      // row b = l16, d = k4 + 4 s
    const double *xp = X + 17 * (16 * q + l16 + 15) + k4;  // column a = 16 q + l16
    for (int m = 16 * q - (A - 1) + r0; m <= 16 * q + 15; m += per) {
        double gv[4], xv[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            gv[s] = gp[16 * m - 4 * s];
            xv[s] = xp[4 * s - 17 * m];
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(gv[s], xv[s], c, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) part[wid * kProdTile + 17 * l16 + 4 * r + k4] = c[r];
}

// After another barrier: output i, -(scale * product).
__device__ __forceinline__ double prod_out(const double *lds, int i, const AdjArgs &a) {
    const int per = kAdjWaves / prod_tiles(a.ns);
    const double *part = lds + prod_g_words(a.ns) + prod_x_words(a.ns);
    const int ca = i >> 4, b = i & 15;
    const double *pp = part + (ca >> 4) * per * kProdTile + 17 * (ca & 15) + b;
    double v = 0.0;
#pragma unroll 8
    for (int w = 0; w < per; ++w) v += pp[w * kProdTile];
    return -(a.scale * v);
}

// Turn t's slot of a ring of accumulators: the sum of its copies (every copy
// loaded before the sum: one memory round trip).
template <typename V>
__device__ __forceinline__ V ring_sum(const V *ring, int t, int ns, int j) {
    const V *in = ring + (size_t)(t % kAdjRing) * kAdjCopies * ns + j;
    V v[kAdjCopies], s = V(0);
#pragma unroll
    for (int c = 0; c < kAdjCopies; ++c) v[c] = in[(size_t)c * ns];
#pragma unroll
    for (int c = 0; c < kAdjCopies; ++c) s += v[c];
    return s;
}
// Clears this workgroup's share of turn t's slot.
template <typename V>
__device__ __forceinline__ void ring_clear(V *ring, int t, int ns) {
    V *out = ring + (size_t)(t % kAdjRing) * kAdjCopies * ns;
    const int total = kAdjCopies * ns;
    for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < total; j += gridDim.x * blockDim.x)
        out[j] = V(0);
}

// ---------------------------------------------------------------------------
// Forward turn t: (xi, ei) -> (xo, eo) (may alias), with p_{t+1} deposited.
// FUSE: V_t is formed here from p_t's deposit; else it is read from a.vt.
// A thread takes pairs of macroparticles (16-byte loads; with an odd count
// the arrays' pad slot is the last pair's second, moved but not deposited),
// loaded two pairs ahead in two register slots, the first two before the
// prologue.
// LDS: the deposit (u64), the interpolation table (reference map), V_t, and
// with FUSE the product's words.
// ---------------------------------------------------------------------------
static size_t adj_turn_lds(int ns, bool fuse) {
    return sizeof(double) * (4 * (size_t)ns + (fuse ? prod_words(ns) : 0));
}

// The per-turn constants of the particle step, in registers: read before the
// prologue's barriers, which no load is moved across.
struct TurnConst {
    double V[kAdjMaxRf], w[kAdjMaxRf], phi[kAdjMaxRf];
    double acc, coeff;
    __device__ __forceinline__ TurnConst(const AdjArgs &a, int t) {
        const double *rf = a.rf + (size_t)t * 3 * a.n_rf;
#pragma unroll
        for (int j = 0; j < kAdjMaxRf; ++j) {
            V[j] = w[j] = phi[j] = 0.0;
            if (j < a.n_rf) {
                V[j] = rf[j];
                w[j] = rf[a.n_rf + j];
                phi[j] = rf[2 * a.n_rf + j];
            }
        }
        acc = a.acc[t];
        coeff = a.drift[t + 1].coeff;
    }
};

// One macroparticle through turn t: induced kick (the table, or V_t and the
// spline weights), RF kick, drift.
template <int MAP>
__device__ __forceinline__ void forward_step(double &x, double &e, const double2 *tab,
                                             const double *vt, const TurnConst &c,
                                             LdsConstDoublePtr stab, const AdjArgs &a) {
    if (MAP == kMapReference) {
        const int k = interp_bin(x, a);
        const double2 se = tab[k >= 0 ? k : 0];
        const double e1 = e + (x * se.x + se.y);  // linear_interp_kick.cpp:60
        e = k >= 0 ? e1 : e;
    } else {
        double wk[3];
        int k;
        e = e + induced_kick(vt, x, a, nullptr, wk, k);
    }
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < kAdjMaxRf; ++j)
        if (j < a.n_rf) s = s + c.V[j] * cephes_sin_tab(c.w[j] * x + c.phi[j], stab);
    e = e + (a.charge * s + c.acc);
    x = x + c.coeff * e;
}

template <int MAP, bool FUSE>
__global__ void __launch_bounds__(kAdjBlock) adj_turn_kernel(const double *xi, const double *ei,
                                                             double *xo, double *eo, int64_t n,
                                                             int t, AdjArgs a) {
    extern __shared__ __align__(16) double sh_turn[];
    __shared__ __align__(16) double sin_tab[kCephesTabDoubles];
    const int ns = a.ns, b = threadIdx.x;  // slice b of this thread (ns <= kAdjBlock)
    double2 *tab = reinterpret_cast<double2 *>(sh_turn);
    double *vl = sh_turn + 2 * ns;
    unsigned long long *hdep = reinterpret_cast<unsigned long long *>(sh_turn + 3 * ns);
    double *prod = sh_turn + 4 * ns;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t i_first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n2 = (n + 1) / 2;
    // everything the prologue and the first two pairs read is asked for at once
    auto load = [&](int64_t i, double2 &x, double2 &e) {
        if (i >= n2) return;
        x = reinterpret_cast<const double2 *>(xi)[i];
        e = reinterpret_cast<const double2 *>(ei)[i];
    };
    double2 xa{}, ea{}, xb{}, eb{};
    load(i_first, xa, ea);
    load(i_first + stride, xb, eb);
    const double bcb = MAP == kMapReference && b < ns ? a.bc[b] : 0.0;
    const TurnConst c(a, t);
    double v0 = 0.0, v1 = 0.0;
    if (FUSE) {
        const double g = prod_load_g<1>(a);
        const double p =
            b < ns ? (double)(long long)ring_sum(a.dep, t, ns, b) * (1.0 / a.fix_scale) : 0.0;
        prod_put(prod, g, p, a);
        if (blockIdx.x == 0 && b < ns) a.prof[(size_t)t * ns + b] = p;
    } else if (b < ns) {
        v0 = a.vt[(size_t)t * ns + b];
        if (b + 1 < ns) v1 = a.vt[(size_t)t * ns + b + 1];
    }
    cephes_tab_fill((LdsDoublePtr)sin_tab);
    if (b < ns) hdep[b] = 0ull;
    if (FUSE) {
        __syncthreads();
        prod_run(prod, a);
        __syncthreads();
        if (b < ns) {
            v0 = prod_out(prod, b, a);
            if (b + 1 < ns) v1 = prod_out(prod, b + 1, a);
            if (blockIdx.x == 0) a.vt[(size_t)t * ns + b] = v0;
        }
        ring_clear(a.dep, t + 2, ns);
    }
    if (MAP == kMapReference) {
        if (b < ns - 1) tab[b] = interp_pair(v0, v1, bcb, a);
    } else if (b < ns) {
        vl[b] = v0;
    }
    __syncthreads();
    const LdsConstDoublePtr stab = (LdsConstDoublePtr)sin_tab;
    auto pair = [&](int64_t i, double2 &x, double2 &e) {
        forward_step<MAP>(x.x, e.x, tab, vl, c, stab, a);
        forward_step<MAP>(x.y, e.y, tab, vl, c, stab, a);
        reinterpret_cast<double2 *>(xo)[i] = x;
        reinterpret_cast<double2 *>(eo)[i] = e;
        const double2 xd = x;
        load(i + 2 * stride, x, e);
        deposit<MAP>(hdep, xd.x, a);
        if (2 * i + 1 < n) deposit<MAP>(hdep, xd.y, a);
    };
    for (int64_t i = i_first; i < n2; i += 2 * stride) {
        pair(i, xa, ea);
        if (i + stride < n2) pair(i + stride, xb, eb);
    }
    deposit_flush(hdep, a, t + 1);
}

// ---------------------------------------------------------------------------
// dt of states t0 + 1 .. t1 - 1 of a segment from state t0, into slots 0, 1, ...
// (stride np doubles): the map is linear in dE, so the reverse pass needs no
// more.  The segment's voltages are known, so nothing joins the particles
// between its turns: they stay in registers, two pairs a thread, and each turn
// only writes (8 B a macroparticle, where a launch a turn reads and writes 32:
// 3.2 us a turn at 1e6, 2.5 of them arithmetic, against 8.6 and a launch gap;
// 3.8 with dE written too).  A turn's table is built in one of two LDS buffers
// while the turn before uses the other; its voltages are loaded a turn ahead
// (its RF programs too: measured the same).
// ---------------------------------------------------------------------------
static size_t adj_segment_lds(int ns) { return sizeof(double) * 6 * (size_t)ns; }

template <int MAP>
__global__ void __launch_bounds__(kAdjBlock) adj_segment_kernel(const double *xi, const double *ei,
                                                                double *slots, int64_t np,
                                                                int64_t n, int t0, int t1,
                                                                AdjArgs a) {
    extern __shared__ __align__(16) double sh_seg[];
    __shared__ __align__(16) double sin_tab[kCephesTabDoubles];
    const int ns = a.ns;
    double2 *tab[2] = {reinterpret_cast<double2 *>(sh_seg),
                       reinterpret_cast<double2 *>(sh_seg + 2 * ns)};
    double *vl[2] = {sh_seg + 4 * ns, sh_seg + 5 * ns};
    cephes_tab_fill((LdsDoublePtr)sin_tab);
    const LdsConstDoublePtr stab = (LdsConstDoublePtr)sin_tab;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t n2 = (n + 1) / 2;
    // kAdjMaxSlices <= kAdjBlock: one slice a thread
    const int b = threadIdx.x;
    const bool has = MAP == kMapReference ? b < ns - 1 : b < ns;
    const double bcb = MAP == kMapReference && has ? a.bc[b] : 0.0;
    double v0 = 0.0, v1 = 0.0;
    auto fetch = [&](int t) {
        if (!has) return;
        v0 = a.vt[(size_t)t * ns + b];
        if (MAP == kMapReference) v1 = a.vt[(size_t)t * ns + b + 1];
    };
    auto put = [&](int t) {
        if (!has) return;
        if (MAP == kMapReference) tab[t & 1][b] = interp_pair(v0, v1, bcb, a);
        else vl[t & 1][b] = v0;
    };
    // every thread runs every step (the barriers), its pairs where it has any
    for (int64_t base = (int64_t)blockIdx.x * blockDim.x; base < n2; base += 2 * stride) {
        const int64_t i = base + threadIdx.x, j = i + stride;
        const bool hi = i < n2, hj = j < n2;
        double2 x0{}, e0{}, x1{}, e1{};
        if (hi) {
            x0 = reinterpret_cast<const double2 *>(xi)[i];
            e0 = reinterpret_cast<const double2 *>(ei)[i];
        }
        if (hj) {
            x1 = reinterpret_cast<const double2 *>(xi)[j];
            e1 = reinterpret_cast<const double2 *>(ei)[j];
        }
        fetch(t0);
        __syncthreads();  // the chunk before has left both buffers
        put(t0);
        for (int t = t0; t < t1 - 1; ++t) {
            __syncthreads();  // turn t's table is in place, turn t - 1's is free
            if (t + 1 < t1 - 1) fetch(t + 1);
            const TurnConst c(a, t);
            const double2 *tb = tab[t & 1];
            const double *vb = vl[t & 1];
            double *xo = slots + (size_t)(t - t0) * np;
            forward_step<MAP>(x0.x, e0.x, tb, vb, c, stab, a);
            forward_step<MAP>(x0.y, e0.y, tb, vb, c, stab, a);
            forward_step<MAP>(x1.x, e1.x, tb, vb, c, stab, a);
            forward_step<MAP>(x1.y, e1.y, tb, vb, c, stab, a);
            if (hi) reinterpret_cast<double2 *>(xo)[i] = x0;
            if (hj) reinterpret_cast<double2 *>(xo)[j] = x1;
            if (t + 1 < t1 - 1) put(t + 1);
        }
    }
}

// Lanes that share one output of a circular product (each a residue class
// of the k range); 16 with 1024-thread workgroups (c5: 2.51e10 against
// 2.42e10 macroparticle-turns/s with 4 lanes and 256 threads).
constexpr int kLanes = 16;

// Circular dot product over k = r, r + kLanes, ... < k_end of G[m(k)] X[k],
// m(k) = (s0 + SGN k) mod n_fft (s0 + SGN k within (-n_fft, 2 n_fft)), G
// read as zero from g_len on; four accumulators so the LDS reads of
// consecutive terms overlap.  Lane r of a group takes residue r: the group
// reads consecutive words.
template <int SGN>
__device__ __forceinline__ double circ_dot(const double *G, int n_fft, int g_len, const double *X,
                                           int r, int k_end, int s0) {
    auto gat = [&](int k) -> double {
        int m = s0 + SGN * k;
        m += m < 0 ? n_fft : 0;
        m -= m >= n_fft ? n_fft : 0;
        const double g = G[m < g_len ? m : 0];
        return m < g_len ? g : 0.0;
    };
    constexpr int L = kLanes;
    double v0 = 0.0, v1 = 0.0, v2 = 0.0, v3 = 0.0;
    int k = r;
    for (; k + 3 * L < k_end; k += 4 * L) {
        v0 = fma(gat(k), X[k], v0);
        v1 = fma(gat(k + L), X[k + L], v1);
        v2 = fma(gat(k + 2 * L), X[k + 2 * L], v2);
        v3 = fma(gat(k + 3 * L), X[k + 3 * L], v3);
    }
    for (; k < k_end; k += L) v0 = fma(gat(k), X[k], v0);
    return (v0 + v1) + (v2 + v3);
}

// An output of a circular product is computed by a group of kLanes lanes;
// the groups stay together because every trip count below is a multiple of
// kLanes.  The group's sum, in every lane.
__device__ __forceinline__ double lanes_sum(double v) {
#pragma unroll
    for (int o = 1; o < kLanes; o <<= 1) v += __shfl_xor(v, o);
    return v;
}

// Outputs per workgroup of the slice-axis kernels (kAdjSliceBlock / kLanes).
constexpr int kAdjSliceBlock = 1024;
constexpr int kAdjSliceOut = kAdjSliceBlock / kLanes;

// p_t from its deposit, stored; with `voltage`, V_t = -scale * (g conv p_t)
// stored too.  Workgroup b owns outputs [64 b, 64 b + 64).
__global__ void __launch_bounds__(kAdjSliceBlock) adj_profile_kernel(AdjArgs a, int t, bool voltage) {
    extern __shared__ double sh[];
    double *p = sh, *gs = sh + a.ns;
    const int ns = a.ns;
    const double inv = 1.0 / a.fix_scale;
    const int o0 = blockIdx.x * kAdjSliceOut, o1 = min(ns, o0 + kAdjSliceOut);
    for (int j = threadIdx.x; j < ns; j += blockDim.x) {
        p[j] = (double)(long long)ring_sum(a.dep, t, ns, j) * inv;
        if (j >= o0 && j < o1) a.prof[(size_t)t * ns + j] = p[j];
    }
    ring_clear(a.dep, t + 2, ns);
    if (!voltage) return;
    for (int m = threadIdx.x; m < a.n_fft; m += blockDim.x) gs[m] = a.g[m];
    __syncthreads();
    // V_t[i] = -scale sum_j g[(i - j) mod n_fft] p[j]
    for (int q = threadIdx.x; q < (o1 - o0) * kLanes; q += blockDim.x) {
        const int i = o0 + q / kLanes, r = q % kLanes;
        const double v = lanes_sum(circ_dot<-1>(gs, a.n_fft, a.n_fft, p, r, ns, i));
        if (r == 0) a.vt[(size_t)t * ns + i] = -(a.scale * v);
    }
}

// ---------------------------------------------------------------------------
// Reverse turn t (xs, x1s: dt_t and dt_{t+1}): see the file comment.  FUSE:
// lp_{t+1} is formed here from lV_{t+1}; else it is read from a.lp.  Pairs of
// macroparticles as in adj_turn_kernel (the pad slot's adjoints stay zero),
// one pair ahead (two take 18.9 us in place of 17.2: 1e6 macroparticles).
// dt_{t+1} is read, not formed again from dE_t: the same traffic, one step of
// the map less (16.5 -> 15.6 us at 1e6 macroparticles), and half the slots.
// LDS: lp_{t+1}, lV_t, the kick's slopes (reference map) or V_t, the bin
// centres, and with FUSE the product's words.
// ---------------------------------------------------------------------------
static size_t adj_reverse_lds(int ns, bool fuse) {
    return sizeof(double) * (4 * (size_t)ns + (fuse ? prod_words(ns) : 0));
}

template <int MAP, bool FUSE>
__global__ void __launch_bounds__(kAdjBlock) adj_reverse_kernel(const double *__restrict__ xs,
                                                                const double *__restrict__ x1s,
                                                                double *__restrict__ lam_x,
                                                                double *__restrict__ lam_e,
                                                                int64_t n, int t, int last,
                                                                AdjArgs a) {
    extern __shared__ __align__(16) double shr[];
    double *slope = shr;
    double *vl = shr;  // spline map: V_t in the slopes' place
    double *lp = shr + a.ns, *lvs = shr + 2 * a.ns, *bcs = shr + 3 * a.ns;
    __shared__ double red[kAdjWaves][2 * kAdjMaxRf];
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t i_first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n2 = (n + 1) / 2;
    struct Pair {
        double2 x{}, x1{}, lx{}, le{};
    };
    auto load = [&](int64_t i, Pair &p) {
        if (i >= n2) return;
        p.x = reinterpret_cast<const double2 *>(xs)[i];
        p.x1 = reinterpret_cast<const double2 *>(x1s)[i];
        p.lx = reinterpret_cast<const double2 *>(lam_x)[i];
        p.le = reinterpret_cast<const double2 *>(lam_e)[i];
    };
    Pair next;
    load(i_first, next);
    const int ns = a.ns, b = threadIdx.x;  // slice b of this thread (ns <= kAdjBlock)
    const TurnConst c(a, t);
    const bool product = FUSE && t + 1 < last;
    double g = 0.0, l = 0.0;
    if (b < ns) {
        const double *vt = a.vt + (size_t)t * ns;
        const double v0 = vt[b], v1 = vt[b + 1 < ns ? b + 1 : b];
        const double bcb = MAP == kMapReference ? a.bc[b] : 0.0;
        if (!product) lp[b] = a.lp[b];
        lvs[b] = 0.0;
        if (product) l = ring_sum(a.lv, t + 1, ns, b);
        if (MAP == kMapReference) {
            bcs[b] = bcb;
            if (b < ns - 1) slope[b] = interp_pair(v0, v1, bcb, a).x;
        } else {
            vl[b] = v0;
        }
    }
    if (product) {
        double *prod = shr + 4 * ns;
        g = prod_load_g<-1>(a);
        if (blockIdx.x == 0 && b < ns) a.lvh[(size_t)(t + 1) * ns + b] = l;
        prod_put(prod, g, l, a);
        __syncthreads();
        prod_run(prod, a);
        __syncthreads();
        if (b < ns) lp[b] = prod_out(prod, b, a);
    }
    if (FUSE) ring_clear(a.lv, t + 2, ns);
    __syncthreads();
    double gsum[2 * kAdjMaxRf];
#pragma unroll
    for (int j = 0; j < 2 * kAdjMaxRf; ++j) gsum[j] = 0.0;
    auto step = [&](double x, double x1, double &lam_x_i, double &lam_e_i, bool own) {
        // the kicks of turn t and their derivatives
        double wk[3], dkick;
        int k;
        if (MAP == kMapReference) {
            k = interp_bin(x, a);
            const double sl = slope[k >= 0 ? k : 0];
            dkick = k >= 0 ? sl : 0.0;
        } else {
            induced_kick(vl, x, a, &dkick, wk, k);
        }
        // constant trip counts with a guard keep sn, cs and gsum in registers
        double sn[kAdjMaxRf], cs[kAdjMaxRf];
        double ds = 0.0;
#pragma unroll
        for (int j = 0; j < kAdjMaxRf; ++j) {
            sn[j] = cs[j] = 0.0;
            if (j < a.n_rf) {
                cephes_sincos(c.w[j] * x + c.phi[j], sn[j], cs[j]);
                ds = ds + c.V[j] * c.w[j] * cs[j];
            }
        }
        // deposit adjoint of p_{t+1} at x1
        double lx = lam_x_i;
        if (MAP == kMapReference) {
            int k1, k2;
            double d;
            if (smooth_bins(x1, a, k1, k2, d)) {
                const double l1 = (k1 >= 0 && k1 < a.ns) ? lp[k1] : 0.0;
                const double l2 = (k2 >= 0 && k2 < a.ns) ? lp[k2] : 0.0;
                lx = lx + (l2 - l1) * a.inv_bw_cut;
            }
        } else {
            double sw[3], sdw[3];
            const int kk = spline(x1, a, sw, sdw);
            if (kk != kNoBin) {
                double s3 = 0.0;
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const int b = kk - 1 + q;
                    if (b >= 0 && b < a.ns) s3 += lp[b] * sdw[q];
                }
                lx = lx + s3 * a.inv_bw_cut;
            }
        }
        const double le2 = lam_e_i + c.coeff * lx;
        lx = lx + le2 * (a.charge * ds);
        if (!own) return;
#pragma unroll
        for (int j = 0; j < kAdjMaxRf; ++j) {
            if (j < a.n_rf) {
                gsum[2 * j] += le2 * a.charge * sn[j];
                gsum[2 * j + 1] += le2 * a.charge * c.V[j] * cs[j];
            }
        }
        lx = lx + le2 * dkick;
        if (MAP == kMapReference) {
            if (k >= 0) {
                const double sk = (x - bcs[k]) * a.inv_bw_bc;
                atomicAdd(&lvs[k], le2 * a.charge * (1.0 - sk));
                atomicAdd(&lvs[k + 1], le2 * a.charge * sk);
            }
        } else if (k != kNoBin) {
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const int b = k - 1 + q;
                if (b >= 0 && b < a.ns) atomicAdd(&lvs[b], le2 * a.charge * wk[q]);
            }
        }
        lam_x_i = lx;
        lam_e_i = le2;
    };
    for (int64_t i = i_first; i < n2; i += stride) {
        Pair p = next;
        load(i + stride, next);
        step(p.x.x, p.x1.x, p.lx.x, p.le.x, true);
        step(p.x.y, p.x1.y, p.lx.y, p.le.y, 2 * i + 1 < n);
        reinterpret_cast<double2 *>(lam_x)[i] = p.lx;
        reinterpret_cast<double2 *>(lam_e)[i] = p.le;
    }
    // per-workgroup RF gradient sums (fixed order: wavefront tree, then
    // waves), added to the workgroup's row over the turns
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int j = 0; j < 2 * kAdjMaxRf; ++j) {
        if (j < 2 * a.n_rf) {
            const double v = wave_sum(gsum[j]);
            if (lane == 0) red[wid][j] = v;
        }
    }
    __syncthreads();
    if ((int)threadIdx.x < 2 * a.n_rf) {
        double v = 0.0;
        for (int q = 0; q < kAdjWaves; ++q) v += red[q][threadIdx.x];
        a.gpart[(size_t)blockIdx.x * 2 * a.n_rf + threadIdx.x] += v;
    }
    double *out = a.lv + ((size_t)(t % kAdjRing) * kAdjCopies + blockIdx.x % kAdjCopies) * a.ns;
    for (int b = threadIdx.x; b < a.ns; b += blockDim.x)
        if (lvs[b] != 0.0) atomic_add_agent(&out[b], lvs[b]);
}

// lV_t from its copies, kept for the pass's correlation, and with `product`
// lp_t = -scale (g corr lV_t): the turns that do not form it in the particle
// launch's prologue, and turn 0's lV_0.  Workgroup b owns 64 outputs.
__global__ void __launch_bounds__(kAdjSliceBlock) adj_iv_kernel(AdjArgs a, int t, bool product) {
    extern __shared__ double sh[];
    const int ns = a.ns;
    double *lvs = sh, *gs = sh + ns;
    const int o0 = blockIdx.x * kAdjSliceOut, o1 = min(ns, o0 + kAdjSliceOut);
    for (int i = threadIdx.x; i < ns; i += blockDim.x) {
        lvs[i] = ring_sum(a.lv, t, ns, i);
        if (i >= o0 && i < o1) a.lvh[(size_t)t * ns + i] = lvs[i];
    }
    if (!product) return;
    // the slot that turn t - 1 adds into (t + 2 is t - 1 modulo the ring)
    ring_clear(a.lv, t + 2, ns);
    for (int m = threadIdx.x; m < a.n_fft; m += blockDim.x) gs[m] = a.g[m];
    __syncthreads();
    for (int q = threadIdx.x; q < (o1 - o0) * kLanes; q += blockDim.x) {
        const int o = o0 + q / kLanes, r = q % kLanes;
        const double v = lanes_sum(circ_dot<1>(gs, a.n_fft, a.n_fft, lvs, r, ns, -o));
        if (r == 0) a.lp[o] = -(a.scale * v);
    }
}

// The pass's correlation: workgroup (b, q) sums the q-th share of corr[m] over
// turns b, b + grid, ... into row b of `part`, for the entries that have a term
// (m < ns, then m > n_fft - ns).  Once a pass, where every turn's slice launch
// held it before.  A turn's share of it is ns^2 products on one CU, so with
// fewer turns than CUs the outputs are split over the others (corr_parts).
// 256 slices: 4.7 us for 50 turns, 6.8 for 100 (one workgroup a turn 10.4 and
// 10.6); 1024 slices: 9.1 us for one turn, 28 for 50, 64 for 100 (113, 116,
// 119).
__host__ __device__ __forceinline__ int corr_outputs(int ns, int n_fft) {
    const int hi0 = ns > n_fft - ns + 1 ? ns : n_fft - ns + 1;
    return ns + (n_fft - hi0);
}
__global__ void __launch_bounds__(kAdjSliceBlock) adj_corr_kernel(AdjArgs a, int turns,
                                                                  double *__restrict__ part) {
    extern __shared__ double sh[];
    const int ns = a.ns, n_out = corr_outputs(ns, a.n_fft), first = a.n_fft - (n_out - ns);
    double *lvs = sh, *p = sh + ns;
    const int per = (n_out + (int)gridDim.y - 1) / (int)gridDim.y;
    const int o0 = (int)blockIdx.y * per, o1 = min(n_out, o0 + per);
    // kLanes lanes an output; an output's sum is added to by the same lane
    // over the turns
    for (int t = blockIdx.x; t < turns; t += gridDim.x) {
        __syncthreads();
        for (int i = threadIdx.x; i < ns; i += blockDim.x) {
            lvs[i] = a.lvh[(size_t)t * ns + i];
            p[i] = a.prof[(size_t)t * ns + i];
        }
        __syncthreads();
        for (int q = o0 * kLanes + (int)threadIdx.x; q < o1 * kLanes; q += blockDim.x) {
            const int o = q / kLanes, r = q % kLanes;
            const int m = o < ns ? o : first + (o - ns);
            const double v = lanes_sum(circ_dot<1>(p, a.n_fft, ns, lvs, r, ns, -m));
            if (r == 0) {
                double *row = part + (size_t)blockIdx.x * n_out + o;
                *row = t == (int)blockIdx.x ? v : *row + v;
            }
        }
    }
}
// corr[m] = sum of the rows, zero elsewhere
__global__ void adj_corr_sum_kernel(const double *__restrict__ part, int rows, int ns, int n_fft,
                                    double *__restrict__ corr) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n_fft) return;
    const int n_out = corr_outputs(ns, n_fft), first = n_fft - (n_out - ns);
    const int o = m < ns ? m : (m >= first ? ns + (m - first) : -1);
    double v = 0.0;
    if (o >= 0)
#pragma unroll 8
        for (int r = 0; r < rows; ++r) v += part[(size_t)r * n_out + o];
    corr[m] = v;
}

// Workgroups of the pass's correlation: a turn each, as many as there are CUs,
// and as many times over, at least a workgroup's 64 outputs each, as CUs are left.
static int corr_rows(int turns) {
    const int cus = device_cu_count();
    return turns < cus ? turns : cus;
}
static int corr_parts(int rows, int n_out) {
    const int most = (n_out + kAdjSliceOut - 1) / kAdjSliceOut, left = device_cu_count() / rows;
    return left < most ? left : most;
}

// Workgroups of the slice-axis kernels: 64 outputs each.
static int adj_slice_grid(int ns) { return (ns + kAdjSliceOut - 1) / kAdjSliceOut; }
// ---------------------------------------------------------------------------
Adjoint::~Adjoint() { release(); }

void Adjoint::invalidate_graphs() {
    if (fwd_exec) (void)hipGraphExecDestroy(fwd_exec);
    if (bwd_exec) (void)hipGraphExecDestroy(bwd_exec);
    fwd_exec = bwd_exec = nullptr;
    fwd_graph_turns = bwd_graph_turns = -1;
}

int Adjoint::ensure_stream() {
    if (own) return BLMI_OK;
    BLMI_HIP_TRY(hipStreamCreateWithFlags(&own, hipStreamNonBlocking));
    BLMI_HIP_TRY(hipEventCreateWithFlags(&ev_in, hipEventDisableTiming));
    BLMI_HIP_TRY(hipEventCreateWithFlags(&ev_out, hipEventDisableTiming));
    return BLMI_OK;
}

int Adjoint::settle() {
    if (in_flight) BLMI_HIP_TRY(hipStreamSynchronize(own));
    in_flight = false;
    return BLMI_OK;
}

void Adjoint::release() {
    invalidate_graphs();
    if (own) (void)hipStreamDestroy(own);
    if (ev_in) (void)hipEventDestroy(ev_in);
    if (ev_out) (void)hipEventDestroy(ev_out);
    own = nullptr;
    ev_in = ev_out = nullptr;
    void *bufs[] = {d_rf, d_acc, d_drift, d_x0, d_work, d_ckpt, d_slots, d_lam, d_dep,
                    d_prof, d_vt, d_g, d_lv, d_lvh, d_lp, d_corr, d_corr_part, d_gpart, d_bc};
    for (void *p : bufs) (void)hipFree(p);
    d_rf = d_acc = d_x0 = d_work = d_ckpt = d_slots = d_lam = nullptr;
    d_prof = d_vt = d_g = d_lv = d_lvh = d_lp = d_corr = d_corr_part = d_gpart = d_bc = nullptr;
    d_drift = nullptr;
    d_dep = nullptr;
}

int Adjoint::init(int64_t n_, int n_rf_, int n_turns_, int n_slices_, int every_) {
    n = n_;
    n_rf = n_rf_;
    n_turns = n_turns_;
    n_slices = n_slices_;
    every = every_;
    BLMI_HIP_TRY(hipGetDevice(&device));
    // a workgroup of 1024 threads per CU, fewer where each has less than a pair
    const int64_t pairs = (n + 1) / 2, want = (pairs + kAdjBlock - 1) / kAdjBlock;
    grid = device_cu_count();
    if (want < grid) grid = want > 0 ? (int)want : 1;
    // dt and dE of a state each take an even number of places (16-byte pairs)
    np = (n + 1) & ~(int64_t)1;
    const size_t nt = (size_t)n_turns + 1;
    const size_t pn = 2 * (size_t)np;
    const int n_ckpt = (n_turns + every - 1) / every;
    BLMI_HIP_TRY(hipMalloc(&d_rf, sizeof(double) * 3 * n_rf * nt));
    BLMI_HIP_TRY(hipMalloc(&d_acc, sizeof(double) * nt));
    BLMI_HIP_TRY(hipMalloc(&d_drift, sizeof(DriftCoeffs<double>) * nt));
    BLMI_HIP_TRY(hipMalloc(&d_x0, sizeof(double) * pn));
    BLMI_HIP_TRY(hipMemset(d_x0, 0, sizeof(double) * pn));  // the pad slots
    BLMI_HIP_TRY(hipMalloc(&d_work, sizeof(double) * pn));
    BLMI_HIP_TRY(hipMalloc(&d_ckpt, sizeof(double) * pn * n_ckpt));
    BLMI_HIP_TRY(hipMalloc(&d_slots, sizeof(double) * (size_t)np * every));
    BLMI_HIP_TRY(hipMalloc(&d_lam, sizeof(double) * pn));
    BLMI_HIP_TRY(hipMalloc(&d_dep, sizeof(unsigned long long) * kAdjRing * kAdjCopies * n_slices));
    BLMI_HIP_TRY(hipMalloc(&d_prof, sizeof(double) * nt * n_slices));
    BLMI_HIP_TRY(hipMalloc(&d_vt, sizeof(double) * nt * n_slices));
    BLMI_HIP_TRY(hipMemset(d_vt, 0, sizeof(double) * nt * n_slices));
    BLMI_HIP_TRY(hipMalloc(&d_lv, sizeof(double) * kAdjRing * kAdjCopies * n_slices));
    BLMI_HIP_TRY(hipMalloc(&d_lvh, sizeof(double) * n_turns * (size_t)n_slices));
    BLMI_HIP_TRY(hipMalloc(&d_lp, sizeof(double) * n_slices));
    BLMI_HIP_TRY(hipMalloc(&d_gpart, sizeof(double) * (size_t)grid * 2 * n_rf));
    fixed_bits = smooth_scale_bits(n);
    return BLMI_OK;
}

int Adjoint::set_particles(const double *dt, const double *dE) {
    BLMI_HIP_TRY(hipMemcpy(d_x0, dt, sizeof(double) * n, hipMemcpyDeviceToDevice));
    BLMI_HIP_TRY(hipMemcpy(d_x0 + np, dE, sizeof(double) * n, hipMemcpyDeviceToDevice));
    // a pass enqueued from a stream that does not wait for the default one
    BLMI_HIP_TRY(hipStreamSynchronize(nullptr));
    forward_done = false;
    return BLMI_OK;
}

int Adjoint::set_programs(const double *rf_host, const double *acc_host, const double *t_rev,
                          double length_ratio, double alpha_order, const double *eta0,
                          const double *eta1, const double *eta2, const double *alpha0,
                          const double *alpha1, const double *alpha2, const double *beta,
                          const double *energy, double charge_) {
    const size_t nt = (size_t)n_turns + 1;
    int rc = settle();  // a forward without its backward reads the programs
    if (rc) return rc;
    // the captured passes hold scalars by value: a changed one re-captures
    if (charge_ != charge) invalidate_graphs();
    charge = charge_;
    BLMI_HIP_TRY(hipMemcpy(d_rf, rf_host, sizeof(double) * 3 * n_rf * nt, hipMemcpyHostToDevice));
    BLMI_HIP_TRY(hipMemcpy(d_acc, acc_host, sizeof(double) * nt, hipMemcpyHostToDevice));
    std::vector<DriftCoeffs<double>> dc(nt);
    for (size_t i = 0; i < nt; ++i)
        dc[i] = make_drift_coeffs<double>(0, t_rev[i], length_ratio, alpha_order, eta0[i], eta1[i],
                                          eta2[i], alpha0[i], alpha1[i], alpha2[i], beta[i],
                                          energy[i]);
    BLMI_HIP_TRY(hipMemcpy(d_drift, dc.data(), sizeof(DriftCoeffs<double>) * nt,
                           hipMemcpyHostToDevice));
    forward_done = false;
    return BLMI_OK;
}

int Adjoint::set_slices(double cl, double cr) {
    const double ibw = (double)n_slices / (cr - cl);  // histogram.cpp:82
    if (cl != cut_left || ibw != inv_bw_cut) invalidate_graphs();
    cut_left = cl;
    inv_bw_cut = ibw;
    const double bw = (cr - cl) / (double)n_slices;  // histogram.cpp:83-85
    lo = cl + bw * 0.5;
    hi = cr - bw * 0.5;
    forward_done = false;
    return BLMI_OK;
}

int Adjoint::set_map(int map_, const double *bc_host) {
    if (map_ != kMapSpline && map_ != kMapReference)
        return blmi_set_error(BLMI_ERR_ARG, "adjoint: unknown map %d", map_);
    if (map_ == kMapReference) {
        if (!bc_host || n_slices < 2)
            return blmi_set_error(BLMI_ERR_ARG, "adjoint: the reference map needs >= 2 bin centres");
        if (!d_bc) BLMI_HIP_TRY(hipMalloc(&d_bc, sizeof(double) * n_slices));
        BLMI_HIP_TRY(hipMemcpy(d_bc, bc_host, sizeof(double) * n_slices, hipMemcpyHostToDevice));
        bc0 = bc_host[0];
        // linear_interp_kick.cpp:33-35
        inv_bw_bc = (double)(n_slices - 1) / (bc_host[n_slices - 1] - bc_host[0]);
    }
    map = map_;
    invalidate_graphs();
    forward_done = false;
    return BLMI_OK;
}

int Adjoint::set_wake(int64_t n_fft_, const double *g_host, double scale_) {
    if (n_fft_ < n_slices || n_fft_ > 8192)
        return blmi_set_error(BLMI_ERR_UNSUPPORTED, "adjoint: n_fft %lld outside [n_slices, 8192]",
                              (long long)n_fft_);
    int rc = settle();  // as set_programs
    if (rc) return rc;
    if (n_fft_ != n_fft || scale_ != scale) invalidate_graphs();
    if (n_fft_ != n_fft) {
        (void)hipFree(d_g);
        (void)hipFree(d_corr);
        (void)hipFree(d_corr_part);
        d_g = d_corr = d_corr_part = nullptr;
        BLMI_HIP_TRY(hipMalloc(&d_g, sizeof(double) * n_fft_));
        BLMI_HIP_TRY(hipMalloc(&d_corr, sizeof(double) * n_fft_));
        BLMI_HIP_TRY(hipMalloc(&d_corr_part, sizeof(double) * corr_outputs(n_slices, (int)n_fft_) *
                                                 (size_t)corr_rows(n_turns)));
    }
    n_fft = n_fft_;
    scale = scale_;
    BLMI_HIP_TRY(hipMemcpy(d_g, g_host, sizeof(double) * n_fft, hipMemcpyHostToDevice));
    // slice-axis kernels: profile + wake (+ adjoint) in LDS, up to 80 KiB
    const int lds_p = (int)(sizeof(double) * ((size_t)n_slices + n_fft));
    BLMI_HIP_TRY(hipFuncSetAttribute((const void *)adj_profile_kernel,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds_p));
    BLMI_HIP_TRY(hipFuncSetAttribute((const void *)adj_iv_kernel,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds_p));
    forward_done = false;
    return BLMI_OK;
}

static AdjArgs adj_args(const Adjoint &j) {
    AdjArgs a{};
    a.n_rf = j.n_rf;
    a.charge = j.charge;
    a.rf = j.d_rf;
    a.acc = j.d_acc;
    a.drift = j.d_drift;
    a.ns = j.n_slices;
    a.cut_left = j.cut_left;
    a.inv_bw_cut = j.inv_bw_cut;
    a.fix_scale = ldexp(1.0, j.fixed_bits);
    a.vt = j.d_vt;
    a.dep = j.d_dep;
    a.lv = j.d_lv;
    a.lp = j.d_lp;
    a.gpart = j.d_gpart;
    a.lo = j.lo;
    a.hi = j.hi;
    a.prof = j.d_prof;
    a.lvh = j.d_lvh;
    a.g = j.d_g;
    a.n_fft = (int)j.n_fft;
    a.scale = j.scale;
    a.bc = j.d_bc;
    a.bc0 = j.bc0;
    a.inv_bw_bc = j.inv_bw_bc;
    return a;
}

// State t's dt and dE of a pass of T turns: the initial copy, a checkpoint, or
// the working arrays, which a turn between checkpoints updates in place and
// which receive the state after the last turn.
static double *state_at(const Adjoint &j, int t, int T) {
    if (t == 0) return j.d_x0;
    if (t % j.every == 0 && t < T) return j.d_ckpt + (size_t)(t / j.every) * 2 * j.np;
    return j.d_work;
}

template <int MAP, bool FUSE>
static int enqueue_forward_map(Adjoint &j, int turns, hipStream_t s) {
    const int64_t n = j.n, np = j.np;
    const int ns = j.n_slices, grid = j.grid;
    const AdjArgs a = adj_args(j);
    const size_t lds_turn = adj_turn_lds(ns, FUSE);
    const size_t lds_slice = sizeof(double) * ((size_t)ns + j.n_fft);
    const int sgrid = adj_slice_grid(ns);
    BLMI_HIP_TRY(hipFuncSetAttribute((const void *)adj_turn_kernel<MAP, FUSE>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_turn));
    // the deposits start cleared (a pass before leaves its last profiles behind)
    int rc = launch_fill<unsigned long long>(j.d_dep, (int64_t)kAdjRing * kAdjCopies * ns, 0ull, s);
    if (rc) return rc;
    hipLaunchKernelGGL(adj_deposit_kernel<MAP>, dim3(grid), dim3(kAdjBlock),
                       sizeof(unsigned long long) * ns, s, j.d_x0, n, a);
    // with every state kept (every == 1) turn t reads checkpoint t and writes
    // checkpoint t + 1, and the reverse pass recomputes nothing
    for (int t = 0; t < turns; ++t) {
        if (!FUSE)
            hipLaunchKernelGGL(adj_profile_kernel, dim3(sgrid), dim3(kAdjSliceBlock), lds_slice, s,
                               a, t, true);
        const double *si = state_at(j, t, turns);
        double *so = state_at(j, t + 1, turns);
        hipLaunchKernelGGL((adj_turn_kernel<MAP, FUSE>), dim3(grid), dim3(kAdjBlock), lds_turn, s,
                           si, si + np, so, so + np, n, t, a);
    }
    hipLaunchKernelGGL(adj_profile_kernel, dim3(sgrid), dim3(kAdjSliceBlock), lds_slice, s, a,
                       turns, false);
    return blmi_check_launch("adjoint_forward");
}

int Adjoint::enqueue_forward(int turns, hipStream_t s) {
    const bool fuse = n_slices <= kAdjFuseSlices;
    if (map == kMapReference)
        return fuse ? enqueue_forward_map<kMapReference, true>(*this, turns, s)
                    : enqueue_forward_map<kMapReference, false>(*this, turns, s);
    return fuse ? enqueue_forward_map<kMapSpline, true>(*this, turns, s)
                : enqueue_forward_map<kMapSpline, false>(*this, turns, s);
}

template <int MAP, bool FUSE>
static int enqueue_backward_map(Adjoint &j, int T, hipStream_t s) {
    const int64_t n = j.n, np = j.np;
    const int ns = j.n_slices, every = j.every, grid = j.grid;
    const size_t pn = 2 * (size_t)np;
    const size_t lds_rev = adj_reverse_lds(ns, FUSE), lds_seg = adj_segment_lds(ns);
    const size_t lds_slice = sizeof(double) * ((size_t)ns + j.n_fft);
    const AdjArgs a = adj_args(j);
    const int sgrid = adj_slice_grid(ns), rows = corr_rows(T);
    BLMI_HIP_TRY(hipFuncSetAttribute((const void *)adj_reverse_kernel<MAP, FUSE>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_rev));
    int rc = launch_fill<double>(j.d_lam, (int64_t)pn, 0.0, s);
    if (!rc) rc = launch_fill<double>(j.d_lv, (int64_t)kAdjRing * kAdjCopies * ns, 0.0, s);
    if (!rc) rc = launch_fill<double>(j.d_gpart, (int64_t)grid * 2 * j.n_rf, 0.0, s);
    if (rc) return rc;
    for (int seg = (T - 1) / every; seg >= 0; --seg) {
        const int t0 = seg * every, t1 = (t0 + every < T) ? t0 + every : T;
        // states t0 and t1 are kept; dt of t0 + 1 .. t1 - 1 go to slots 0 .. t1 - t0 - 2
        const double *s0 = state_at(j, t0, T);
        const double *x1 = state_at(j, t1, T);
        if (t1 - t0 > 1)
            hipLaunchKernelGGL(adj_segment_kernel<MAP>, dim3(grid), dim3(kAdjBlock), lds_seg, s, s0,
                               s0 + np, j.d_slots, np, n, t0, t1, a);
        for (int t = t1 - 1; t >= t0; --t) {
            const double *x0 = t == t0 ? s0 : j.d_slots + (size_t)(t - t0 - 1) * np;
            hipLaunchKernelGGL((adj_reverse_kernel<MAP, FUSE>), dim3(grid), dim3(kAdjBlock), lds_rev,
                               s, x0, x1, j.d_lam, j.d_lam + np, n, t, T, a);
            x1 = x0;
            if (!FUSE || t == 0)
                hipLaunchKernelGGL(adj_iv_kernel, dim3(sgrid), dim3(kAdjSliceBlock), lds_slice, s, a,
                                   t, !FUSE && t > 0);
        }
    }
    const int parts = corr_parts(rows, corr_outputs(ns, (int)j.n_fft));
    hipLaunchKernelGGL(adj_corr_kernel, dim3(rows, parts), dim3(kAdjSliceBlock),
                       sizeof(double) * 2 * (size_t)ns, s, a, T, j.d_corr_part);
    hipLaunchKernelGGL(adj_corr_sum_kernel, dim3((unsigned)((j.n_fft + 63) / 64)), dim3(64), 0, s,
                       j.d_corr_part, rows, ns, (int)j.n_fft, j.d_corr);
    return blmi_check_launch("adjoint_backward");
}

int Adjoint::enqueue_backward(int T, hipStream_t s) {
    const bool fuse = n_slices <= kAdjFuseSlices;
    if (map == kMapReference)
        return fuse ? enqueue_backward_map<kMapReference, true>(*this, T, s)
                    : enqueue_backward_map<kMapReference, false>(*this, T, s);
    return fuse ? enqueue_backward_map<kMapSpline, true>(*this, T, s)
                : enqueue_backward_map<kMapSpline, false>(*this, T, s);
}

// Capture `enqueue` on the own stream into *exec (once per turn count).
template <typename F>
static int capture(hipStream_t own, hipGraphExec_t *exec, F enqueue) {
    BLMI_HIP_TRY(hipStreamBeginCapture(own, hipStreamCaptureModeThreadLocal));
    int rc = enqueue();
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(own, &g);
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess)
        return blmi_set_error(BLMI_ERR_HIP, "hipStreamEndCapture: %s", hipGetErrorString(e));
    hipError_t ie = hipGraphInstantiate(exec, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ie != hipSuccess)
        return blmi_set_error(BLMI_ERR_HIP, "hipGraphInstantiate: %s", hipGetErrorString(ie));
    return BLMI_OK;
}

int Adjoint::forward(int turns, double *profile_out, hipStream_t user) {
    if (!d_g) return blmi_set_error(BLMI_ERR_ARG, "adjoint: set the wake first");
    if (turns < 1 || turns > n_turns)
        return blmi_set_error(BLMI_ERR_ARG, "adjoint: turns %d outside [1, %d]", turns, n_turns);
    int rc = ensure_stream();
    if (rc) return rc;
    if (!fwd_exec || fwd_graph_turns != turns) {
        if (fwd_exec) (void)hipGraphExecDestroy(fwd_exec);
        fwd_exec = nullptr;
        rc = capture(own, &fwd_exec, [&] { return enqueue_forward(turns, own); });
        if (rc) return rc;
        fwd_graph_turns = turns;
    }
    BLMI_HIP_TRY(hipEventRecord(ev_in, user));
    BLMI_HIP_TRY(hipStreamWaitEvent(own, ev_in, 0));
    in_flight = true;
    BLMI_HIP_TRY(hipGraphLaunch(fwd_exec, own));
    BLMI_HIP_TRY(hipMemcpyAsync(profile_out, d_prof + (size_t)turns * n_slices,
                                sizeof(double) * n_slices, hipMemcpyDeviceToDevice, own));
    BLMI_HIP_TRY(hipEventRecord(ev_out, own));
    BLMI_HIP_TRY(hipStreamWaitEvent(user, ev_out, 0));
    forward_done = true;
    forward_turns = turns;
    return BLMI_OK;
}

int Adjoint::backward(const double *dprofile, double *grad_rf_host, double *corr_host,
                      hipStream_t user) {
    if (!forward_done) return blmi_set_error(BLMI_ERR_ARG, "adjoint: run forward first");
    const int T = forward_turns;
    int rc = ensure_stream();
    if (rc) return rc;
    if (!bwd_exec || bwd_graph_turns != T) {
        if (bwd_exec) (void)hipGraphExecDestroy(bwd_exec);
        bwd_exec = nullptr;
        rc = capture(own, &bwd_exec, [&] { return enqueue_backward(T, own); });
        if (rc) return rc;
        bwd_graph_turns = T;
    }
    BLMI_HIP_TRY(hipEventRecord(ev_in, user));
    BLMI_HIP_TRY(hipStreamWaitEvent(own, ev_in, 0));
    BLMI_HIP_TRY(hipMemcpyAsync(d_lp, dprofile, sizeof(double) * n_slices, hipMemcpyDeviceToDevice,
                                own));
    BLMI_HIP_TRY(hipGraphLaunch(bwd_exec, own));
    std::vector<double> gp((size_t)grid * 2 * n_rf);
    BLMI_HIP_TRY(hipMemcpyAsync(gp.data(), d_gpart, sizeof(double) * gp.size(),
                                hipMemcpyDeviceToHost, own));
    BLMI_HIP_TRY(hipMemcpyAsync(corr_host, d_corr, sizeof(double) * n_fft, hipMemcpyDeviceToHost,
                                own));
    BLMI_HIP_TRY(hipStreamSynchronize(own));
    in_flight = false;
    for (int j = 0; j < 2 * n_rf; ++j) {
        double v = 0.0;
        for (int b = 0; b < grid; ++b) v += gp[(size_t)b * 2 * n_rf + j];
        grad_rf_host[j] = v;
    }
    return BLMI_OK;
}

}  // namespace blmi

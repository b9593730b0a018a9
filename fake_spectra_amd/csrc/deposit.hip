// Fused SPH-kernel x Voigt deposit into LDS-staged sightline rows.
//
// Reference: ParticleInterp::compute_tau (fake_spectra/part_int.cpp:20-51)
// loops over sightlines and, per nearby particle, calls
// LineAbsorption::add_tau_particle (absorption.cpp:212-279), which walks
// pixels outward from the particle in both directions, adds
//     taulast = amp * dens * tau_kern_outer(vlow, vlow + dv) / velfac
// and stops after the first pixel with taulast < tautail.
// tau_kern_outer/tau_kern_inner (singleabs.h:104-167) average 7 interior
// kernel samples of K(q) * Re w over the pixel, with odd-point trapezoid
// sub-sampling when the pixel is wider than b/2.
//
// GPU mapping:
//  * one work item = (sightline, line, range of its pairs); a persistent grid
//    pulls items heaviest-first from a queue; the row of the sightline lives
//    in LDS as float64 and is flushed with coalesced stores (or FP64 atomics
//    when a sightline's pairs are split across several items);
//  * a wavefront sets up to 32 pairs up, one per lane, and its groups of 16 (32,
//    64) lanes each walk one of them, lanes on consecutive pixels; the
//    sequential tail cut becomes a ballot: the first lane whose taulast falls
//    below tautail ends the walk, lanes up to it deposit.  A walk that reaches
//    the far wing goes on by the whole wavefront, 64 pixels at a time;
//  * the mapping position -> velocity -> pixel, the pixel and sub-sample
//    offsets and the accumulation are FP64, as in the reference; the kernel
//    weights and the Voigt profile are FP32 (voigt.h);
//  * a pixel whose FP32 taulast lies within 2e-5 relative of tautail is
//    re-evaluated in FP64 so the tail-cut decision matches the reference;
//    pairs with a damping parameter above kA32Max are evaluated in FP64.
// Column density (compute_colden, part_int.cpp:53-84 with
// add_colden_particle, absorption.cpp:167-210) is all FP64, one lane per
// (pair, pixel).
#include "fsamd_internal.h"
#include "plan.h"
#include "voigt.h"
#include "deposit.h"
#include "wing_table.h"

#include <mutex>
#include <unordered_map>

namespace fsamd {

__device__ __attribute__((aligned(16))) const float d_ptab[kPTableSize] = FSAMD_P_COEF_INIT;
__device__ __attribute__((aligned(16))) const float d_dtab[kPTableSize] = FSAMD_P_DCOEF_INIT;   // dG/d(u^2)
constexpr int kG64Size = FSAMD_G64_NPIECE * FSAMD_G64_NCOEF;
__device__ const double d_gtab64[kG64Size] = FSAMD_G64_COEF_INIT;

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr double kGuard = 2e-5;
constexpr int kWingTerms = 10;

// Far-wing coefficient tables.  The profile's asymptotic series in x = 1/u^2,
//   H(a,u) = (a/sqrt(pi)) sum_k (p_k - a^2 q_{k-1}) u^(-2k-2),
// p_k = (2k+1)!!/2^k, q_k = C(2k+3,3) (2k-1)!!/2^k (voigt.h), is expanded
// about the pixel centre U over the sample offsets c (Taylor in c/U); the
// even moments m_j = sum w c^(2j) of the pixel's weighted samples then give
//   sum_samples w H = sum_n X^(n+1) sum_{k<=n} g_k C(2n+1, 2(n-k)) m_(n-k).
__constant__ double c_wing_p[kWingTerms] = {1.0, 1.5, 3.75, 13.125, 59.0625, 324.84375, 2111.484375,
                                             15836.1328125, 134607.12890625, 1278767.724609375};
__constant__ double c_wing_q[kWingTerms] = {1.0, 5.0, 26.25, 157.5, 1082.8125, 8445.9375, 73901.953125,
                                             717904.6875, 7672606.34765625, 89513740.72265625};
static_assert(FSAMD_WING_NTERMS == kWingTerms, "wing_table.h");
__constant__ double c_wing_T[(FSAMD_WING_TMAX + 1) * kWingTerms] = FSAMD_WING_T_INIT;
__constant__ double c_binom_even[kWingTerms * kWingTerms] = FSAMD_BINOM_EVEN_INIT;
__constant__ double c_binom_odd[kWingTerms * kWingTerms] = FSAMD_BINOM_ODD_INIT;

// singleabs.h:17-26
__device__ inline double sph_cubic_kernel(double q)
{
    const double norm = 32. / 4 / kPi;
    if (q >= 1) return 0;
    if (q < 0.5) return norm * (1 - 6 * q * q + 6 * q * q * q);
    const double r = 1. - q;
    return norm * (2 * (r * r * r));
}

// singleabs.h:31-42: quintic spline of support 1 as a sum of truncated fifth
// powers, 9/(40 pi) sum_k c_k max(0, r_k - 3q)^5, (r, c) = (3, 1), (2, -6), (1, 15)
__device__ inline double sph_quintic_kernel(double q)
{
    const double norm = 9. / 40 / kPi;
    if (q >= 1) return 0;
    const double t3 = 3. - 3. * q, t2 = 2. - 3. * q, t1 = 1. - 3. * q;
    double f = t3 * t3 * t3 * t3 * t3;
    if (t2 > 0) f -= 6. * (t2 * t2 * t2 * t2 * t2);
    if (t1 > 0) f += 15. * (t1 * t1 * t1 * t1 * t1);
    return norm * f;
}

// Kernel weight of tau_kern_inner (singleabs.h:158-163): the cubic or quintic
// spline, 3/(4 pi) for the tophat, and no weight (1) for any other id, which
// takes none of the reference's branches there.
__device__ inline double kernel_weight(int kernel, double q)
{
    if (kernel == kCubicSpline) return sph_cubic_kernel(q);
    if (kernel == kSphQuintic) return sph_quintic_kernel(q);
    if (kernel == kTopHat) return 3. / 4. / kPi;
    return 1.0;
}

// sqrt(x) for 1e-300 < x < 1e300 to about an ulp: the hardware's reciprocal
// square root, one step of Goldschmidt's iteration and a Newton correction.
__device__ inline double sqrt_nr(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

__device__ inline LineDesc line_of(const DepositArgs &A, int k) { return A.lines[k]; }

// Sightline data needed to recompute dr2 exactly as the binning did.
struct LosInfo {
    int ax;
    double key, lproj2;
};

__device__ inline LosInfo los_info(const DepositArgs &A, int s)
{
    LosInfo L;
    L.ax = A.axis[s];
    const double *c = &A.cofm[3 * (size_t)s];
    if (L.ax == 1) {
        L.key = c[1];
        L.lproj2 = c[2];
    } else if (L.ax == 2) {
        L.key = c[0];
        L.lproj2 = c[2];
    } else {
        L.key = c[0];
        L.lproj2 = c[1];
    }
    return L;
}

// index_table.cpp:70-87 with the particle coordinates of index_table.cpp:33-40
__device__ inline double pair_dr2(const LosInfo &L, const float *pp, double box)
{
    float first, second;
    if (L.ax == 1) {
        first = pp[1];
        second = pp[2];
    } else if (L.ax == 2) {
        first = pp[0];
        second = pp[2];
    } else {
        first = pp[0];
        second = pp[1];
    }
    double dr = fabs((double)first - L.key);
    if (dr > 0.5 * box) dr = box - dr;
    double d2 = dr * dr;
    dr = fabs((double)second - L.lproj2);
    if (dr > 0.5 * box) dr = box - dr;
    d2 += dr * dr;
    return d2;
}

// z mod nbins in [0, nbins) (absorption.cpp:257-259); walks stay within half a
// box of a pixel inside the box, so one add or subtract covers all but
// particles with extreme peculiar velocities.
__device__ inline int wrap_pixel(int z, int nbins)
{
    if (z >= 0 && z < nbins) return z;
    if (z < 0 && z >= -nbins) return z + nbins;
    if (z >= nbins && z < 2 * nbins) return z - nbins;
    int j = z % nbins;
    return j < 0 ? j + nbins : j;
}

// Box lengths by which pixel z lies outside [0, nbins): a walk from there is
// the same walk moved back by as many.
__device__ inline int box_shift(int z, int nbins)
{
    if (z >= 0 && z < nbins) return 0;
    const int q = z / nbins;
    return z - q * nbins < 0 ? q - 1 : q;
}

// A pixel of a walk that starts inside the box (walks go at most half a box).
__device__ inline int wrap_near(int z, int nbins)
{
    if (z >= nbins) z -= nbins;
    return z < 0 ? z + nbins : z;
}

// Per-pair constants of LineAbsorption::add_tau_particle and SingleAbsorber as
// the walks read them.  They lie in LDS: uniform over a lane group, they are
// read with broadcast loads where they are used and take no vector registers
// of the per-pixel loop.  Velocities in units of b carry the scale of the
// profile's argument (voigt_uscale, close to kUScale).
struct PairRec {
    double vel;      // velfac*ppos + pvel (absorption.cpp:234)
    double ibs;      // voigt_uscale / b
    double dss;      // sub-sample spacing, bintov / max(np - 1, 1) * ibs
    double scale;    // amp * dens * dvk / velfac: taulast = scale * (sample sum)
    double snear;    // scale / max(np - 1, 1), for the sum over sub-samples
    double qs;       // spacing of the kernel samples (singleabs.h:146-157), vhigh / 4 * ibs
    float W[4];      // kernel weights of the centre sample and the 3 above it (K is even)
    // Far wing: for a pixel centred at U (units of b) with |U| >= ufar the
    // 7 x np samples sum to Y (C0 + C1 Y + ... + C9 Y^9), Y = (ufar/U)^2.
    float Cw[kWingTerms];
    VoigtP vp;       // constants of the FP32 profile
    float ufsq;      // (voigt_uscale ufar)^2
    int zmax;
    int shape;       // near-step shape of the main kernel (step_shape)
    int k;           // the pair, counted from the work item's first (main kernel)
};
static_assert(sizeof(PairRec) == 144, "PairRec layout: W on a 16-byte boundary");

struct PairTau : PairRec {
    double b;        // btherm (absorption.cpp:220)
    double inv_b;
    double dvk;      // 2 vhigh / NGRID (singleabs.h:146)
    double vhigh, vdr2, vsmooth, aa;
    double ufar;
    double scale_nd; // amp * dvk / velfac (scale without the density)
    double temp;     // particle temperature
    int part;        // particle index
    int fp64, wide;
    int np;          // sub-samples per pixel (1 = midpoint)
    int wing_ready;  // Cw computed
};

// u times its scale, u = (vv_i - vouter)/b of the kernel sample i - 3 = j from the
// centre, from s = vouter/b times the scale: in FP64 and rounded once, so u keeps half an ulp
// where the two nearly cancel.
__device__ inline float sample_us(double qs, int j, double s) { return (float)__builtin_fma((double)j, qs, -s); }

__device__ inline void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Shuffle of a double from lane `src` of the same kG-lane group.
template <int kG>
__device__ inline double shfl_d(double v, int src)
{
    const long long b = __double_as_longlong(v);
    const int lo = __shfl((int)(b & 0xffffffffll), src, kG);
    const int hi = __shfl((int)(b >> 32), src, kG);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// sum_i K(q_i) Re w((vv_i - vouter)/b + i a), FP32 profile; the sample
// offsets from the FP64 anchor s, vouter/b times its scale.  kA3 = false: the light form
// of the profile (pairs with a <= kA3Drop).
template <bool kA3 = true>
__device__ inline float inner32(const PairRec &P, double s, const float *ptab)
{
    const VoigtP vp = P.vp;
    const double qs = P.qs;
    const float4 w4 = *(const float4 *)P.W;
    const float W[4] = {w4.x, w4.y, w4.z, w4.w};
    float sE = 0.0f, sG = 0.0f;
#pragma unroll  // full: 5% faster than unrolling by 2 at 256^3 and 512^3 (same operation order)
    for (int j = -3; j <= 3; ++j) {
        float E, G;
        voigt_terms<kA3>(vp, sample_us(qs, j, s), ptab, E, G);
        const float w = W[j < 0 ? -j : j];
        sE = __builtin_fmaf(w, E, sE);
        sG = __builtin_fmaf(w, G, sG);
    }
    return __builtin_fmaf(-vp.two_a_sqpi, sG, sE);
}

// The same sum for a pair whose samples may lie beyond the profile's table.
__device__ inline float inner32_wide(const PairRec &P, double s, const float *ptab)
{
    const VoigtP vp = P.vp;
    const double qs = P.qs;
    float sE = 0.0f, sG = 0.0f;
#pragma unroll 1
    for (int j = -3; j <= 3; ++j) {
        float E, G;
        voigt_terms<true, true>(vp, sample_us(qs, j, s), ptab, E, G);
        const float w = P.W[j < 0 ? -j : j];
        sE = __builtin_fmaf(w, E, sE);
        sG = __builtin_fmaf(w, G, sG);
    }
    return __builtin_fmaf(-vp.two_a_sqpi, sG, sE);
}

// One sample of that sum (i = 1 .. kNGrid - 1) with the FP64 profile and FP64
// kernel weights.
__device__ inline double sample64(const PairTau &P, double vouter, int kernel, int i, const double *gtab64)
{
    const double vv = i * P.dvk - P.vhigh;
    const double q = sqrt(P.vdr2 + vv * vv) / P.vsmooth;
    const double u = (vv - vouter) / P.b;
    return kernel_weight(kernel, q) * (P.aa <= (double)kA32Max ? voigt64_small(P.aa, u, gtab64) : voigt64(P.aa, u));
}

// The whole sum on one lane.
__device__ __noinline__ double inner64(const PairTau &P, double vouter, int kernel, const double *gtab64)
{
    double total = 0;
#pragma unroll 1
    for (int i = 1; i < kNGrid; ++i) total += sample64(P, vouter, kernel, i, gtab64);
    return total;
}

// amp*dens*tau_kern_outer(vlow, vlow+bintov)/velfac  (absorption.cpp:255; singleabs.h:104-126)
template <bool k64>
__device__ inline double taulast_pixel(const PairTau &P, double vlow, double bintov, double velfac, int kernel,
                                       const float *ptab, const double *gtab64)
{
    const double vhighp = vlow + bintov;
    const double width = vhighp - vlow;
    if (!k64) {
        const double U = (vlow + 0.5 * bintov) * P.inv_b;
        if (fabs(U) >= P.ufar) {
            const float Y = (float)(P.ufar * P.ufar) * __builtin_amdgcn_rcpf((float)(U * U));
            float S = P.Cw[kWingTerms - 1];
#pragma unroll
            for (int t = kWingTerms - 2; t >= 0; --t) S = __builtin_fmaf(S, Y, P.Cw[t]);
            return P.scale * (double)(S * Y);
        }
    }
    auto inner = [&](double v) {
        return k64 ? inner64(P, v, kernel, gtab64)
               : (double)(P.wide ? inner32_wide(P, v * P.ibs, ptab) : inner32(P, v * P.ibs, ptab));
    };
    if (width < P.b / 2.) return P.scale * inner((vhighp + vlow) / 2.);
    const int np = 2 * ceil(width / (P.b / 2.) / 2) + 1.;
    const double dv = width / (np - 1);
    double total = 0.5 * inner(vlow);
    for (int i = 1; i < np - 1; ++i) total += inner(i * dv + vlow);
    total += 0.5 * inner(vhighp);
    return P.scale * (total / (np - 1));
}

template <int kG>
__device__ inline double group_sum(double v)
{
#pragma unroll
    for (int o = kG / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kG);
    return v;
}

// taulast_pixel<true> of one pixel by a whole lane group, its 7 x np samples
// over the lanes: a pixel that decides a tail cut is usually the only one of
// its group, and its samples in turn on one lane would be the walk's latency.
template <int kG>
__device__ inline double taulast_group64(const PairTau &P, double vlow, double bintov, int kernel, int glane,
                                         const double *gtab64)
{
    const double vhighp = vlow + bintov;
    const double width = vhighp - vlow;
    int np = 1;
    if (!(width < P.b / 2.)) np = 2 * ceil(width / (P.b / 2.) / 2) + 1.;
    const double dv = width / (np - 1);
    double total = 0;
    for (int m = glane; m < (kNGrid - 1) * np; m += kG) {
        const int j = m / (kNGrid - 1), i = m - j * (kNGrid - 1) + 1;
        const double v = np == 1 ? (vhighp + vlow) / 2. : j == 0 ? vlow : j == np - 1 ? vhighp : j * dv + vlow;
        const double h = sample64(P, v, kernel, i, gtab64);
        total += np > 1 && (j == 0 || j == np - 1) ? 0.5 * h : h;
    }
    total = group_sum<kG>(total);
    return P.scale * (np == 1 ? total : total / (np - 1));
}

// x^n for 0 <= n < 16 by squaring, with a uniform instruction stream.
__device__ inline double ipow(double x, int n)
{
    double r = 1.0;
#pragma unroll
    for (int bit = 0; bit < 4; ++bit) {
        if (n & (1 << bit)) r *= x;
        x *= x;
    }
    return r;
}

// Far-wing coefficients of one pair.  The sample offsets from the pixel
// centre are c = x_i - y_j with x_i = vv_i/b the kernel samples (weights W_i)
// and y_j the sub-sample offsets of tau_kern_outer (singleabs.h:110-125,
// trapezoid weights t_j); both sets are symmetric, so the even moments of c
// factor:  m_n = sum_k C(2n,2k) X_k Y_(n-k),  X_k = sum W_i x_i^2k,
// Y_k = sum t_j y_j^2k.  Offsets are measured in units of ufar so that all
// coefficients stay within FP32 range:  C'_n = sum_(k+j=n) g_k ufar^(-2k-2)
// C(2n+1,2j) m'_j with m'_j the moments of c/ufar.  Lane n < 10 builds the
// n-th moments and coefficient and stores C'_n.  The kernel samples are
// x_i = (vhigh/b)(i-3)/4 (singleabs.h:146-149), so X_k takes the three
// positive offsets with the summed weights of each +- pair; Y_k = h^2k T[m][k]
// for a pixel of half-width h in np = m + 1 sub-samples, with T tabulated
// exactly (wing_table.h) up to m = FSAMD_WING_TMAX.
template <int kG>
__device__ inline void wing_setup(PairTau &P, double bintov, int lane)
{
    const double inv_u = 1.0 / P.ufar;
    const int np = P.np;
    const int m1 = np - 1;
    const int n = lane < kWingTerms ? lane : 0;
    // Y_n: pixel sub-samples
    double Yn;
    if (m1 == 0) {
        Yn = n == 0 ? 1.0 : 0.0;
    } else if (m1 <= FSAMD_WING_TMAX) {
        const double h = 0.5 * bintov * P.inv_b * inv_u;
        Yn = ipow(h * h, n) * c_wing_T[m1 * kWingTerms + n];
    } else {
        const double dv = bintov / m1;
        Yn = 0.0;
        for (int j = 0; j < np; ++j) {
            const double y = (j * dv - 0.5 * bintov) * P.inv_b * inv_u;
            const double t = ((j == 0 || j == m1) ? 0.5 : 1.0) / m1;
            Yn += t * ipow(y * y, n);
        }
    }
    // m'_n = sum_k C(2n,2k) X_k Y_(n-k), X_k by running powers
    const double c4 = 0.25 * P.vhigh * P.inv_b * inv_u, c5 = 2.0 * c4, c6 = 3.0 * c4;
    const double x4 = c4 * c4, x5 = c5 * c5, x6 = c6 * c6;
    const double w4 = 2.0 * P.W[1], w5 = 2.0 * P.W[2], w6 = 2.0 * P.W[3];
    double p4 = 1.0, p5 = 1.0, p6 = 1.0, mom = 0.0;
#pragma unroll 1
    for (int k = 0; k < kWingTerms; ++k) {
        double xk = w4 * p4 + w5 * p5 + w6 * p6;
        if (k == 0) xk += (double)P.W[0];
        p4 *= x4;
        p5 *= x5;
        p6 *= x6;
        const double yk = shfl_d<kG>(Yn, n - k < 0 ? 0 : n - k);
        if (k <= n) mom += c_binom_even[n * kWingTerms + k] * xk * yk;
    }
    // C'_n = sum_(k+j=n) g_k ufar^(-2k-2) C(2n+1, 2j) m'_j
    const double a = P.aa, a2 = a * a, iu2 = inv_u * inv_u, u2 = P.ufar * P.ufar;
    // j = 0..n walks k = n..0: start from ufar^(-2n-2)
    double C = 0.0, gs = a * (1.0 / kSqrtPi) * iu2 * ipow(iu2, n);
#pragma unroll 1
    for (int j = 0; j < kWingTerms; ++j) {
        const double mj = shfl_d<kG>(mom, j);
        if (j > 0) gs *= u2;
        if (j <= n) {
            const int k = n - j;
            const double binom = c_binom_odd[n * kWingTerms + j];
            const double qk = k > 0 ? c_wing_q[k - 1] : 0.0;
            C += gs * (c_wing_p[k] - a2 * qk) * binom * mj;
        }
    }
    if (lane < kWingTerms) P.Cw[lane] = (float)C;
}

// Sub-sample grid of one walk step in the main kernel.  A step evaluates one
// 7-sample kernel sum per lane and round, on the sub-sample grid of
// tau_kern_outer (singleabs.h:104-126) laid out across the lanes: adjacent
// pixels share their boundary sub-sample, so a step of p pixels with np
// sub-samples each needs p (np - 1) + 1 sums; midpoint pixels (np = 1) need
// one each.  Pairs whose grid exceeds kRoundsMax rounds take the FP64 path.
constexpr int kRoundsMax = 4;

struct StepShape {
    int nm1;      // np - 1 (0: midpoint)
    int pstep;    // pixels per step
    __device__ inline int packed() const { return nm1 | (pstep << 16); }
};
static_assert(64 * kRoundsMax < (1 << 16), "StepShape::packed");

__device__ inline StepShape unpack_shape(int s) { return StepShape{s & 0xffff, s >> 16}; }

// A step's work beside its sums (the pair's state, trapezoid, tail cut, deposit)
// costs as much as one and a half rounds of sums, so groups of 16 and 32 lanes
// take two rounds where pixels have several sub-samples: 16 lanes 15 pixels of 3
// in place of 7, 7 of 5 in place of 3.  256^3 x 5000 x 2048, two lines, 89.9 ->
// 85.1 ms; with metals (12288 x 1024) 268 -> 206; top-hat, 512^3, 193 -> 153.
// Three or four rounds cost more past the cut than they save (214 and 225 with
// metals), and so do two of 64 lanes (323 -> 362).  Wider grids: as many rounds
// as two pixels take.
__device__ inline StepShape step_shape(int np, int kg)
{
    StepShape sh;
    sh.nm1 = np - 1;
    sh.pstep = kg;
    if (sh.nm1 > 0) {
        const int rounds = sh.nm1 >= kg ? min(kRoundsMax, (2 * sh.nm1 + kg) / kg) : kg < 64 ? 2 : 1;
        sh.pstep = min(kg, (kg * rounds - 1) / sh.nm1);
    }
    return sh;
}

// A fix-up entry's dir: the direction of a deferred walk, or a whole pair.
enum { kFixPair64 = 0, kFixPair = 2 };

// Append a walk to the fix-up list.  The counter is 64-bit, so it cannot wrap
// within a launch; entries past the capacity only raise the overflow flag.
__device__ inline void push_fixup(const DepositArgs &A, long long k, int item, int z0, int count, int dir)
{
    const unsigned long long slot = atomicAdd(&A.fix_count[0], 1ull);
    if (slot < (unsigned long long)A.fix_cap)
        A.fix[slot] = Fixup{k, item, z0, count, dir};
    else
        atomicOr(&A.fix_count[1], 1ull);
}

// Lanes of a wave are split into groups of kG lanes; each group walks its own
// (pair, direction) stream, kG consecutive pixels per step.
template <int kG>
__device__ inline unsigned long long group_bits(unsigned long long m, int lane)
{
    if (kG == 64) return m;
    return (m >> ((lane / kG) * kG)) & ((1ull << kG) - 1ull);
}

// The first lane of this lane's group whose bit is set in m (counted from the
// group's first lane), kG if none.
template <int kG>
__device__ inline int group_first(unsigned long long m, int lane)
{
    if (kG == 64) return m ? __builtin_ctzll(m) : 64;
    unsigned b = lane & 32 ? (unsigned)(m >> 32) : (unsigned)m;
    if (kG == 32) return b ? __builtin_ctz(b) : 32;
    b = (b >> (lane & 16)) & 0xffffu;
    return __builtin_ctz(b | 0x10000u);
}

// Bit `i` (< kG) of this lane's group in m.
template <int kG>
__device__ inline bool group_bit(unsigned long long m, int lane, int i)
{
    if (kG == 64) return (m >> i) & 1ull;
    const unsigned b = lane & 32 ? (unsigned)(m >> 32) : (unsigned)m;
    return (b >> ((kG == 16 ? lane & 16 : 0) + i)) & 1u;
}

struct LaneStats {
    long long pairs = 0, pixels = 0, px64 = 0, pairs64 = 0, samples = 0, evaluated = 0, sums = 0, far = 0;
    // wave cycles (s_memtime, counted by lane 0 of each wavefront) in pair
    // set-up, far-wing set-up and walk steps, wave iterations, and the
    // iterations in which at least one group set up a pair
    long long cyc_setup = 0, cyc_wing = 0, cyc_walk = 0, iters = 0, setup_iters = 0;
};

// Per-pair scalars of LineAbsorption::add_tau_particle (absorption.cpp:218-247)
// and SingleAbsorber's constructor (singleabs.h:81-90).
struct PairConsts {
    double vel, b, inv_b, dvk, vhigh, vdr2, vsmooth, aa, scale, scale_nd, ufar;
    float temp;
    int zmax, np, fp64, wide;
};

// Pair kk (the particle at pair_part[kk]).  Returns false if the particle does
// not reach the sightline (absorption.cpp:232; on the Voronoi mesh, if it owns
// no segment of it, absorption.cpp:221-229).  fp64 routes the pair to the
// FP64 path.  wide: samples of a near step may lie beyond the profile's table
// (supports of more than 5700 Doppler widths); such a pair is walked in FP32 by the
// fix-up kernel, and by a launch of its own in the adjoint: their code in the main
// kernels costs every call 2.4% (256^3 x 5000 x 2048, two lines, 76.5 -> 78.3 ms) and the
// adjoint's 8%.  In FP64, the other way out, 43 such particles of 32768 took half of
// a call (1.05 ms, 0.58 so) and 4700 three quarters (8.3 ms, 3.6 so).
__device__ inline bool pair_consts(const DepositArgs &A, int line, const LineDesc &L, const LosInfo &los,
                                   long long kk, int max_sums, PairConsts &C)
{
    const int p = A.pair_part[kk];
    const float4 r0 = *(const float4 *)&A.rec[p].x;
    const float4 r1 = *(const float4 *)&A.rec[p].vx;
    const float pp[3] = {r0.x, r0.y, r0.z};
    const float temp = r1.w;
    const float dens = A.rec[p].dens[line];
    const float ppos = pp[los.ax - 1];
    const float pvel = los.ax == 1 ? r1.x : (los.ax == 2 ? r1.y : r1.z);
    const double b = L.bfac * sqrt((double)temp);
    double pos1 = (double)ppos, vdr2, vsmooth, vhigh;
    if (A.seg) {
        // Voronoi mesh: the segment ends take the places of dr2 and h
        // (part_int.cpp:42-43), the segment centre that of the position and
        // the kernel spans half the segment (absorption.cpp:221-237,
        // singleabs.h:84-88)
        const float2 sg = A.seg[kk];
        const double lo = (double)sg.x;
        if (lo > 2 * A.vbox / A.velfac || (double)sg.y > 2 * A.vbox / A.velfac) return false;
        pos1 = (lo + (double)sg.y) / 2.;
        vdr2 = A.velfac * lo;
        vsmooth = A.velfac * (double)sg.y;
        vhigh = (vdr2 > 0 && vsmooth > 0) ? (vsmooth - vdr2) / 2. : 0;
    } else {
        const double dr2 = pair_dr2(los, pp, A.box);
        const float smooth = r0.w;
        const float sm2 = smooth * smooth;
        if ((double)sm2 - dr2 <= 0) return false;            // absorption.cpp:232
        double val1 = A.velfac * dr2;
        val1 *= A.velfac;
        vdr2 = val1;
        vsmooth = A.velfac * (double)smooth;
        vhigh = vsmooth * vsmooth > vdr2 ? sqrt(vsmooth * vsmooth - vdr2) : 0;   // singleabs.h:83
    }
    const double vel = A.velfac * pos1 + (double)pvel;
    const double inv_b = 1.0 / b;
    // a = voigt_fac/b, amp = sigma_a/sqrt(pi) (c/1e5)/b (absorption.cpp:238,244),
    // by one reciprocal: within 2 ulp of the reference's quotients
    const double aa = L.voigt_fac * inv_b;
    const double bintov = A.vbox / A.nbins;
    const double amp = L.sigma_a * (kLight / 1e5 / kSqrtPi) * inv_b;
    const double dvk = 2. * vhigh / kNGrid;
    const double xs = bintov * inv_b;     // bintov / (b/2) / 2 (singleabs.h:114)
    int np = 1;
    if (!(bintov < b / 2.)) np = 2 * ceil(xs) + 1.;
    // The reference sizes the sub-sample grid per pixel from vhigh - vlow,
    // which equals bintov up to the rounding of vlow + bintov (~1e-13
    // relative); the walk uses one grid per pair, so a pair whose grid could
    // differ between pixels (bintov/b at a switch point to 1e-12) goes to the
    // FP64 path, which follows the reference pixel by pixel.
    const bool grid_edge = fabs(bintov - b / 2.) <= 1e-12 * bintov || (np > 1 && fabs(xs - rint(xs)) <= 1e-12 * xs);
    const double dmax = (vhigh - dvk) * inv_b + (np > 1 ? 0.5 * bintov * inv_b : 0.0);
    C.ufar = fmax(7.0 + dmax, 3.0 * dmax);
    // pixels wider than max_sums sub-samples do not fit one walk step; a near step
    // reaches up to 4 * 64 sub-samples of half a b past ufar
    const double reach = C.ufar + dmax + 130.0;
    C.wide = !(reach <= kVoigtUMax);
    C.fp64 = A.force_fp64 || !(aa <= (double)kA32Max) || grid_edge || np - 1 > max_sums - 1 ||
             !(reach <= kVoigtUWide);
    C.vel = vel;
    C.b = b;
    C.inv_b = inv_b;
    C.dvk = dvk;
    C.vhigh = vhigh;
    C.vdr2 = vdr2;
    C.vsmooth = vsmooth;
    C.aa = aa;
    C.scale = amp * (double)dens * dvk * A.inv_velfac;
    C.scale_nd = amp * dvk * A.inv_velfac;
    C.temp = temp;
    C.zmax = (int)floor(vel / bintov);
    C.np = np;
    return true;
}

// Kernel weight of interior sample i (singleabs.h:145-152).
__device__ inline float sample_weight(const DepositArgs &A, const PairConsts &C, int i)
{
    const double vv = (i + 1) * C.dvk - C.vhigh;
    const double q = sqrt(C.vdr2 + vv * vv) / C.vsmooth;
    return (float)kernel_weight(A.kernel, q);
}

// Set up one pair in the wave's LDS slot; returns false if the particle does
// not reach the sightline.  Every lane of the wave calls it.
template <int kG>
__device__ inline bool setup_pair(const DepositArgs &A, int line, const LineDesc &L, const LosInfo &los, long long kk,
                                  PairTau &P, int lane, int max_sums = 1 << 30)
{
    PairConsts C;
    if (!pair_consts(A, line, L, los, kk, max_sums, C)) return false;
    const int p = A.pair_part[kk];
    const double bintov = A.vbox / A.nbins;
    wave_sync();   // the previous pair's constants are no longer read
    if (lane < 4) P.W[lane] = sample_weight(A, C, lane + 3);
    if (lane == 0) {
        P.vel = C.vel;
        P.b = C.b;
        P.inv_b = C.inv_b;
        P.dvk = C.dvk;
        P.vhigh = C.vhigh;
        P.vdr2 = C.vdr2;
        P.vsmooth = C.vsmooth;
        P.aa = C.aa;
        P.zmax = C.zmax;
        P.fp64 = C.fp64;
        P.wide = C.wide;
        P.vp = make_voigt_p(C.fp64 ? 0.0 : C.aa, C.aa <= (double)kA3Drop);
        P.scale = C.scale;
        P.scale_nd = C.scale_nd;
        P.temp = (double)C.temp;
        P.part = p;
        P.np = C.np;
        P.ufar = C.ufar;
        P.ibs = voigt_uscale(P.vp, C.fp64 ? 0.0 : C.aa) * C.inv_b;
        P.qs = 0.25 * C.vhigh * P.ibs;
        P.wing_ready = 0;
    }
    wave_sync();
    return true;
}

// The main kernel sets pairs up in batches, one pair per lane of a wavefront,
// into the wavefront's kRecs records: the FP64 set-up (pair constants, kernel
// weights and the ten far-wing coefficients) runs on up to kRecs lanes at once
// instead of on the few lanes of one lane group.  A group walks its pair in
// the record where it lies.  Which records are free, and which hold pairs of
// either class, are three masks of the wavefront: the groups take pairs of one
// class as long as there are some, so that the near steps of the wavefront
// mostly run the light code (a step runs the full code, 180 instead of 85
// instructions a sum, if any of its groups needs it) and its four groups the
// same number of rounds.  The one class is the light profile on several
// sub-samples; the other the full profile, and midpoint pixels: fields have few of
// one or of the other, and a class of each costs more in refills than it
// saves.  Against a ring in claim order whose records were copied to a slot per
// group: 99.3 -> 89.6 ms at 256^3 x 5000 x 2048, two lines; 301 -> 269 with a metal
// line (half of its pairs full) at 12288 x 1024; midpoint pixels apart 84.2 -> 80.5
// and 202.5 -> 203.2.
constexpr int kRecs = kWaveClaim;
static_assert(kRecs == 32, "the record masks are 32-bit");
// Fewest free records worth a set-up, whose cost hardly depends on their number,
// while others wait: 12 -> 24 82.2 -> 80.5 and 208.5 -> 203.2 ms; 28 the same.
constexpr int kRefillRoom = 24;

// The far-wing coefficients of wing_setup for one pair, all ten on one lane
// (the batched set-up), with
//   C_n = a/(sqrt(pi) ufar^2) sum_(k<=n) (p_k - a^2 q_(k-1)) ufar^(-2k) C(2n+1, 2(n-k)) m_(n-k):
// every term is positive and the powers of 1/ufar that underflow for wide
// supports (FP32: k > 4 at 1e4 Doppler widths) are those of negligible terms.  With
// a/(sqrt(pi)) ufar^(-2n-2) taken first FP32 lost whole coefficients from ufar = 150
// on: tau was off by 5e-5 at supports of 3000 b, the temperature response of the far
// wing by 1.4e-5 at 300 b and 1.1e-4 at 1000 b (now 2e-7; the series' own truncation
// is 7e-7 at |U| = ufar).  c0 = vhigh/b and h = half the pixel
// width over b, both in units of ufar; W the kernel weights at offsets 0, 1/4, 1/2,
// 3/4 of vhigh; m1 = sub-samples - 1 (at most FSAMD_WING_TMAX).  Real: float for
// the optical depth, double for the adjoint (2.1M particles, 1024 sightlines, forward
// and adjoint 15.1 -> 15.5 ms).
// kAdj: CwT receives the coefficients of the sum of W (H + u dH/du + a dH/da),
// from that operator on the term a p_k u^(-2k-2) - a^3 q_(k-1) u^(-2k-2); its
// leading one is zero.
template <typename Real, bool kAdj>
__device__ __noinline__ void wing_coeffs(Real c0, Real h, int m1, float W0, float W1, float W2, float W3, Real a,
                                         Real ufar, float *Cw, float *CwT)
{
    Real Y[kWingTerms];
    if (m1 == 0) {
        Y[0] = 1;
#pragma unroll
        for (int n = 1; n < kWingTerms; ++n) Y[n] = 0;
    } else {
        const Real h2 = h * h;
        Real pw = 1;
#pragma unroll
        for (int n = 0; n < kWingTerms; ++n) {
            Y[n] = pw * (Real)c_wing_T[m1 * kWingTerms + n];
            pw *= h2;
        }
    }
    // kernel samples at +-(c0/4, c0/2, 3c0/4) and 0
    const Real x1 = (Real)0.0625 * c0 * c0, x2 = (Real)0.25 * c0 * c0, x3 = (Real)0.5625 * c0 * c0;
    const Real w1 = 2 * (Real)W1, w2 = 2 * (Real)W2, w3 = 2 * (Real)W3;
    Real X[kWingTerms];
    Real p1 = 1, p2 = 1, p3 = 1;
#pragma unroll
    for (int k = 0; k < kWingTerms; ++k) {
        X[k] = fma(w1, p1, fma(w2, p2, k == 0 ? fma(w3, p3, (Real)W0) : w3 * p3));
        p1 *= x1;
        p2 *= x2;
        p3 *= x3;
    }
    Real m[kWingTerms];
#pragma unroll
    for (int n = 0; n < kWingTerms; ++n) {
        Real t = 0;
#pragma unroll
        for (int k = 0; k <= n; ++k) t = fma((Real)c_binom_even[n * kWingTerms + k] * X[k], Y[n - k], t);
        m[n] = t;
    }
    const Real iu = 1 / ufar, iu2 = iu * iu, a2 = a * a, lead = a * (Real)(1.0 / kSqrtPi) * iu2;
    Real g[kWingTerms], gT[kWingTerms];
    Real pw = 1;   // ufar^(-2k)
#pragma unroll
    for (int k = 0; k < kWingTerms; ++k) {
        const Real pk = (Real)c_wing_p[k], qk = k > 0 ? (Real)c_wing_q[k - 1] : 0;
        g[k] = pw * (pk - a2 * qk);
        if (kAdj) gT[k] = pw * ((2 * k - 2) * a2 * qk - 2 * k * pk);
        pw *= iu2;
    }
#pragma unroll
    for (int n = 0; n < kWingTerms; ++n) {
        Real cn = 0, cT = 0;
#pragma unroll
        for (int j = 0; j <= n; ++j) {
            const Real bm = (Real)c_binom_odd[n * kWingTerms + j] * m[j];
            cn = fma(g[n - j], bm, cn);
            if (kAdj) cT = fma(gT[n - j], bm, cT);
        }
        Cw[n] = (float)(lead * cn);
        if (kAdj) CwT[n] = (float)(lead * cT);
    }
}

// K(q) (singleabs.h:17-42 and kernel_weight), q^2 > 0, without branches on q.
__device__ inline float kernel_weight_q2(int kernel, double q2)
{
    const double q = sqrt_nr(q2 + 1e-290);
    if (kernel == kCubicSpline) {
        const double t = fmax(1.0 - q, 0.0), h = fmax(0.5 - q, 0.0);
        return (float)(32. / 4 / kPi * 2.0 * (t * t * t - 4.0 * (h * h * h)));
    }
    if (kernel == kSphQuintic) {
        const double t3 = fmax(3.0 - 3.0 * q, 0.0), t2 = fmax(2.0 - 3.0 * q, 0.0), t1 = fmax(1.0 - 3.0 * q, 0.0);
        const double p3 = t3 * t3, p2 = t2 * t2, p1 = t1 * t1;
        return (float)(9. / 40 / kPi * (p3 * p3 * t3 - 6.0 * (p2 * p2 * t2) + 15.0 * (p1 * p1 * t1)));
    }
    return kernel == kTopHat ? (float)(3. / 4. / kPi) : 1.0f;
}

// The record of this lane's pair if its bit is set in m: the r-th pair goes to
// the r-th free record.  Lane l stands for record l and sends its number to the
// lane of its rank; `used` says whether record l gets a pair.
__device__ inline int free_record(unsigned free, unsigned long long m, int lane, bool &used)
{
    const bool isfree = lane < kRecs && ((free >> (lane & 31)) & 1u);
    const int frank = __popc(free & ((1u << (lane & 31)) - 1u));
    used = isfree && frank < __popcll(m);
    const int nth = __builtin_amdgcn_ds_permute(4 * (isfree ? frank : 63), lane);
    return __shfl(nth, __popcll(m & ((1ull << lane) - 1ull)), 64);
}

// Pairs to claim for a wavefront: its free records, fewer near the end of the
// item so that the block's wavefronts finish together.
__device__ inline int pairs_wanted(long long left, int waves, int groups, int nfree)
{
    const long long share = left / (2 * waves);
    int want = nfree;
    if (share < want) want = (int)(share > 2 * groups ? share : 2 * groups);
    return min(want, nfree);
}

// Claim up to `want` (at most the free records) pairs of item w for the
// wavefront, set them up one per lane and put those of the main kernel into free
// records; FP64 and wide pairs go straight to the fix-up list.  Every lane of the
// wavefront calls it; `more` says whether the item has pairs left.
template <int kG, bool kStats>
__device__ inline void refill_wave(const DepositArgs &A, const WorkItem &w, int gitem, const LineDesc &L,
                                   const LosInfo &los, unsigned long long *next, PairRec *recs, int lane, int want,
                                   unsigned &free, unsigned &light, unsigned &full, bool &more, LaneStats &st)
{
    unsigned long long base = 0;
    if (lane == 0) base = atomicAdd(next, (unsigned long long)want);
    base = (unsigned long long)__shfl((long long)base, 0, 64);
    const long long kk = (long long)base + lane;
    const double bintov = A.vbox / A.nbins;
    bool enq = false;
    PairConsts C;
    if (lane < want && kk < w.p1 && pair_consts(A, w.line, L, los, kk, kG * kRoundsMax, C)) {
        if (kStats) st.pairs++;
        if (C.fp64 || C.wide) {
            if (kStats) st.pairs64 += C.fp64;
            push_fixup(A, kk, gitem, C.zmax, A.nbins / 2, C.fp64 ? kFixPair64 : kFixPair);
        } else {
            enq = true;
        }
    }
    const unsigned long long m = __ballot(enq);
    bool used;
    const int slot = free_record(free, m, lane, used);
    wave_sync();   // the records' former pairs have been read
    if (enq) {
        PairRec &r = recs[slot];
        const int shift = box_shift(C.zmax, A.nbins);
        // the walk uses the light form of the profile for a <= kA3Drop, as a
        // property of the pair: its coefficients are zero, so the full form
        // gives the same values and the result does not depend on which
        // pairs share a wavefront
        const VoigtP vp = make_voigt_p(C.aa, C.aa <= (double)kA3Drop);
        r.vp = vp;
        const double us = voigt_uscale(vp, C.aa), ibs = us * C.inv_b;
        const double inv_m = C.np > 1 ? 1.0 / (C.np - 1) : 1.0;
        r.vel = shift ? C.vel - shift * A.vbox : C.vel;
        r.zmax = C.zmax - shift * A.nbins;
        r.ibs = ibs;
        r.dss = bintov * inv_m * ibs;
        r.scale = C.scale;
        r.snear = C.scale * inv_m;
        r.qs = 0.25 * C.vhigh * ibs;
        r.k = (int)(kk - w.p0);   // a row has fewer than 2^31 pairs (one per particle)
        const double inv_s2 = 1.0 / (C.vsmooth * C.vsmooth);
        float W[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const double vv = (i + 4) * C.dvk - C.vhigh;
            W[i] = kernel_weight_q2(A.kernel, (C.vdr2 + vv * vv) * inv_s2);
        }
        *(float4 *)r.W = make_float4(W[0], W[1], W[2], W[3]);
        // the walk compares with ufar rounded to FP32, the unit of the coefficients
        const float ufar = (float)C.ufar;
        r.ufsq = (float)((us * ufar) * (us * ufar));
        const StepShape sh = step_shape(C.np, kG);
        r.shape = sh.packed();
        // far-wing coefficients, in units of that ufar
        const double iu = 1.0 / (double)ufar;
        wing_coeffs<float, false>((float)(C.vhigh * C.inv_b * iu), (float)(0.5 * bintov * C.inv_b * iu), sh.nm1, W[0], W[1],
                           W[2], W[3], (float)C.aa, ufar, r.Cw, nullptr);
    }
    wave_sync();
    const unsigned mine = (unsigned)__ballot(used);
    const PairRec &mr = recs[lane & 31];
    const unsigned other = (unsigned)__ballot(used && (mr.vp.a3 != 0.0f || unpack_shape(mr.shape).nm1 == 0));
    free &= ~mine;
    light |= mine & ~other;
    full |= other;
    more = (long long)base + want < w.p1;
}

// Voigt samples the reference evaluates for one pixel (singleabs.h:110-125).
__device__ inline int pixel_samples(const PairRec &P, double vlow, double bintov)
{
    const double b = kUScale / P.ibs;
    const double vhighp = vlow + bintov;
    const double width = vhighp - vlow;
    if (width < b / 2.) return kNGrid - 1;
    const int np = 2 * ceil(width / (b / 2.) / 2) + 1.;
    return (kNGrid - 1) * np;
}

template <bool kLds>
__device__ inline void row_add(double *p, double v)
{
    if (kLds)
        atomicAdd(p, v);          // ds_add_f64
    else
        unsafeAtomicAdd(p, v);    // global_atomic_add_f64
}

// The FP32 deposit kernel defers any decision it cannot make exactly; the
// fix-up kernel re-evaluates guard-band pixels in FP64, or evaluates whole
// pairs in FP64.
enum { kWalkGuarded = 1, kWalkFull64 = 2 };

// One step of kG consecutive pixels of a fix-up walk (lane glane of the group),
// each pixel evaluated on its own as tau_kern_outer does (singleabs.h:104-126,
// sub-sample grid from the pixel's own vhigh - vlow), in FP32 with the guard
// band re-evaluated in FP64 (kWalkGuarded), or all in FP64.  Returns true when
// the walk is over (tail cut reached or end of the window).
template <int kG, int kMode, bool kStats>
__device__ inline bool walk_chunk(const DepositArgs &A, const PairTau &P, double *row, const float *ptab,
                                  const double *gtab64, int z0, int dir, int count, int c, int lane, LaneStats &st,
                                  int &walked)
{
    const int glane = lane % kG;
    const double bintov = A.vbox / A.nbins;
    const double tt = A.tautail;
    const int idx = c + glane;
    const bool valid = idx < count;
    const int z = z0 + dir * idx;
    double t = 0, vlow = 0;
    if (valid) {
        vlow = z * bintov - P.vel;                                  // absorption.cpp:252
        t = taulast_pixel<kMode == kWalkFull64>(P, vlow, bintov, A.velfac, A.kernel, ptab, gtab64);
        if (kStats) {
            st.evaluated++;
            if (kMode != kWalkFull64 && fabs((vlow + 0.5 * bintov) * P.inv_b) >= P.ufar)
                st.far++;
            else
                st.sums += pixel_samples(P, vlow, bintov) / (kNGrid - 1);
        }
    }
    if (kMode == kWalkGuarded) {
        // pixels past the first certain cut are not needed
        const unsigned long long sure =
            group_bits<kG>(__ballot(valid && t < tt && !(fabs(t - tt) <= kGuard * tt)), lane);
        unsigned long long band = group_bits<kG>(__ballot(valid && fabs(t - tt) <= kGuard * tt), lane);
        if (sure) band &= (sure & (0ull - sure)) - 1ull;
        while (band) {
            const int g = __builtin_ctzll(band);
            band &= band - 1ull;
            const double t64 = taulast_group64<kG>(P, (z0 + dir * (c + g)) * bintov - P.vel, bintov, A.kernel, glane,
                                                   gtab64);
            if (glane == g) {
                t = t64;
                if (kStats) st.px64++;
            }
        }
    }
    const unsigned long long mb = group_bits<kG>(__ballot(valid && t < tt), lane);
    const int first = mb ? __builtin_ctzll(mb) : kG;
    if (valid && glane <= first) {
        row_add<false>(&row[wrap_pixel(z, A.nbins)], t);
        if (kStats) {
            st.pixels++;
            st.samples += pixel_samples(P, vlow, bintov);
        }
    }
    if (mb != 0) {
        walked = c + first + 1;
        return true;
    }
    if (c + kG >= count) {
        walked = count;
        return true;
    }
    return false;
}

// The tail cut's guard band as two limits: a pixel above hi goes on, below lo
// it ends the walk, between them FP64 decides (the fix-up kernel).
struct CutBand {
    double lo, hi;
};

__device__ inline CutBand cut_band(double tautail)
{
    const double guard = kGuard * fabs(tautail);
    return CutBand{tautail - guard, tautail + guard};
}

// A walk that has reached the far wing, by the whole wavefront, 64 pixels at a
// time: |U| only grows from there, so this ends the walk.  zf: its next pixel,
// count: the pixels left.  P and the arguments are uniform, so the tail cut
// (deposit up to and including the first pixel below tautail,
// absorption.cpp:260-263) is scalar work.  In steps of 4 x kG pixels by the
// walk's own group (four rounds of ~90 instructions in which the other groups
// idle) the kernel took 127 instead of 94 ms at 256^3 x 5000 x 2048, two lines.
// Returns the pixels walked, or -1 where the decision went to the fix-up
// kernel.
template <bool kLds, bool kStats>
__device__ inline int far_walk(const DepositArgs &A, const PairRec &P, double *row, int zf, int dir, int count,
                               const CutBand &cut, int lane, LaneStats &st, long long k, int item)
{
    const double bintov = A.vbox / A.nbins;
    for (int i0 = 0; i0 < count; i0 += 64) {
        const int i = i0 + lane;
        const bool valid = i < count;
        const int z = zf + dir * i;
        const double vlow = z * bintov - P.vel;
        const double Us = (vlow + 0.5 * bintov) * P.ibs;
        const float Y = P.ufsq * __builtin_amdgcn_rcpf((float)(Us * Us));
        float S = P.Cw[kWingTerms - 1];
#pragma unroll
        for (int q = kWingTerms - 2; q >= 0; --q) S = __builtin_fmaf(S, Y, P.Cw[q]);
        const double t = P.scale * (double)(S * Y);
        const unsigned long long stop = __ballot(valid && t <= cut.hi), below = __ballot(valid && t < cut.lo);
        const int first = stop ? __builtin_ctzll(stop) : 64;
        const bool sure = stop && ((below >> (first & 63)) & 1ull);
        if (kStats && valid) {
            st.evaluated++;
            st.far++;
        }
        if (valid && (lane < first || (lane == first && sure))) {
            row_add<kLds>(&row[wrap_near(z, A.nbins)], t);
            if (kStats) {
                st.pixels++;
                st.samples += pixel_samples(P, vlow, bintov);
            }
        }
        if (stop) {
            if (sure) return i0 + first + 1;
            // the FP32 value of the deciding pixel is too close to tautail
            if (lane == 0) push_fixup(A, k, item, zf + dir * (i0 + first), count - (i0 + first), dir);
            return -1;
        }
    }
    return count;
}

// One near step of a walk (lane glane of a kG-lane group): the next sh.pstep
// pixels from zf in direction dir, on the sub-sample grid they share; vf =
// zf's lower end relative to the pair, `left` the pixels left; `sbuf` is the
// group's LDS scratch of kG * kRoundsMax floats.  Returns the pixels walked if
// the walk is over (tail cut or end of the window), -1 where that decision
// goes to the fix-up kernel, 0 if it goes on after the sh.pstep pixels.
template <int kG, bool kLds, bool kStats>
__device__ inline int near_step(const DepositArgs &A, const PairRec &P, float *sbuf, double *row, const float *ptab,
                                int zf, double vf, int dir, int left, const CutBand &cut, int lane, LaneStats &st,
                                long long p0, int item, int &adv)
{
    const int glane = lane % kG;
    const double bintov = A.vbox / A.nbins;
    const StepShape sh = unpack_shape(P.shape);
    const int nm1 = sh.nm1;
    const int pcount = min(sh.pstep, left);
    // pairs with a <= kA3Drop carry the light form of the profile (zero a^3
    // and exponent coefficients); when every pair of this near step of the
    // wavefront does, the light code runs (a wavefront-uniform branch with
    // the same results)
    const bool a3 = __ballot(P.vp.a3 != 0.0f) != 0ull;
    wave_sync();   // the previous step's reads of sbuf are done
    {
        // Sub-sample m of the step, in increasing velocity: sub-sample m mod
        // (np-1) of its pixel (singleabs.h:118-121) up to the rounding of m dv
        // against the pixel's own vlow, or (np = 1) pixel m's centre
        // (singleabs.h:113); positions in u's scale.
        const int nsub = nm1 == 0 ? pcount : __mul24(pcount, nm1) + 1;
        const double dss = P.dss;
        double sv = vf * P.ibs;
        if (nm1 == 0) sv = __builtin_fma(0.5, dss, sv);
        if (dir < 0) sv = __builtin_fma((double)__mul24(1 - pcount, max(nm1, 1)), dss, sv);   // its lowest pixel
        for (int m = glane; m < nsub; m += kG) {
            const double at = __builtin_fma((double)m, dss, sv);
            sbuf[m] = a3 ? inner32<true>(P, at, ptab) : inner32<false>(P, at, ptab);
            if (kStats) st.sums++;
        }
    }
    wave_sync();
    const bool valid = glane < pcount;
    double t = 0;
    if (valid) {
        // trapezoid over the pixel's sub-samples (singleabs.h:116-125); np = 1:
        // both ends are the one sample
        const int j = dir > 0 ? glane : pcount - 1 - glane;
        const float *sp = sbuf + (nm1 == 0 ? j : __mul24(j, nm1));
        double tot = 0.5 * ((double)sp[0] + (double)sp[nm1]);
        for (int kk = 1; kk < nm1; ++kk) tot += (double)sp[kk];
        t = P.snear * tot;
        if (kStats) st.evaluated++;
    }
    adv = pcount;
    const unsigned long long stop = __ballot(valid && t <= cut.hi), below = __ballot(valid && t < cut.lo);
    const int first = group_first<kG>(stop, lane);
    const bool sure = first < kG && group_bit<kG>(below, lane, first & (kG - 1));
    const int z = zf + dir * glane;
    if (valid && (glane < first || (glane == first && sure))) {
        row_add<kLds>(&row[wrap_near(z, A.nbins)], t);
        if (kStats) {
            st.pixels++;
            st.samples += pixel_samples(P, z * bintov - P.vel, bintov);
        }
    }
    if (first < kG) {
        if (sure) return first + 1;
        // the FP32 value of the deciding pixel is too close to tautail
        if (glane == 0) push_fixup(A, p0 + P.k, item, zf + dir * first, left - first, dir);
        return -1;
    }
    return pcount >= left ? left : 0;
}

// Record the pixels walked in one direction of pair k (for the adjoint).
__device__ inline void record_window(const DepositArgs &A, int line, long long k, int dir, int len)
{
    if (A.win) A.win[((long long)line * A.npairs + k) * 2 + (dir < 0 ? 1 : 0)] = len;
}

// Whether the next kg pixels of a fix-up walk reach pixels that use the
// far-wing expansion (|U| only grows along a walk after its first pixel).
__device__ inline bool step_needs_wing(const PairTau &P, double bintov, int z0, int dir, int c, int kg, int count)
{
    const int last = min(c + kg - 1, count - 1);
    const double U0 = ((z0 + dir * c) * bintov - P.vel + 0.5 * bintov) * P.inv_b;
    const double U1 = ((z0 + dir * last) * bintov - P.vel + 0.5 * bintov) * P.inv_b;
    return fmax(fabs(U0), fabs(U1)) >= P.ufar;
}

// Walk one direction with a kG-lane group (fix-up kernel): pixels z0,
// z0+dir, ... for at most `count` pixels, until and including the tail cut.
template <int kG, int kMode, bool kStats>
__device__ inline int walk_fix(const DepositArgs &A, PairTau &P, double *row, const float *ptab,
                               const double *gtab64, int z0, int dir, int count, int lane, LaneStats &st)
{
    const double bintov = A.vbox / A.nbins;
    const int glane = lane % kG;
    int walked = 0;
    for (int c = 0; c < count; c += kG) {
        if (kMode != kWalkFull64 && !P.wing_ready && step_needs_wing(P, bintov, z0, dir, c, kG, count)) {
            wing_setup<kG>(P, bintov, glane);
            if (glane == 0) P.wing_ready = 1;
            wave_sync();
        }
        if (walk_chunk<kG, kMode, kStats>(A, P, row, ptab, gtab64, z0, dir, count, c, lane, st, walked))
            return walked;
    }
    return walked;
}

// Lanes per fix-up entry: most deferred walks end a few pixels past the
// deciding pixel, and its 7 (or 21) samples fill half of 16 lanes, so a
// wavefront works on four entries at once.
constexpr int kFixG = 16;

// 4 waves per SIMD: measured 8% faster at c1 than the 3 the register count
// allows by default (a few dwords of spill in the pair setup).  kStats adds
// the per-lane event counts (A.stats set).
template <int kG, bool kLds, bool kStats, int kBlock>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void tau_kernel(DepositArgs A, const WorkItem *items, int item_base,
                                                       int use_queue)
{
    constexpr int kWavesPerBlock = kBlock / 64;
    constexpr int kGroupsPerWave = 64 / kG;
    extern __shared__ double smem[];
    // The table has a row for every row number (5 exponent and 5 mantissa bits),
    // a NaN's too.
    struct Lds {
        __attribute__((aligned(16))) float ptab[kPTableSize];
        PairRec recs[kWavesPerBlock * kRecs];
        float sub_sums[kBlock * kRoundsMax];
    };
    __shared__ Lds lds;
    __shared__ int s_item;
    __shared__ unsigned long long s_next;
    const float *ptab = lds.ptab;
    for (int i = threadIdx.x; i < kPTableSize / 4; i += kBlock)
        reinterpret_cast<float4 *>(lds.ptab)[i] = reinterpret_cast<const float4 *>(d_ptab)[i];
    const int lane = threadIdx.x & 63;
    const int glane = lane % kG;
    const int gid = threadIdx.x / kG;
    float *sbuf = lds.sub_sums + gid * kG * kRoundsMax;
    PairRec *recs = lds.recs + (threadIdx.x / 64) * kRecs;
    // the leader lanes of the wavefront's groups
    const unsigned long long leaders = kG == 64 ? 1ull : (kG == 32 ? 0x0000000100000001ull :
                                                         0x0001000100010001ull);
    const double bintov = A.vbox / A.nbins;
    const int half = A.nbins / 2;
    const CutBand cut = cut_band(A.tautail);
    LaneStats st;
    int it = use_queue ? 0 : blockIdx.x;
    for (;;) {
        int item;
        __syncthreads();
        if (use_queue) {
            if (threadIdx.x == 0) s_item = atomicAdd(A.queue, 1);
            __syncthreads();
            item = s_item;
        } else {
            item = it;
            it += gridDim.x;
        }
        if (item >= A.nitems) break;
        const int gitem = item_base + item;
        const WorkItem w = items[gitem];
        const LineDesc L = line_of(A, w.line);
        double *out_row = L.out + (size_t)w.los * A.nbins;
        double *row = kLds ? smem : out_row;
        if (kLds)
            for (int j = threadIdx.x; j < A.nbins; j += kBlock) row[j] = 0.0;
        if (threadIdx.x == 0) s_next = (unsigned long long)w.p0;
        __syncthreads();
        const LosInfo los = los_info(A, w.los);
        // group state: dir 0 = needs a pair, +1/-1 = walking, 2 = no pairs left;
        // rec: its record; c: pixels walked in this direction
        int dir = 0, c = 0, z0 = 0, rec = 0;
        // the wavefront's records: free, waiting by class (full: the other class,
        // see kRecs), and the class it takes pairs from
        unsigned free = ~0u, light = 0, full = 0;
        bool more = half > 0, take_full = false;   // a row of one pixel has no window (absorption.cpp:249-279)
        for (;;) {
            long long tc0 = 0;
            const unsigned long long needing = __ballot(dir == 0) & leaders;
            if (kStats) {
                tc0 = clock64();
                if (lane == 0) {
                    st.iters++;
                    st.setup_iters += needing != 0ull;
                }
            }
            if (needing) {
                const int nneed = __popcll(needing);
                if (more && __popc(take_full ? full : light) < nneed && __popc(free) >= kRefillRoom) {
                    int want = pairs_wanted((long long)w.p1 - (long long)__atomic_load_n(&s_next, __ATOMIC_RELAXED),
                                            kWavesPerBlock, kGroupsPerWave, __popc(free));
                    if (A.claim < want) want = A.claim;
                    if (want < 1) want = 1;
                    want = __builtin_amdgcn_readfirstlane(want);
                    refill_wave<kG, kStats>(A, w, gitem, L, los, &s_next, recs, lane, want, free, light, full, more, st);
                }
                if ((take_full ? full : light) == 0) take_full = !take_full;
                for (unsigned long long nm = needing; nm && (light | full); nm &= nm - 1ull) {
                    const bool f = light == 0 || (take_full && full != 0);
                    const int at = __builtin_ctz(f ? full : light);
                    if (f)
                        full &= full - 1u;
                    else
                        light &= light - 1u;
                    if (lane / kG == __builtin_ctzll(nm) / kG) {
                        rec = at;
                        dir = 1;
                        c = 0;
                        z0 = recs[at].zmax;
                    }
                }
                if (dir == 0 && !more) dir = 2;   // neither records nor pairs left
            }
            const bool walking = (dir == 1 || dir == -1);
            if (!__ballot(dir != 2)) break;
            long long tc1 = 0;
            if (kStats) tc1 = clock64();
            const PairRec &P = recs[rec];
            // a step whose first pixel lies in the far wing takes the rest of its
            // walk there, one such walk of the wavefront after the other
            const int zf = z0 + dir * c;
            const double vf = zf * bintov - P.vel;   // absorption.cpp:252
            const double uc = (vf + 0.5 * bintov) * P.ibs;
            const bool far = walking && uc * uc >= (double)P.ufsq;
            int n = 0, adv = 0;
            for (unsigned long long fm = __ballot(far) & leaders; fm; fm &= fm - 1ull) {
                const int src = __builtin_ctzll(fm);
                const PairRec &Q = recs[__builtin_amdgcn_readlane(rec, src)];
                const int fn = far_walk<kLds, kStats>(A, Q, row, __builtin_amdgcn_readlane(zf, src),
                                                      __builtin_amdgcn_readlane(dir, src),
                                                      half - __builtin_amdgcn_readlane(c, src), cut, lane, st, w.p0 + Q.k, gitem);
                if (lane / kG == src / kG) n = fn;
            }
            long long tc2 = 0;
            if (kStats) tc2 = clock64();
            if (walking && !far)
                n = near_step<kG, kLds, kStats>(A, P, sbuf, row, ptab, zf, vf, dir, half - c, cut, lane, st, w.p0, gitem, adv);
            if (kStats && lane == 0) {
                const long long tc3 = clock64();
                st.cyc_setup += tc1 - tc0;
                st.cyc_wing += tc2 - tc1;
                st.cyc_walk += tc3 - tc2;
            }
            bool ended = false;
            if (walking) {
                if (n > 0 && glane == 0) record_window(A, w.line, w.p0 + P.k, dir, c + n);
                if (n == 0) {
                    c += adv;
                } else if (dir == 1) {
                    dir = -1;
                    z0 -= 1;
                    c = 0;
                } else {
                    dir = 0;
                    ended = true;
                }
            }
            for (unsigned long long em = __ballot(ended) & leaders; em; em &= em - 1ull)
                free |= 1u << __builtin_amdgcn_readlane(rec, __builtin_ctzll(em));
        }
        if (kLds) {
            __syncthreads();
            if (w.direct) {
                for (int j = threadIdx.x; j < A.nbins; j += kBlock) out_row[j] = row[j];
            } else {
                for (int j = threadIdx.x; j < A.nbins; j += kBlock) {
                    const double v = row[j];
                    if (v != 0.0) unsafeAtomicAdd(&out_row[j], v);
                }
            }
        }
    }
    if (kStats && A.stats) {
        atomicAdd((unsigned long long *)&A.stats[0], (unsigned long long)st.pairs);
        atomicAdd((unsigned long long *)&A.stats[1], (unsigned long long)st.pixels);
        atomicAdd((unsigned long long *)&A.stats[3], (unsigned long long)st.pairs64);
        atomicAdd((unsigned long long *)&A.stats[4], (unsigned long long)st.samples);
        atomicAdd((unsigned long long *)&A.stats[5], (unsigned long long)st.evaluated);
        atomicAdd((unsigned long long *)&A.stats[6], (unsigned long long)st.sums);
        atomicAdd((unsigned long long *)&A.stats[7], (unsigned long long)st.far);
        if (lane == 0) {
            atomicAdd((unsigned long long *)&A.stats[8], (unsigned long long)st.cyc_setup);
            atomicAdd((unsigned long long *)&A.stats[9], (unsigned long long)st.cyc_wing);
            atomicAdd((unsigned long long *)&A.stats[10], (unsigned long long)st.cyc_walk);
            atomicAdd((unsigned long long *)&A.stats[11], (unsigned long long)st.iters);
            atomicAdd((unsigned long long *)&A.stats[12], (unsigned long long)st.setup_iters);
        }
    }
}

// Deferred walks, after the deposit kernel has written its rows: one lane
// group per fix-up entry, deposits straight into the output with FP64 atomics.
//
// Bound: the latency of an entry's FP64 samples where few walks are deferred,
// FP64 VALU where millions are.  With voigt64_small in place of w64 and a
// deciding pixel's samples over the group instead of in turn on one lane: 109M
// pair-lines of 2048 pixels 3192 -> 224 us, 1.4M of 1501 1089 -> 28 us, 32768
// particles and 64 sightlines 174 -> 18 us.
template <bool kStats>
__global__ __launch_bounds__(kThreads) void tau_fixup_kernel(DepositArgs A, const WorkItem *items)
{
    constexpr int kGroups = kThreads / kFixG;
    struct Lds {
        __attribute__((aligned(16))) float ptab[kPTableSize];
        PairTau pslot[kGroups];
    };
    __shared__ Lds lds;
    __shared__ double gtab64[kG64Size];
    const float *ptab = lds.ptab;
    const int n = (int)min(A.fix_count[0], (unsigned long long)A.fix_cap);
    if (blockIdx.x * kGroups >= n) return;
    for (int i = threadIdx.x; i < kPTableSize / 4; i += kThreads)
        reinterpret_cast<float4 *>(lds.ptab)[i] = reinterpret_cast<const float4 *>(d_ptab)[i];
    for (int i = threadIdx.x; i < kG64Size; i += kThreads) gtab64[i] = d_gtab64[i];
    __syncthreads();
    const int lane = threadIdx.x & 63, gid = threadIdx.x / kFixG, glane = lane % kFixG;
    PairTau &P = lds.pslot[gid];
    LaneStats st;
    const int half = A.nbins / 2;
    for (int e = blockIdx.x * kGroups + gid; e < n; e += gridDim.x * kGroups) {
        const Fixup f = A.fix[e];
        const WorkItem w = items[f.item];
        const LineDesc L = line_of(A, w.line);
        double *out_row = L.out + (size_t)w.los * A.nbins;
        const LosInfo los = los_info(A, w.los);
        if (!setup_pair<kFixG>(A, w.line, L, los, f.k, P, glane)) continue;
        if (f.dir == kFixPair64) {
            const int lf = walk_fix<kFixG, kWalkFull64, kStats>(A, P, out_row, ptab, gtab64, P.zmax, 1, half, lane, st);
            const int lb = walk_fix<kFixG, kWalkFull64, kStats>(A, P, out_row, ptab, gtab64, P.zmax - 1, -1, half, lane, st);
            if (glane == 0) {
                record_window(A, w.line, f.k, 1, lf);
                record_window(A, w.line, f.k, -1, lb);
            }
        } else if (f.dir == kFixPair) {
            const int lf = walk_fix<kFixG, kWalkGuarded, kStats>(A, P, out_row, ptab, gtab64, P.zmax, 1, half, lane, st);
            const int lb = walk_fix<kFixG, kWalkGuarded, kStats>(A, P, out_row, ptab, gtab64, P.zmax - 1, -1, half, lane, st);
            if (glane == 0) {
                record_window(A, w.line, f.k, 1, lf);
                record_window(A, w.line, f.k, -1, lb);
            }
        } else {
            // the walk's z0 counts from the box that holds its first pixel
            if (glane == 0) P.vel -= box_shift(P.zmax, A.nbins) * A.vbox;
            wave_sync();
            const int l = walk_fix<kFixG, kWalkGuarded, kStats>(A, P, out_row, ptab, gtab64, f.z0, f.dir, f.count, lane, st);
            if (glane == 0) record_window(A, w.line, f.k, f.dir, (half - f.count) + l);
        }
    }
    if (kStats && A.stats) {
        atomicAdd((unsigned long long *)&A.stats[1], (unsigned long long)st.pixels);
        atomicAdd((unsigned long long *)&A.stats[2], (unsigned long long)st.px64);
        atomicAdd((unsigned long long *)&A.stats[4], (unsigned long long)st.samples);
        atomicAdd((unsigned long long *)&A.stats[5], (unsigned long long)st.evaluated);
        atomicAdd((unsigned long long *)&A.stats[6], (unsigned long long)st.sums);
        atomicAdd((unsigned long long *)&A.stats[7], (unsigned long long)st.far);
    }
}

// ---------------------------------------------------------------------------
// Adjoint of the optical depth.
//
// For a pair, taulast(z) = scale * S(z), S = sum_samples t_j W_i H(a, u_ij),
// u_ij = (vv_i - vouter_j)/b, vouter_j = z*bintov - vel + e_j, scale =
// amp dens dvk/velfac with amp ~ 1/b, b = bfac sqrt(T), a = voigt_fac/b.
// With g(z) = dL/dtau at the pixel:
//   dL/d dens = sum_z g scale/dens S
//   dL/d vel  = sum_z g scale/b SU,          SU = sum t W dH/du
//   dL/d T    = -sum_z g scale/(2T) ST,      ST = sum t W (H + u dH/du + a dH/da)
// over exactly the pixels the forward deposited (recorded windows); the
// discrete choices (window ends, pixel index, sub-sample count) are held
// fixed.  Far-wing pixels use the same moment expansion as the forward, with
// a second coefficient set for ST and the derivative of the first for SU.

// The same three sums with the FP64 Faddeeva function and FP64 kernel weights,
// for the pairs the forward evaluates in FP64 (damping parameter above
// kA32Max, or a sub-sample count on a switch point).  With L = Im w:
//   dH/du = -2(uH - aL),  u dH/du + a dH/da = -2(u^2 - a^2)H + 4auL - 2a/sqrt(pi).
__device__ __noinline__ void adj_inner64(double aa, double b, double dvk, double vhigh, double vdr2, double vsmooth,
                                         double vouter, int kernel, double &S, double &SU, double &SF)
{
    for (int i = 1; i < kNGrid; ++i) {
        const double vv = i * dvk - vhigh;
        const double W = kernel_weight(kernel, sqrt(vdr2 + vv * vv) / vsmooth);
        const double u = (vv - vouter) / b;
        double H, L;
        w64(u, aa, H, L);
        S += W * H;
        SU += W * (-2.0 * (u * H - aa * L));
        SF += W * (-2.0 * (u * u - aa * aa) * H + 4.0 * aa * u * L - aa * kTwoOverSqrtPi);
    }
}

// One pixel of an FP64 pair: the sums averaged over the pixel's own
// sub-sample grid, as tau_kern_outer builds it (singleabs.h:104-126) and as
// the forward's FP64 walk evaluates it.
__device__ inline void adj_pixel64(const PairTau &P, double vlow, double bintov, int kernel, double &S, double &SU,
                                   double &SF)
{
    const double vhighp = vlow + bintov;
    const double width = vhighp - vlow;
    S = SU = SF = 0.0;
    if (width < P.b / 2.) {
        adj_inner64(P.aa, P.b, P.dvk, P.vhigh, P.vdr2, P.vsmooth, (vhighp + vlow) / 2., kernel, S, SU, SF);
        return;
    }
    const int np = 2 * ceil(width / (P.b / 2.) / 2) + 1.;
    const double dv = width / (np - 1);
    double s0 = 0, u0 = 0, f0 = 0;
    adj_inner64(P.aa, P.b, P.dvk, P.vhigh, P.vdr2, P.vsmooth, vlow, kernel, s0, u0, f0);
    adj_inner64(P.aa, P.b, P.dvk, P.vhigh, P.vdr2, P.vsmooth, vhighp, kernel, s0, u0, f0);
    S = 0.5 * s0;
    SU = 0.5 * u0;
    SF = 0.5 * f0;
    for (int i = 1; i < np - 1; ++i)
        adj_inner64(P.aa, P.b, P.dvk, P.vhigh, P.vdr2, P.vsmooth, i * dv + vlow, kernel, S, SU, SF);
    const double inv = 1.0 / (np - 1);
    S *= inv;
    SU *= inv;
    SF *= inv;
}

// A pair of the adjoint: its window's pixels zlo .. zlo + n - 1, of which the first
// nfl and the last n - nfl - nn lie in the far wing (|U| >= ufar).
struct AdjRec {
    double s0;        // the lower end of pixel zlo over b, in u's scale
    double ibs, dss, qs;   // as PairRec
    float W[4];
    double scale_nd;  // amp * dvk / velfac (scale without the density)
    double inv_nm1;   // 1 / max(np - 1, 1)
    float Cw[kWingTerms], CwT[kWingTerms];
    VoigtP vp;
    float a2, ufsq, dens, temp;
    int zlo, n, nfl, nn, nm1, part;
};
static_assert(sizeof(AdjRec) == 208, "AdjRec layout: W on a 16-byte boundary");

constexpr int kAdjThreads = 1024;
constexpr int kAdjWaves = kAdjThreads / 64;

// Claim `want` pairs for the wavefront and set up those with a window, as
// refill_wave does for the forward.  FP64 pairs go to the list of
// tau_adjoint64_kernel.  kWide: the wide pairs alone; without it they are left out
// and the second bit of fix_count[1] tells that there are some.
template <bool kWide>
__device__ inline void refill_adjoint(const DepositArgs &A, const WorkItem &w, int item, const LineDesc &L,
                                      const LosInfo &los, unsigned long long *next, AdjRec *recs, int lane, int want,
                                      unsigned &free, unsigned &light, unsigned &full, bool &more)
{
    unsigned long long base = 0;
    if (lane == 0) base = atomicAdd(next, (unsigned long long)want);
    base = (unsigned long long)__shfl((long long)base, 0, 64);
    const long long kk = (long long)base + lane;
    const double bintov = A.vbox / A.nbins;
    bool enq = false, left_out = false;
    int lf = 0, lb = 0;
    PairConsts C;
    if (lane < want && kk < w.p1) {
        const long long wi = ((long long)w.line * A.npairs + kk) * 2;
        lf = A.win[wi];
        lb = A.win[wi + 1];
        if (lf + lb > 0 && pair_consts(A, w.line, L, los, kk, FSAMD_WING_TMAX, C)) {
            enq = !C.fp64 && (bool)C.wide == kWide;
            if (!kWide && C.fp64) push_fixup(A, kk, item, 0, 0, kFixPair64);
            left_out = !kWide && !C.fp64 && C.wide;
        }
    }
    if (!kWide && __ballot(left_out) && lane == 0) atomicOr(&A.fix_count[1], 2ull);
    const unsigned long long m = __ballot(enq);
    bool used;
    const int slot = free_record(free, m, lane, used);
    wave_sync();   // the records' former pairs have been read
    if (enq) {
        AdjRec &r = recs[slot];
        VoigtP vp = make_voigt_p(C.aa, C.aa <= (double)kA3Drop);
        vp.a3 = (float)(C.aa * C.aa * (-1.0 / 6.0));   // in the short form too (GradSums)
        r.vp = vp;
        const double us = voigt_uscale(vp, C.aa), ibs = us * C.inv_b;
        const double inv_m = C.np > 1 ? 1.0 / (C.np - 1) : 1.0;
        const int zlo = C.zmax - lb, n = lf + lb;
        const double s0 = (zlo * bintov - C.vel) * ibs, bxs = bintov * ibs;   // absorption.cpp:252
        r.s0 = s0;
        r.ibs = ibs;
        r.dss = bxs * inv_m;
        r.qs = 0.25 * C.vhigh * ibs;
        r.inv_nm1 = inv_m;
        r.scale_nd = C.scale_nd;
        r.a2 = (float)(C.aa * C.aa);
        const double inv_s2 = 1.0 / (C.vsmooth * C.vsmooth);
        float W[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const double vv = (i + 4) * C.dvk - C.vhigh;
            W[i] = kernel_weight_q2(A.kernel, (C.vdr2 + vv * vv) * inv_s2);
        }
        *(float4 *)r.W = make_float4(W[0], W[1], W[2], W[3]);
        const float ufar = (float)C.ufar;
        r.ufsq = (float)((us * ufar) * (us * ufar));
        const double iu = 1.0 / (double)ufar;
        wing_coeffs<double, true>(C.vhigh * C.inv_b * iu, 0.5 * bintov * C.inv_b * iu, C.np - 1, W[0], W[1], W[2], W[3],
                                  C.aa, (double)ufar, r.Cw, r.CwT);
        // far-wing pixels: those whose centre s0 + (j + 1/2) bxs lies at or beyond +-ufar
        const double c0 = s0 + 0.5 * bxs, inv_x = 1.0 / bxs, uf = us * ufar;
        const double jl = floor((-uf - c0) * inv_x) + 1.0, jr = ceil((uf - c0) * inv_x);
        const int nfl = (int)fmin(fmax(jl, 0.0), (double)n), end = (int)fmin(fmax(jr, (double)nfl), (double)n);
        r.nfl = nfl;
        r.nn = end - nfl;
        r.zlo = zlo;
        r.n = n;
        r.nm1 = C.np - 1;
        r.part = A.pair_part[kk];
        r.dens = A.rec[r.part].dens[w.line];
        r.temp = C.temp;
    }
    wave_sync();
    const unsigned mine = (unsigned)__ballot(used);
    const unsigned fulls = (unsigned)__ballot(used && recs[lane & 31].vp.l2 != 0.0f);
    free &= ~mine;
    light |= mine & ~fulls;
    full |= fulls;
    more = (long long)base + want < w.p1;
}

// One grid point of a pair: the sums (GradSums) of the kernel samples around s.
template <bool kFull>
__device__ inline void adj_point(const AdjRec &P, double s, const float *tab, float &S, float &SU, float &ST,
                                 float &SP)
{
    const VoigtP vp = P.vp;
    const double qs = P.qs;
    const float a2 = P.a2;
    const float4 w4 = *(const float4 *)P.W;
    const float W[4] = {w4.x, w4.y, w4.z, w4.w};
    GradSums g;
#pragma unroll
    for (int j = -3; j <= 3; ++j) g.add<kFull>(vp, a2, W[j < 0 ? -j : j], sample_us(qs, j, s), tab);
    g.finish(vp, a2, S, SU, ST, SP);
}

// The same for a wide pair.
__device__ inline void adj_point_wide(const AdjRec &P, double s, const float *tab, float &S, float &SU, float &ST,
                                      float &SP)
{
    const VoigtP vp = P.vp;
    const double qs = P.qs;
    const float a2 = P.a2;
    GradSums g;
#pragma unroll 1
    for (int j = -3; j <= 3; ++j) g.add<true, true>(vp, a2, P.W[j < 0 ? -j : j], sample_us(qs, j, s), tab);
    g.finish(vp, a2, S, SU, ST, SP);
}

// Bound: VALU issue (32 instructions a sample in the short form).  Structured as
// tau_kernel: pairs set up one per lane into records, walked in place by lane
// groups, pairs of the short and of the full form in runs, far-wing pixels by the
// whole wavefront.
// Here the windows are known: a group walks the grid points of its pair's near
// pixels, each once, weighted by the trapezoid weights and dL/dtau of the
// pixels it belongs to.  One block of 16 wavefronts a CU shares the table of G
// and K (32 KB) and the row.  kRow: the row of dL/dtau in LDS; a row that does
// not fit beside the records (above about 3000 pixels) is read where it is.  kWide:
// the pass over the wide pairs, where a first pass met some.
// 2.1M particles, 1024 sightlines of 1024 pixels, forward and adjoint: 37.9 -> 15.9
// ms.
template <int kG, bool kRow, bool kWide>
__global__ __launch_bounds__(kAdjThreads) __attribute__((amdgpu_waves_per_eu(4))) void tau_adjoint_kernel(
    DepositArgs A, const WorkItem *items)
{
    constexpr int kGroupsPerWave = 64 / kG;
    extern __shared__ double grow_lds[];   // dL/dtau of the item's sightline and line
    struct Lds {
        __attribute__((aligned(16))) float tab[2 * kPTableSize];
        AdjRec recs[kAdjWaves * kRecs];
    };
    __shared__ Lds lds;
    __shared__ int s_item;
    __shared__ unsigned long long s_next;
    for (int i = threadIdx.x; i < kPTableSize / 4; i += kAdjThreads) {
        reinterpret_cast<float4 *>(lds.tab)[2 * i] = reinterpret_cast<const float4 *>(d_ptab)[i];
        reinterpret_cast<float4 *>(lds.tab)[2 * i + 1] = reinterpret_cast<const float4 *>(d_dtab)[i];
    }
    const float *tab = lds.tab;
    const int lane = threadIdx.x & 63;
    const int glane = lane % kG;
    AdjRec *recs = lds.recs + (threadIdx.x / 64) * kRecs;
    const unsigned long long leaders = kG == 64 ? 1ull : (kG == 32 ? 0x0000000100000001ull : 0x0001000100010001ull);
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) s_item = atomicAdd(A.queue, 1);
        __syncthreads();
        const int item = s_item;
        if (item >= A.nitems) break;
        const WorkItem w = items[item];
        const LineDesc L = line_of(A, w.line);
        const double *grad_row = L.out + (size_t)w.los * A.nbins;
        if (kRow)
            for (int j = threadIdx.x; j < A.nbins; j += kAdjThreads) grow_lds[j] = grad_row[j];
        const double *grow = kRow ? grow_lds : grad_row;
        if (threadIdx.x == 0) s_next = (unsigned long long)w.p0;
        __syncthreads();
        const LosInfo los = los_info(A, w.los);
        // group state: 0 needs a pair, 1 walks rec's grid points from c on, 2 no pairs left
        int state = 0, c = 0, rec = 0;
        double aS = 0, aU = 0, aT = 0, aP = 0;   // aU, aP: without 1 / scale and 1 / scale^2 (GradSums)
        unsigned free = ~0u, light = 0, full = 0;
        bool more = true, take_full = false;
        for (;;) {
            const unsigned long long needing = __ballot(state == 0) & leaders;
            if (needing) {
                if (more && __popc(take_full ? full : light) < __popcll(needing) && __popc(free) >= kRefillRoom) {
                    int want = pairs_wanted((long long)w.p1 - (long long)__atomic_load_n(&s_next, __ATOMIC_RELAXED),
                                            kAdjWaves, kGroupsPerWave, __popc(free));
                    want = __builtin_amdgcn_readfirstlane(want < 1 ? 1 : want);
                    refill_adjoint<kWide>(A, w, item, L, los, &s_next, recs, lane, want, free, light, full, more);
                }
                if ((take_full ? full : light) == 0) take_full = !take_full;
                for (unsigned long long nm = needing; nm && (light | full); nm &= nm - 1ull) {
                    const bool f = light == 0 || (take_full && full != 0);
                    const int at = __builtin_ctz(f ? full : light);
                    if (f)
                        full &= full - 1u;
                    else
                        light &= light - 1u;
                    if (lane / kG == __builtin_ctzll(nm) / kG) {
                        rec = at;
                        state = 1;
                        c = 0;
                        aS = aU = aT = aP = 0;
                    }
                }
                if (state == 0 && !more) state = 2;
            }
            if (!__ballot(state != 2)) break;
            const AdjRec &P = recs[rec];
            const int nm1 = P.nm1;
            const int npts = state != 1 || P.nn == 0 ? 0 : nm1 == 0 ? P.nn : P.nn * nm1 + 1;
            const bool any_full = __ballot(state == 1 && P.vp.l2 != 0.0f) != 0ull;
            const int m = c + glane;
            if (m < npts) {
                // grid point m: sub-sample kk of near pixel jj (singleabs.h:110-125)
                const int jj = nm1 == 0 ? m : (int)((m + 0.5) * P.inv_nm1);
                const int kk = nm1 == 0 ? 1 : m - jj * nm1;
                const int z = P.zlo + P.nfl + jj;
                double wgt = jj < P.nn ? grow[wrap_pixel(z, A.nbins)] : 0.0;
                if (kk == 0) wgt = 0.5 * (wgt + (jj > 0 ? grow[wrap_pixel(z - 1, A.nbins)] : 0.0));
                const double dss = P.dss;
                const double s = __builtin_fma((double)P.nfl * (nm1 == 0 ? 1 : nm1) + m + (nm1 == 0 ? 0.5 : 0.0), dss, P.s0);
                float S, SU, ST, SP;
                if (kWide)
                    adj_point_wide(P, s, tab, S, SU, ST, SP);
                else if (any_full)
                    adj_point<true>(P, s, tab, S, SU, ST, SP);
                else
                    adj_point<false>(P, s, tab, S, SU, ST, SP);
                aS = __builtin_fma(wgt, (double)S, aS);
                aU = __builtin_fma(wgt, (double)SU, aU);
                aT = __builtin_fma(wgt, (double)ST, aT);
                aP = __builtin_fma(wgt, (double)SP, aP);
            }
            c += kG;
            const bool ended = state == 1 && c >= npts;
            const unsigned long long em = __ballot(ended) & leaders;
            if (!em) continue;
            if (ended) {
                // the trapezoid's weights, and the scale (voigt_uscale) from l1
                const double k2 = (double)P.vp.l1 * (-1.0 / kLog2E) / (1.0 + 2.0 * (double)P.a2);   // 1 / scale^2
                const double k1 = kUScale * (0.5 * k2 + 0.5 / (kUScale * kUScale));   // its root, next to 1 / kUScale
                aS *= P.inv_nm1;
                aU *= P.inv_nm1 * k1;
                aT = P.inv_nm1 * __builtin_fma(k2, aP, aT);
            }
            for (unsigned long long fm = em; fm; fm &= fm - 1ull) {
                const int src = __builtin_ctzll(fm);
                const int at = __builtin_amdgcn_readlane(rec, src);
                const AdjRec &Q = recs[at];
                free |= 1u << at;   // its reads below come before the next set-up
                const int nfar = Q.n - Q.nn;
                if (nfar == 0) continue;
                const double bxs = Q.dss * (Q.nm1 == 0 ? 1 : Q.nm1);
                double fS = 0, fU = 0, fT = 0;
                for (int i = lane; i < nfar; i += 64) {
                    const int j = i < Q.nfl ? i : i + Q.nn;
                    const double Us = __builtin_fma((double)j + 0.5, bxs, Q.s0);
                    const float Y = Q.ufsq * __builtin_amdgcn_rcpf((float)(Us * Us));
                    float s = Q.Cw[kWingTerms - 1], d = kWingTerms * Q.Cw[kWingTerms - 1], f = Q.CwT[kWingTerms - 1];
#pragma unroll
                    for (int t = kWingTerms - 2; t >= 0; --t) {
                        s = __builtin_fmaf(s, Y, Q.Cw[t]);
                        d = __builtin_fmaf(d, Y, (t + 1.0f) * Q.Cw[t]);
                        f = __builtin_fmaf(f, Y, Q.CwT[t]);
                    }
                    const double g = grow[wrap_pixel(Q.zlo + j, A.nbins)] * (double)Y;
                    fS = __builtin_fma(g, (double)s, fS);
                    fU = __builtin_fma(g * (2.0 * kUScale) / Us, (double)d, fU);
                    fT = __builtin_fma(g, (double)f, fT);
                }
                // each lane of the pair's group takes the lanes of its number
#pragma unroll
                for (int o = 32; o >= kG; o >>= 1) {
                    fS += __shfl_xor(fS, o, 64);
                    fU += __shfl_xor(fU, o, 64);
                    fT += __shfl_xor(fT, o, 64);
                }
                if (lane / kG == src / kG) {
                    aS += fS;
                    aU += fU;
                    aT += fT;
                }
            }
            const double tS = group_sum<kG>(aS), tU = group_sum<kG>(aU), tT = group_sum<kG>(aT);
            if (ended) {
                if (glane == 0) {
                    const double scale = P.scale_nd * (double)P.dens;
                    unsafeAtomicAdd(&L.grad_dens[P.part], P.scale_nd * tS);
                    unsafeAtomicAdd(&A.grad_vel[3 * (size_t)P.part + los.ax - 1], scale * P.ibs * (1 / kUScale) * tU);
                    unsafeAtomicAdd(&A.grad_temp[P.part], -scale / (2.0 * (double)P.temp) * tT);
                }
                state = 0;
            }
        }
    }
}

// The adjoint of the pairs the forward evaluated in FP64 (listed by
// tau_adjoint_kernel in the fix-up list): one kFixG-lane group per pair, the
// window's pixels with the FP64 Faddeeva function and FP64 kernel weights,
// dL/dtau read from HBM.
__global__ __launch_bounds__(kThreads) void tau_adjoint64_kernel(DepositArgs A, const WorkItem *items)
{
    constexpr int kGroups = kThreads / kFixG;
    __shared__ PairTau pslot[kGroups];
    const int lane = threadIdx.x & 63, gid = threadIdx.x / kFixG, glane = lane % kFixG;
    PairTau &P = pslot[gid];
    const double bintov = A.vbox / A.nbins;
    const int n = (int)min(A.fix_count[0], (unsigned long long)A.fix_cap);
    for (int e = blockIdx.x * kGroups + gid; e < n; e += gridDim.x * kGroups) {
        const Fixup f = A.fix[e];
        const WorkItem w = items[f.item];
        const LineDesc L = line_of(A, w.line);
        const double *grad_row = L.out + (size_t)w.los * A.nbins;
        const LosInfo los = los_info(A, w.los);
        if (!setup_pair<kFixG>(A, w.line, L, los, f.k, P, glane)) continue;
        const long long wi = ((long long)w.line * A.npairs + f.k) * 2;
        const int lf = A.win[wi], lb = A.win[wi + 1];
        const int nw = lf + lb;
        const int zlo = P.zmax - lb;   // the window: pixels zlo .. zlo + nw - 1
        double aS = 0, aU = 0, aF = 0;
        for (int j = glane; j < nw; j += kFixG) {
            const int z = zlo + j;
            double S, SU, SF;
            adj_pixel64(P, z * bintov - P.vel, bintov, A.kernel, S, SU, SF);   // absorption.cpp:252
            const double g = grad_row[wrap_pixel(z, A.nbins)];
            aS += g * S;
            aU += g * SU;
            aF += g * SF;
        }
        aS = group_sum<kFixG>(aS);
        aU = group_sum<kFixG>(aU);
        aF = group_sum<kFixG>(aF);
        if (glane == 0) {
            const int p = P.part;
            unsafeAtomicAdd(&L.grad_dens[p], P.scale_nd * aS);
            unsafeAtomicAdd(&A.grad_vel[3 * (size_t)p + los.ax - 1], P.scale * P.inv_b * aU);
            unsafeAtomicAdd(&A.grad_temp[p], -P.scale / (2.0 * P.temp) * (aS + aF));
        }
    }
}

int launch_tau_adjoint64(const DepositArgs &A, const WorkItem *items, int nblocks, hipStream_t s)
{
    tau_adjoint64_kernel<<<nblocks, kThreads, 0, s>>>(A, items);
    FSAMD_HIP(hipGetLastError());
    return FSAMD_OK;
}

// A kernel's static LDS, or a conservative 64 KiB if the runtime cannot say.
static size_t static_lds(const void *fn)
{
    hipFuncAttributes a;
    if (hipFuncGetAttributes(&a, fn) != hipSuccess) {
        (void)hipGetLastError();
        return 65536;
    }
    return a.sharedSizeBytes;
}

// Whether the adjoint keeps its row in LDS beside its records and table, whose
// size is the same at every group width.
static bool adjoint_row_in_lds(int nbins)
{
    return deposit_lds_bytes(nbins) + static_lds((const void *)tau_adjoint_kernel<16, true, false>) <= 160 * 1024;
}

template <int kG, bool kRow, bool kWide>
static int launch_adjoint(const DepositArgs &A, const WorkItem *items, int nblocks, hipStream_t s)
{
    const size_t shm = kRow ? deposit_lds_bytes(A.nbins) : 0;
    if (int rc = raise_lds_limit((const void *)tau_adjoint_kernel<kG, kRow, kWide>, shm)) return rc;
    tau_adjoint_kernel<kG, kRow, kWide><<<nblocks, kAdjThreads, shm, s>>>(A, items);
    FSAMD_HIP(hipGetLastError());
    return FSAMD_OK;
}

int launch_tau_adjoint(int gsize, bool wide, const DepositArgs &A, const WorkItem *items, int nblocks, hipStream_t s)
{
    if (wide) return launch_adjoint<16, false, true>(A, items, nblocks, s);
    const bool row = adjoint_row_in_lds(A.nbins);
    if (gsize == 16)
        return row ? launch_adjoint<16, true, false>(A, items, nblocks, s) : launch_adjoint<16, false, false>(A, items, nblocks, s);
    if (gsize == 32)
        return row ? launch_adjoint<32, true, false>(A, items, nblocks, s) : launch_adjoint<32, false, false>(A, items, nblocks, s);
    return row ? launch_adjoint<64, true, false>(A, items, nblocks, s) : launch_adjoint<64, false, false>(A, items, nblocks, s);
}

// ---------------------------------------------------------------------------
// Column density

// Sums over kernel samples of the truncated powers the splines consist of
// (singleabs.h:17-42): the cubic is 2 ((1-q)+^3 - 4 (1/2-q)+^3) over its norm,
// the quintic (3-3q)+^5 - 6 (2-3q)+^5 + 15 (1-3q)+^5.  No branch on q.
template <int kKernel>
struct ShapeSum {
    double s1 = 0, s2 = 0, s3 = 0;
    __device__ inline void add(double q2)
    {
        const double q = sqrt_nr(q2);
        if (kKernel == kCubicSpline) {
            const double t = fmax(1.0 - q, 0.0), h = fmax(0.5 - q, 0.0);
            s1 = __builtin_fma(t * t, t, s1);
            s2 = __builtin_fma(h * h, h, s2);
        } else {
            const double t3 = fmax(__builtin_fma(-3.0, q, 3.0), 0.0), t2 = fmax(__builtin_fma(-3.0, q, 2.0), 0.0),
                         t1 = fmax(__builtin_fma(-3.0, q, 1.0), 0.0);
            const double p3 = t3 * t3, p2 = t2 * t2, p1 = t1 * t1;
            s1 = __builtin_fma(p3 * p3, t3, s1);
            s2 = __builtin_fma(p2 * p2, t2, s2);
            s3 = __builtin_fma(p1 * p1, t1, s3);
        }
    }
    __device__ inline void halve()
    {
        s1 *= 0.5;
        s2 *= 0.5;
        if (kKernel != kCubicSpline) s3 *= 0.5;
    }
    __device__ inline double kernel_sum() const
    {
        if (kKernel == kCubicSpline) return 32. / 4 / kPi * 2.0 * (s1 - 4.0 * s2);
        return 9. / 40 / kPi * (s1 - 6.0 * s2 + 15.0 * s3);
    }
};

// absorption.cpp:53-74 (cubic), 76-97 (quintic): the trapezoid of 8 intervals
template <int kKernel>
__device__ inline double kern_trapezoid(double zlow, double zhigh, double inv_s2, double dr2)
{
    const double dz = (zhigh - zlow) / kNGrid;
    const double d2 = dr2 * inv_s2 + 1e-290;   // keeps q^2 above zero for sqrt_nr
    ShapeSum<kKernel> sum;
    sum.add(__builtin_fma(zlow * zlow, inv_s2, d2));
    sum.add(__builtin_fma(zhigh * zhigh, inv_s2, d2));
    sum.halve();
#pragma unroll
    for (int i = 1; i < kNGrid; ++i) {
        const double zz = __builtin_fma((double)i, dz, zlow);
        sum.add(__builtin_fma(zz * zz, inv_s2, d2));
    }
    return dz * sum.kernel_sum();
}

// kern_frac of one pixel [zlow, zhigh]: absorption.cpp:129-134 (mesh), 53-97
// and 109-115 (tophat, also the reference's default for any other id,
// absorption.cpp:136-148)
__device__ inline double kern_frac(int kernel, double zlow, double zhigh, double inv_s2, double dr2, double zrange)
{
    zlow = fmax(zlow, -zrange);
    zhigh = fmin(zhigh, zrange);
    if (kernel == kCubicSpline) return zlow > zhigh ? 0.0 : kern_trapezoid<kCubicSpline>(zlow, zhigh, inv_s2, dr2);
    if (kernel == kSphQuintic) return zlow > zhigh ? 0.0 : kern_trapezoid<kSphQuintic>(zlow, zhigh, inv_s2, dr2);
    const double len = fmax(0., zhigh - zlow);
    return kernel == kVoronoiMesh ? len : 3. / 4. / kPi * len;
}

// One pair as its pixels need it.
struct ColPair {
    double pos1, zrange, dr2, inv_s2;
    long long start;          // first of the pair's slots in the batch
    int zlow, pad;
};

// Dynamic LDS of a column-density block per field: its row and its density
// of each pair the wavefronts hold.
static size_t colden_lds_bytes(int nbins) { return deposit_lds_bytes(nbins) + sizeof(float) * kColThreads; }

// Work item: one sightline (or a range of its pairs) and up to A.fields
// fields, part w.line of them; their rows lie side by side in LDS.
//
// Bound: FP64 VALU (9 kernel values a pixel and pair).  A wavefront takes 64
// pairs, one per lane, and then runs over all their (pair, pixel) slots 64 at
// a time, so that supports of a few pixels and of hundreds fill the lanes
// alike, and a pixel's kernel fraction serves every field.  12.5M pairs of
// ~45 pixels, 5 fields of 1024 pixels: 168 ms with one lane a pair and one
// field an item, 5.6 ms so (81% of the VALU issue slots busy, 98% of lanes;
// the samples rolled instead of unrolled: 6.1 ms).
template <bool kLds>
__global__ __launch_bounds__(kColThreads) void colden_kernel(DepositArgs A, const WorkItem *items, int item_base,
                                                             int use_queue)
{
    extern __shared__ double smem[];
    __shared__ int s_item;
    __shared__ unsigned long long s_next;
    __shared__ ColPair pairs[kColThreads];
    __shared__ int marks[kColThreads];
    const int lane = threadIdx.x & 63, wbase = threadIdx.x & ~63;
    ColPair *mine = pairs + wbase;
    int *mark = marks + wbase;
    // [field][pair of the block], after the rows
    float *dens = (float *)(smem + (kLds ? (size_t)A.fields * A.nbins : 0)) + wbase;
    const unsigned long long below = (1ull << lane) - 1ull;
    const double boxtokpc = A.vbox / A.nbins / A.velfac;   // absorption.cpp:188
    int it = use_queue ? 0 : blockIdx.x;
    for (;;) {
        int item;
        __syncthreads();
        if (use_queue) {
            if (threadIdx.x == 0) s_item = atomicAdd(A.queue, 1);
            __syncthreads();
            item = s_item;
        } else {
            item = it;
            it += gridDim.x;
        }
        if (item >= A.nitems) break;
        const WorkItem w = items[item_base + item];
        const int f0 = w.line * A.fields, nf = min(A.fields, A.nlines - f0);
        if (kLds)
            for (int j = threadIdx.x; j < nf * A.nbins; j += kColThreads) smem[j] = 0.0;
        if (threadIdx.x == 0) s_next = (unsigned long long)w.p0;
        __syncthreads();
        const LosInfo los = los_info(A, w.los);
        for (;;) {
            unsigned long long base = 0;
            if (lane == 0) base = atomicAdd(&s_next, 64ull);
            base = (unsigned long long)__shfl((long long)base, 0, 64);
            if ((long long)base >= w.p1) break;
            const long long k = (long long)base + lane;
            // the pair of this lane
            bool have = k < w.p1;
            ColPair P;
            int p = 0;
            long long npix = 0;
            if (have) {
                p = A.pair_part[k];
                const float *pp = &A.pos[3 * (size_t)p];
                float smooth;
                P.pos1 = pp[los.ax - 1];
                if (A.seg) {
                    // Voronoi mesh: the segment ends replace dr2 and h
                    // (absorption.cpp:170-187): centre and half length
                    const float2 sg = A.seg[k];
                    P.dr2 = (double)sg.x;
                    smooth = sg.y;
                    have = !(P.dr2 > 2 * A.vbox / A.velfac || (double)smooth > 2 * A.vbox / A.velfac);
                    P.pos1 = (P.dr2 + (double)smooth) / 2.;
                    P.zrange = ((double)smooth - P.dr2) / 2.;
                } else {
                    P.dr2 = pair_dr2(los, pp, A.box);
                    smooth = A.h[p];
                    const float sm2 = smooth * smooth;
                    have = !((double)sm2 - P.dr2 <= 0);              // absorption.cpp:182
                    P.zrange = have ? sqrt((double)sm2 - P.dr2) : 0.0;
                }
                P.inv_s2 = 1.0 / ((double)smooth * (double)smooth);
                if (have) {
                    P.zlow = (int)floor((P.pos1 - P.zrange) / boxtokpc);
                    npix = max(0ll, (long long)(int)ceil((P.pos1 + P.zrange) / boxtokpc) - P.zlow + 1);
                }
            }
            have = npix > 0;
            // its slots: exclusive scan of the pixel counts
            long long incl = npix;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const long long t = __shfl_up(incl, d, 64);
                if (lane >= d) incl += t;
            }
            const long long total = __shfl(incl, 63, 64);
            P.start = incl - npix;
            const unsigned long long live = __ballot(have);
            wave_sync();   // the previous batch's pairs have been read
            if (have) {
                const int at = __popcll(live & below);
                ColPair &d = mine[at];
                for (int f = 0; f < nf; ++f) dens[f * kColThreads + at] = A.lines[f0 + f].dens[p];
                d.pos1 = P.pos1;
                d.zrange = P.zrange;
                d.dr2 = P.dr2;
                d.inv_s2 = P.inv_s2;
                d.start = P.start;
                d.zlow = P.zlow;
            }
            for (long long s0 = 0; s0 < total; s0 += 64) {
                // pair of slot s0 + lane: the pairs that start at or before it,
                // by marking the slots at which one starts
                mark[lane] = 0;
                wave_sync();
                const long long rel = P.start - s0;
                if (have && rel >= 0 && rel < 64) mark[(int)rel] = 1;
                wave_sync();
                const unsigned long long starts = __ballot(mark[lane] != 0);
                const int before = __popcll(__ballot(have && rel < 0));
                if (s0 + lane < total) {
                    const int at = before + __popcll(starts & (below << 1 | 1ull)) - 1;
                    const ColPair &c = mine[at];
                    const int z = c.zlow + (int)(s0 + lane - c.start);
                    const double plow = boxtokpc * z - c.pos1;
                    const double frac = kern_frac(A.kernel, plow, plow + boxtokpc, c.inv_s2, c.dr2, c.zrange);
                    const int j = wrap_pixel(z, A.nbins);
                    for (int f = 0; f < nf; ++f) {
                        double *row = kLds ? smem + (size_t)f * A.nbins : A.lines[f0 + f].out + (size_t)w.los * A.nbins;
                        row_add<kLds>(&row[j], (double)dens[f * kColThreads + at] * frac);
                    }
                }
                wave_sync();   // the marks have been read
            }
        }
        if (kLds) {
            __syncthreads();
            for (int f = 0; f < nf; ++f) {
                double *out_row = A.lines[f0 + f].out + (size_t)w.los * A.nbins;
                const double *row = smem + (size_t)f * A.nbins;
                for (int j = threadIdx.x; j < A.nbins; j += kColThreads) {
                    if (w.direct)
                        out_row[j] = row[j];
                    else if (row[j] != 0.0)
                        unsafeAtomicAdd(&out_row[j], row[j]);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Isolated throughput of the FP32 sample evaluator (kernel weight x profile),
// no memory traffic: each thread walks u = (tid + i * stride) * du over
// [0, umax), the mix of core and wing samples of a pixel window.

__global__ __launch_bounds__(kThreads) void voigt_peak_kernel(long long per_thread, double du, double umax,
                                                              float a, float *sink)
{
    __shared__ __attribute__((aligned(16))) float ptab[kPTableSize];
    for (int i = threadIdx.x; i < kPTableSize; i += kThreads) ptab[i] = d_ptab[i];
    __syncthreads();
    const VoigtP va = make_voigt_p(a, false);
    const long long tid = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    const long long nthreads = (long long)gridDim.x * blockDim.x;
    float acc = 0.0f;
    const float w = 0.25f;
    double u = fmod((double)tid * du, umax);
    const double step = fmod((double)nthreads * du, umax);
    for (long long i = 0; i < per_thread; ++i) {
        acc = __builtin_fmaf(w, voigt32(va, (float)u, ptab), acc);
        u += step;
        if (u >= umax) u -= umax;
    }
    if (acc == -1.0f) sink[0] = acc;   // keeps the loop live; never true
}

// H(a, u_i) by the deposit kernel's FP32 profile at the points u_i rounded
// to FP32, one lane per point (the profile's accuracy check); the damping
// parameter is set up as for a pair.
__global__ __launch_bounds__(kThreads) void voigt_eval_kernel(const double *u, long long n, double a, float *out)
{
    __shared__ __attribute__((aligned(16))) float ptab[kPTableSize];
    for (int i = threadIdx.x; i < kPTableSize; i += kThreads) ptab[i] = d_ptab[i];
    __syncthreads();
    const VoigtP va = make_voigt_p(a, false);
    for (long long i = blockIdx.x * (long long)kThreads + threadIdx.x; i < n; i += (long long)gridDim.x * kThreads)
        out[i] = voigt32(va, (float)u[i], ptab);
}

int launch_voigt_eval(const double *u, long long n, double a, float *out, hipStream_t s)
{
    if (n <= 0) return FSAMD_OK;
    const long long nb = std::min<long long>((n + kThreads - 1) / kThreads, 4096);
    voigt_eval_kernel<<<(int)nb, kThreads, 0, s>>>(u, n, a, out);
    FSAMD_HIP(hipGetLastError());
    return FSAMD_OK;
}

// ---------------------------------------------------------------------------
// Launchers

size_t deposit_lds_bytes(int nbins) { return sizeof(double) * (size_t)nbins; }

static size_t colden_shm(bool lds, int nbins, int fields)
{
    return (size_t)fields * (lds ? colden_lds_bytes(nbins) : colden_lds_bytes(0));
}

template <int kG>
static size_t tau_static_lds(int waves)
{
    switch (waves) {
    case 2: return static_lds((const void *)tau_kernel<kG, true, false, 128>);
    case 8: return static_lds((const void *)tau_kernel<kG, true, false, 512>);
    default: return static_lds((const void *)tau_kernel<kG, true, false, 256>);   // the counting variant's too
    }
}

size_t deposit_static_lds(bool tau, int gsize, int waves)
{
    // (column density: with the densities of one field)
    if (!tau) return static_lds((const void *)colden_kernel<true>) + colden_lds_bytes(0);
    return gsize == 16 ? tau_static_lds<16>(waves) : gsize == 32 ? tau_static_lds<32>(waves) : tau_static_lds<64>(waves);
}

int raise_lds_limit(const void *fn, size_t shm)
{
    static std::mutex m;
    static std::unordered_map<const void *, size_t> limit;
    std::lock_guard<std::mutex> g(m);
    size_t &cur = limit[fn];
    if (shm > cur) {
        FSAMD_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
        cur = shm;
    }
    return FSAMD_OK;
}

template <int kG, bool kLds, bool kStats, int kBlock>
static int launch_tau_k(const DepositArgs &A, const WorkItem *items, int item_base, int nblocks, int use_queue,
                        size_t shm, hipStream_t s)
{
    int rc;
    if (kLds && (rc = raise_lds_limit((const void *)tau_kernel<kG, kLds, kStats, kBlock>, shm))) return rc;
    tau_kernel<kG, kLds, kStats, kBlock><<<nblocks, kBlock, shm, s>>>(A, items, item_base, use_queue);
    return FSAMD_OK;
}

// Wavefronts per block (per sightline work item) of the tau kernel: 2, 4 or
// 8 with the row in LDS; the counting variant and the global-row variant
// are built for 4 only.
int effective_waves(bool lds, bool stats, int waves)
{
    if (stats || !lds) return 4;
    return waves == 2 || waves == 8 ? waves : 4;
}

template <int kG, bool kLds>
static int launch_tau(const DepositArgs &A, const WorkItem *items, int item_base, int nblocks, int use_queue,
                      size_t shm, int waves, hipStream_t s)
{
    if (A.stats) return launch_tau_k<kG, kLds, true, 256>(A, items, item_base, nblocks, use_queue, shm, s);
    if constexpr (!kLds) {
        return launch_tau_k<kG, kLds, false, 256>(A, items, item_base, nblocks, use_queue, shm, s);
    } else {
        switch (effective_waves(kLds, false, waves)) {
        case 2: return launch_tau_k<kG, kLds, false, 128>(A, items, item_base, nblocks, use_queue, shm, s);
        case 8: return launch_tau_k<kG, kLds, false, 512>(A, items, item_base, nblocks, use_queue, shm, s);
        default: return launch_tau_k<kG, kLds, false, 256>(A, items, item_base, nblocks, use_queue, shm, s);
        }
    }
}

int launch_deposit(bool tau, bool lds, int gsize, int waves, const DepositArgs &A, const WorkItem *items,
                   int item_base, int nblocks, int use_queue, hipStream_t s)
{
    const size_t shm = tau ? (lds ? deposit_lds_bytes(A.nbins) : 0) : colden_shm(lds, A.nbins, A.fields);
    int rc = FSAMD_OK;
    if (tau) {
        if (gsize == 16)
            rc = lds ? launch_tau<16, true>(A, items, item_base, nblocks, use_queue, shm, waves, s)
                     : launch_tau<16, false>(A, items, item_base, nblocks, use_queue, shm, waves, s);
        else if (gsize == 32)
            rc = lds ? launch_tau<32, true>(A, items, item_base, nblocks, use_queue, shm, waves, s)
                     : launch_tau<32, false>(A, items, item_base, nblocks, use_queue, shm, waves, s);
        else
            rc = lds ? launch_tau<64, true>(A, items, item_base, nblocks, use_queue, shm, waves, s)
                     : launch_tau<64, false>(A, items, item_base, nblocks, use_queue, shm, waves, s);
        if (rc) return rc;
    } else {
        if (lds) {
            if (int rc2 = raise_lds_limit((const void *)colden_kernel<true>, shm)) return rc2;
            colden_kernel<true><<<nblocks, kColThreads, shm, s>>>(A, items, item_base, use_queue);
        } else {
            colden_kernel<false><<<nblocks, kColThreads, shm, s>>>(A, items, item_base, use_queue);
        }
    }
    FSAMD_HIP(hipGetLastError());
    return FSAMD_OK;
}

int launch_tau_fixup(const DepositArgs &A, const WorkItem *items, int nblocks, hipStream_t s)
{
    // the counting variant only when counters are collected
    if (A.stats)
        tau_fixup_kernel<true><<<nblocks, kThreads, 0, s>>>(A, items);
    else
        tau_fixup_kernel<false><<<nblocks, kThreads, 0, s>>>(A, items);
    FSAMD_HIP(hipGetLastError());
    return FSAMD_OK;
}

int launch_voigt_peak(long long per_thread, int nblocks, double du, double umax, float a, float *sink,
                      hipStream_t s)
{
    voigt_peak_kernel<<<nblocks, kThreads, 0, s>>>(per_thread, du, umax, a, sink);
    FSAMD_HIP(hipGetLastError());
    return FSAMD_OK;
}

template <int kG, int kBlock>
static int occ_tau_k(bool lds, size_t shm)
{
    int nb = 0;
    hipError_t e = lds ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, tau_kernel<kG, true, false, kBlock>, kBlock, shm)
                       : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, tau_kernel<kG, false, false, 256>, 256, 0);
    // (the global-row variant is built with 256 threads only: effective_waves)
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return 1;
    }
    return nb;
}

template <int kG>
static int occ_tau(bool lds, size_t shm, int waves)
{
    switch (effective_waves(lds, false, waves)) {
    case 2: return occ_tau_k<kG, 128>(lds, shm);
    case 8: return occ_tau_k<kG, 512>(lds, shm);
    default: return occ_tau_k<kG, 256>(lds, shm);
    }
}

// Fields a column-density item takes: all of them, or as many (in parts of
// nearly equal size) as leave room for a second block on the CU, and one
// where a single row is larger than that.
int colden_fields(int nlines, int nbins)
{
    constexpr size_t kCuLds = 160 * 1024;
    const size_t room = kCuLds / 2 - std::min(kCuLds / 2, static_lds((const void *)colden_kernel<true>) + 1024);
    const int most = (int)std::max<size_t>(1, room / colden_lds_bytes(nbins));
    const int parts = (nlines + most - 1) / most;
    return (nlines + parts - 1) / parts;
}

int deposit_blocks_per_cu(bool tau, bool lds, int gsize, int waves, int nbins, int fields)
{
    int nb = 0;
    const size_t shm = tau ? (lds ? deposit_lds_bytes(nbins) : 0) : colden_shm(lds, nbins, fields);
    if (tau) {
        nb = gsize == 16 ? occ_tau<16>(lds, shm, waves)
             : gsize == 32 ? occ_tau<32>(lds, shm, waves) : occ_tau<64>(lds, shm, waves);
    } else {
        hipError_t e = lds ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, colden_kernel<true>, kColThreads, shm)
                           : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, colden_kernel<false>, kColThreads, shm);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            nb = 1;
        }
    }
    return nb < 1 ? 1 : nb;
}

}  // namespace fsamd

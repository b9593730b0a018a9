// Device Voigt profile H(a, u) = Re w(u + i a), w the Faddeeva function.
//
// The reference evaluates Re w with the FP64 Faddeeva package
// (fake_spectra/singleabs.h:56-61 -> Faddeeva.cpp:679-971).  The fused
// deposit kernel evaluates it in FP32 instead, for damping parameters
// 0 <= a <= kA32Max, from two expansions:
//
//    H = exp(a^2 - u^2) cos(2au) - (2a/sqrt(pi)) G(u) - (a^3/sqrt(pi)) Z(u)
//  with G = 1 - 2u D(u) = D'(u) (D: Dawson's integral).  This is the Taylor
//  series of w about the real axis, whose even terms sum to Re exp(-z^2) and
//  whose odd terms are those of the entire function (2i/sqrt(pi)) D(z); the
//  a^5 term is below 1e-7 relative for a <= 0.04.  G comes from one table of
//  cubics in t = 16u^2 + 2 (profile_table.h) whose row number and bin edge are
//  bits of t, so core, transition and wing are one code without selects, and
//  exp(a^2 - u^2) cos(2au) is one exp2 of a polynomial in u^2;
//  D''' = (4u^2 - 6) G + 2, and -12 G^2 beyond u = 20.
//
// u arrives in FP32.  The deposit subtracts the sub-sample velocity from the
// kernel-sample offset in FP64 and rounds the difference, so u carries half
// an ulp even where the two nearly cancel; u^2 and the exponent of
// exp(a^2 - u^2) are FP32, and exp amplifies their relative error by ~2u^2
// ln2: the Gaussian term carries ~1.2e-7 u^2 relative error on top of the
// expansions' 3.6e-7 (measured against scipy.special.wofz, a <= 0.04,
// 0 <= u <= 3000).  Summed over a pixel's samples this stays two orders
// below the 1e-5 tau tolerance and the 2e-5 tail-cut guard band.
//
// An FP64 Faddeeva w(z) (voigt64) backs the FP32 path: pixels whose tail-cut
// decision sits within a guard band of tautail, and pairs with a > kA32Max.
// It is accurate to ~1e-13 relative on the path's domain:
//   real axis: w(x) = exp(-x^2) + (2i/sqrt(pi)) D(x), D by Rybicki's sum;
//   |z| >= 8 or y >= 2: Laplace continued fraction;
//   otherwise: Taylor series in y about the real axis.
#pragma once
#include <hip/hip_runtime.h>
#include "profile_table.h"
#include "dawson64_table.h"

namespace fsamd {

constexpr float kA32Max = 0.04f;
constexpr float kInvSqrtPiF = 0.56418958354775628695f;
constexpr double kSqrtPi = 1.77245385090551602729;
constexpr double kTwoOverSqrtPi = 1.12837916709551257390;
constexpr double kLog2E = 1.44269504088896340736;

// Damping parameters up to which the deposit uses the light form of the
// profile: without the a^3 term and with the Gaussian exponent cut to
// a^2 - (1 + 2a^2) u^2.  For a <= kA3Drop the two together change H by at
// most 5.5e-7 relative over all u (the a^3 term at u ~ 3.2; measured against
// scipy.special.wofz).
constexpr float kA3Drop = 2e-3f;

// The profile takes kUScale u, so that t is one fma.
constexpr double kUScale = 4.0;

// Per-pair constants of the FP32 profile.
struct VoigtP {
    // log2 of Re exp(-(u + ia)^2) = exp(a^2 - u^2) cos(2au), with ln cos x =
    // -x^2/2 - x^4/12 - x^6/45 - ...:  l0 + l1 t + l2 u^4 + l3 u^6, t = 16u^2 + 2,
    // from log2(e) (a^2 - (1 + 2a^2) u^2 - (4/3) a^4 u^4 - (64/45) a^6 u^6); the
    // dropped term, (17/2520)(2au)^8, changes H by < 5e-9 relative for a <= 0.04
    float l0, l1, l2, l3;
    float two_a_sqpi;   // 2a/sqrt(pi)
    float a3;           // -a^2/6, 0 in the light form
};

// light (a <= kA3Drop): the terms of the light form are zero, so the full
// code gives the light form's values.
__device__ inline VoigtP make_voigt_p(double a, bool light)
{
    const double a2 = a * a, lc1 = -(1.0 + 2.0 * a2) * kLog2E;
    VoigtP v;
    v.l0 = (float)(a2 * kLog2E - 0.125 * lc1);
    v.l1 = (float)(0.0625 * lc1);
    v.l2 = light ? 0.0f : (float)(-(4.0 / 3.0) * a2 * a2 * kLog2E);
    v.l3 = light ? 0.0f : (float)(-(64.0 / 45.0) * a2 * a2 * a2 * kLog2E);
    v.two_a_sqpi = (float)(a * kTwoOverSqrtPi);
    v.a3 = light ? 0.0f : (float)(a2 * (-1.0 / 6.0));
    return v;
}

// The scale that pair's offsets carry: kUScale up to the rounding of l1, which it
// takes up, so that the Gaussian's exponent l1 t has none of it (it would cost
// up to 6e-8 u^2 of the Gaussian; the table's argument is off by 6e-8 instead, which
// costs G no more than that).
__device__ inline double voigt_uscale(const VoigtP &v, double a)
{
    const double exact = -(1.0 + 2.0 * a * a) * (kLog2E / 16.0);
    return kUScale - 0.5 * kUScale * (16.0 / kLog2E) * (exact - (double)v.l1);   // (exact / l1)^(1/2) kUScale
}

// Largest |u| whose t lies in the table, and the floats the table takes.
constexpr double kVoigtUMax = 2.3e4;
// Beyond it (the wide forms below) G = -1/(2u^2), exact to 3e-9, up to where u^4 a^4
// leaves the range of FP32 numbers.
constexpr float kVoigtTMax = (float)(2ull << FSAMD_P_OCTAVES);
constexpr double kVoigtUWide = 1e8;
constexpr int kPTableSize = FSAMD_P_OCTAVES * FSAMD_P_BINS * 4;
static_assert(FSAMD_P_BINS == 32 && kUScale * kUScale * kVoigtUMax * kVoigtUMax + 2.0 < (double)(2ull << FSAMD_P_OCTAVES),
              "profile_table.h");
static_assert(FSAMD_P_OCTAVES == 32, "a row for every value of the five exponent bits");

// The two terms of H(a, u) = E - (2a/sqrt(pi)) G at u = us/kUScale, |u| <= kVoigtUMax:
// sums over samples take them separately and combine them once.  The
// Gaussian's exponent and the table's argument come from the same t; its
// mantissa's first 5 bits and exponent name the row, its remaining bits are
// the cubic's variable.  14 VALU instructions and one 16-byte LDS read a
// sample in the light form (kA3 = false; 22 and two reads with a table in u and
// a selected wing row), 22 in the full one (35).  kWide: any |u| <= kVoigtUWide, with
// the same values in the table's range.
template <bool kA3 = true, bool kWide = false>
__device__ inline void voigt_terms(const VoigtP &v, float us, const float *tab, float &E, float &G)
{
    const float t = __builtin_fmaf(us, us, 2.0f);
    float y = __builtin_fmaf(t, v.l1, v.l0);
    if (kA3) {
        const float p = __builtin_fmaf(t, 0.0625f, -0.125f);
        y = __builtin_fmaf(p * p, __builtin_fmaf(p, v.l3, v.l2), y);
    }
    E = __builtin_amdgcn_exp2f(y);    // 0 once y passes the FP32 range
    const unsigned edge = __float_as_uint(t) & 0xfffc0000u;
    const float d = t - __uint_as_float(edge);
    const float4 c = *(const float4 *)((const char *)tab + __builtin_amdgcn_ubfe(edge, 14, 14));
    G = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(c.w, d, c.z), d, c.y), d, c.x);
    if (kWide && t >= kVoigtTMax) G = -8.0f * __builtin_amdgcn_rcpf(t);
    if (kA3) {
        // -(a^2/6) D''': (4u^2 - 6) G + 2 loses its digits as 1/u^4, where G -> -1/(2u^2)
        const float D = t > 6402.0f ? G * (G * -12.0f) : __builtin_fmaf(__builtin_fmaf(t, 0.25f, -6.5f), G, 2.0f);
        G = __builtin_fmaf(v.a3, D, G);
    }
}

// H(a, u) at any u (diagnostics): beyond the table the asymptotic series.
__device__ inline float voigt32(const VoigtP &v, float u, const float *tab)
{
    if (!(__builtin_fabsf(u) <= (float)kVoigtUMax)) {
        const float x = 1.0f / (u * u);
        return 0.5f * v.two_a_sqpi * __builtin_fmaf(1.5f * x, x, x);
    }
    float E, G;
    voigt_terms(v, (float)kUScale * u, tab, E, G);
    return __builtin_fmaf(-v.two_a_sqpi, G, E);
}

// ---------------------------------------------------------------------------
// Profile derivatives for the adjoint, FP32.  Besides H the adjoint needs Hu =
// dH/du and F = u dH/du + a dH/da (the response to the thermal width b: all
// sample offsets and a scale as 1/b).  With C = exp(a^2 - u^2) cos(2au), G =
// D'(u), K = dG/d(u^2), x = 2au and T = tan(x)/x - 1:
//   H  = C - (2a/sqrt(pi)) (G - (a^2/6) D''')
//   Hu = -2u [C (1 + 2a^2 (1 + T)) + (2a/sqrt(pi)) (K - (a^2/12) D''''/u)]
//   F  = -2u^2 C (1 + 4a^2 (1 + T)) + 2a^2 C
//        - (2a/sqrt(pi)) [2u^2 (K - (a^2/12) D''''/u) + G - (a^2/2) D''']
// with D''' = (4u^2 - 6) G + 2, D''''/u = -2 D''' - 12 K, beyond u = 20 -12 G^2 and
// -48 G K.  G and K are rows of one index (profile_table.h): no branch on u.
// The short form (a <= kA3Drop) leaves out T and the exponent's terms in u^4 and
// u^6, at most 5e-9 there, and D''' and D'''' beyond u = 20, where they are 1e-8
// of G and K.  It keeps them below: saturated absorbers have gradients from |u| = 3 to 5
// alone, where without them half of the density's were off by more than 1.6e-7 at
// a = 1.95e-3 (2.3e-8 with them; the temperature's 2.3e-7, 7e-8).  2.1M particles, 1024
// sightlines, forward and adjoint: 15.1 ms without them, 15.9 so, 17.2 with the
// full form from a = 5e-4 on.  The table holds K times kKScale, which keeps its
// coefficients normal numbers.
//
// Sums over samples of weight w, in u' = kUScale u: every factor that depends
// on the pair alone is applied once, by finish().
constexpr float kKScale = (float)(1ull << FSAMD_P_DSCALE);

struct GradSums {
    float cC = 0, cG = 0, uC = 0, uK = 0, pC = 0, pK = 0;   // w C, w G, w u' C, w u' K, w u'^2 C, w u'^2 K
    float cD = 0;                                           // w D'''
    float uT = 0, pT = 0;                                   // full form: w u' C T, w u'^2 C T

    // tab: 8 floats a row, G's cubic and K's.  kWide: as in voigt_terms.
    template <bool kFull, bool kWide = false>
    __device__ inline void add(const VoigtP &v, float a2, float w, float us, const float *tab)
    {
        const float t = __builtin_fmaf(us, us, 2.0f);
        float y = __builtin_fmaf(t, v.l1, v.l0);
        if (kFull) {
            const float p = __builtin_fmaf(t, 0.0625f, -0.125f);
            y = __builtin_fmaf(p * p, __builtin_fmaf(p, v.l3, v.l2), y);
        }
        const float C = __builtin_amdgcn_exp2f(y);
        const unsigned edge = __float_as_uint(t) & 0xfffc0000u;
        const float d = t - __uint_as_float(edge);
        const float4 *row = (const float4 *)((const char *)tab + 2 * __builtin_amdgcn_ubfe(edge, 14, 14));
        const float4 g = row[0], k = row[1];
        float G = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(g.w, d, g.z), d, g.y), d, g.x);
        float K = __builtin_fmaf(__builtin_fmaf(__builtin_fmaf(k.w, d, k.z), d, k.y), d, k.x);
        if (kWide && t >= kVoigtTMax) {
            G = -8.0f * __builtin_amdgcn_rcpf(t);
            K = (2.0f * kKScale * G) * G;
        }
        const float wC = w * C, xC = us * wC;
        const bool far = t > 6402.0f;
        float D = __builtin_fmaf(__builtin_fmaf(t, 0.25f, -6.5f), G, 2.0f);
        if (kFull) {
            D = far ? G * (G * -12.0f) : D;
            // D''''/u times kKScale
            const float D4 = far ? G * (K * -48.0f) : __builtin_fmaf(-12.0f, K, (-2.0f * kKScale) * D);
            K = __builtin_fmaf(0.5f * v.a3, D4, K);
            // x^2 = a^2 u'^2 / 4
            const float x2 = 0.25f * a2 * (t - 2.0f);
            const float xT = xC * (x2 * __builtin_fmaf(x2, 2.0f / 15.0f, 1.0f / 3.0f));
            uT += xT;
            pT = __builtin_fmaf(us, xT, pT);
        } else {
            D = far ? 0.0f : D;
            K = __builtin_fmaf(-kKScale * v.a3, D, __builtin_fmaf(-6.0f * v.a3, far ? 0.0f : K, K));
        }
        cD = __builtin_fmaf(w, D, cD);
        cC += wC;
        uC += xC;
        pC = __builtin_fmaf(us, xC, pC);
        cG = __builtin_fmaf(w, G, cG);
        const float xK = us * (w * K);
        uK += xK;
        pK = __builtin_fmaf(us, xK, pK);
    }
    // S = sum w H; SU with sum w Hu = SU / scale; ST and SP with sum w (H + F) = ST +
    // SP / scale^2, scale the pair's voigt_uscale.  H and F cancel to the next
    // order in the wings, so their sum is formed before it is rounded; and
    // H + F integrates to nearly zero over the profile, so the scale, whose
    // rounding would not average out, is left to the caller.
    __device__ inline void finish(const VoigtP &v, float a2, float &S, float &SU, float &ST, float &SP) const
    {
        const float A = v.two_a_sqpi;
        S = __builtin_fmaf(-A, __builtin_fmaf(v.a3, cD, cG), cC);
        SU = -2.0f * (__builtin_fmaf(2.0f * a2, uC + uT, uC) + A * ((1.0f / kKScale) * uK));
        ST = __builtin_fmaf(2.0f * a2, cC, cC) - 2.0f * A * __builtin_fmaf(2.0f * v.a3, cD, cG);
        SP = -2.0f * __builtin_fmaf((1.0f / kKScale) * A, pK, __builtin_fmaf(4.0f * a2, pC + pT, pC));
    }
};

// ---------------------------------------------------------------------------
// FP64 Faddeeva w(z), y >= 0.

__device__ __noinline__ double dawson64(double x)
{
    const double ax = fabs(x);
    if (ax < 0.2) {
        double t = 1.0, s = 1.0;
        const double m = -2.0 * ax * ax;
#pragma unroll 1
        for (int k = 1; k < 14; k++) {
            t *= m / (2 * k + 1);
            s += t;
        }
        return x * s;
    }
    const double h = 0.2;
    const double n0 = 2.0 * floor(0.5 * ax / h + 0.5);
    const double xp = ax - n0 * h;
    const double e1 = exp(2.0 * xp * h), e2 = e1 * e1;
    double up = e1, dn = 1.0 / e1, s = 0.0;
#pragma unroll 1
    for (int i = 0; i < 22; i++) {
        const double n = 2 * i + 1;
        const double g = exp(-(n * h) * (n * h));
        s += g * (up / (n0 + n) + dn / (n0 - n));
        up *= e2;
        dn /= e2;
    }
    const double d = exp(-xp * xp) * s / kSqrtPi;
    return x < 0 ? -d : d;
}

__device__ __noinline__ void w64_contfrac(double x, double y, int nterms, double &wr, double &wi)
{
    double tr = x, ti = y;
    for (int k = nterms; k >= 1; k--) {
        const double den = tr * tr + ti * ti;
        const double c = 0.5 * k / den;
        tr = x - c * tr;
        ti = y + c * ti;
    }
    const double den = tr * tr + ti * ti;
    wr = ti / den / kSqrtPi;
    wi = tr / den / kSqrtPi;
}

__device__ __noinline__ void w64_taylor_y(double x, double y, double &wr, double &wi)
{
    const double w0r = exp(-x * x), w0i = kTwoOverSqrtPi * dawson64(x);
    const double w1r = -2.0 * x * w0r, w1i = -2.0 * x * w0i + kTwoOverSqrtPi;
    double sr = w0r - y * w1i, si = w0i + y * w1r;
    double cr = 0.0, ci = y;
    double pr = w0r, pim = w0i, qr = w1r, qi = w1i;
    int small = 0;
    for (int k = 1; k < 200; k++) {
        const double nr = -2.0 * x * qr - 2.0 * k * pr;
        const double ni = -2.0 * x * qi - 2.0 * k * pim;
        pr = qr;
        pim = qi;
        qr = nr;
        qi = ni;
        const double t = cr;
        cr = -ci * y / (k + 1);
        ci = t * y / (k + 1);
        const double tr = cr * qr - ci * qi, ti = cr * qi + ci * qr;
        sr += tr;
        si += ti;
        if (fabs(tr) + fabs(ti) <= 1e-19 * (fabs(sr) + fabs(si))) {
            if (++small >= 3) break;
        } else {
            small = 0;
        }
    }
    wr = sr;
    wi = si;
}

__device__ inline void w64(double x, double y, double &wr, double &wi)
{
    const double ax = fabs(x);
    double r, i;
    if (y == 0.0) {
        r = exp(-ax * ax);
        i = kTwoOverSqrtPi * dawson64(ax);
    } else if (ax * ax + y * y >= 64.0) {
        w64_contfrac(ax, y, 60, r, i);
    } else if (y >= 2.0) {
        w64_contfrac(ax, y, 400, r, i);
    } else {
        w64_taylor_y(ax, y, r, i);
    }
    wr = r;
    wi = x < 0 ? -i : i;
}

// Re w(u + ia) for 0 <= a <= kA32Max to ~1e-13 relative, without the sums and
// recurrences of w64: nearly every guard-band pixel has such an a.
// |u| < 10: w's Taylor series in a about the real axis to a^9 D^(9): its even
// terms are exp(a^2 - u^2) cos(2au), its odd ones the odd derivatives of
// Dawson's integral, G = D' from pieces of degree 11 in u (gtab64,
// dawson64_table.h) and the others by
//   D''' = (4u^2 - 6) D' + 2,  D^(n+2) = (4u^2 - 4n - 2) D^(n) - 4n(n-1) D^(n-2);
// |u| >= 10: the asymptotic series w ~ (i/sqrt(pi)) sum_n (2n-1)!!/2^n z^-(2n+1),
// 14 terms in complex arithmetic.
__device__ inline double voigt64_small(double a, double u, const double *gtab64)
{
    const double x = fabs(u), p = u * u;
    if (x >= FSAMD_G64_UMAX) {
        // r = 1/z^2, s = sum_n c_n r^n
        const double q = 1.0 / (p + a * a);
        const double ir = x * q, ii = -a * q;              // 1/z
        const double rr = ir * ir - ii * ii, ri = 2.0 * ir * ii;
        double sr = 1.0, si = 0.0;
#pragma unroll 1
        for (int n = 14; n >= 1; --n) {
            const double c = n - 0.5;                      // c_n / c_(n-1)
            const double tr = sr * rr - si * ri, ti = sr * ri + si * rr;
            sr = 1.0 + c * tr;
            si = c * ti;
        }
        // Re (i s / z), and the Gaussian for a = 0
        return exp(a * a - p) - (ir * si + ii * sr) * (1.0 / kSqrtPi);
    }
    const int k = (int)(x * FSAMD_G64_PER_UNIT);
    const double v = x - (k + 0.5) * (1.0 / FSAMD_G64_PER_UNIT);
    const double *c = gtab64 + k * FSAMD_G64_NCOEF;
    double d1 = c[FSAMD_G64_NCOEF - 1];
#pragma unroll
    for (int i = FSAMD_G64_NCOEF - 2; i >= 0; --i) d1 = __builtin_fma(d1, v, c[i]);
    const double a2 = a * a, p4 = 4.0 * p;
    const double d3 = (p4 - 6.0) * d1 + 2.0;
    const double d5 = (p4 - 14.0) * d3 - 24.0 * d1;
    const double d7 = (p4 - 22.0) * d5 - 80.0 * d3;
    const double d9 = (p4 - 30.0) * d7 - 168.0 * d5;
    const double odd = d1 - a2 * (1.0 / 6.0) * (d3 - a2 * (1.0 / 20.0) * (d5 - a2 * (1.0 / 42.0) * (d7 - a2 * (1.0 / 72.0) * d9)));
    // cos(2au), 2au <= 0.8
    const double m = -4.0 * a2 * p;
    double cs = 1.0;
#pragma unroll
    for (int n = 9; n >= 1; --n) cs = __builtin_fma(cs, m * (1.0 / ((2 * n - 1) * (2 * n))), 1.0);
    return exp(a2 - p) * cs - kTwoOverSqrtPi * a * odd;
}

__device__ inline double voigt64(double a, double u)
{
    double r, i;
    w64(u, a, r, i);
    return r;
}

}  // namespace fsamd

// Flux statistics on device-resident optical depths: the mean-flux rescale
// (py_module.cpp:235-262, fluxstatistics.py:26-39), spectrograph smoothing
// (spec_utils.py:5-25), the 1D flux power (fluxstatistics.py:71-108) and the
// flux PDF (fluxstatistics.py:41-49).  All FP64, HBM-bound streaming kernels.
#include "exp_table.h"
#include "fsamd_internal.h"

#include <algorithm>
#include <cmath>
#include <numeric>
#include <type_traits>
#include <vector>

namespace fsamd {

constexpr int kFluxThreads = 256;

template <typename T>
__device__ inline T wave_sum(T v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

// Block-wide sum of kN values per thread; thread 0 returns the totals.
template <int kN>
__device__ inline void block_sum(double (&v)[kN])
{
    __shared__ double part[kN][kFluxThreads / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < kN; ++i) {
        const double s = wave_sum(v[i]);
        if (lane == 0) part[i][wid] = s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 0; i < kN; ++i) {
            double s = 0;
            for (int w = 0; w < kFluxThreads / 64; ++w) s += part[i][w];
            v[i] = s;
        }
    }
    __syncthreads();
}

__device__ const __attribute__((aligned(16))) double d_exp[2 * FSAMD_EXP_N] = FSAMD_EXP_INIT;

// exp(x), |x| cut at 800 where it is 0 or infinite; kNeg: for x <= 0, where one
// fmax cuts (it drops a NaN, which the callers' x cannot be or which they keep):
// table of 2^(j/128) as hi + lo in LDS, polynomial of degree 6 in the rest
// |r| <= ln 2 / 256 (truncation 5e-19); the last addition's rounding is all but
// 0.01 of the 0.51 ulp of its error.  17 instructions where the math library's
// takes 36, which bounded the kernels below instead of HBM.
template <bool kNeg>
__device__ inline double flux_exp(double x, const double2 *tab)
{
    x = kNeg ? fmax(x, -800.0) : x < -800.0 ? -800.0 : x > 800.0 ? 800.0 : x;
    constexpr double kRound = 6755399441055744.0;   // 1.5 2^52: the sum's low bits are rint
    const double kd = __builtin_fma(x, FSAMD_EXP_INV, kRound);
    const int k = __double2loint(kd);
    const double kf = kd - kRound;
    const double r = __builtin_fma(kf, -FSAMD_EXP_STEP_LO, __builtin_fma(kf, -FSAMD_EXP_STEP_HI, x));
    const double2 T = tab[k & (FSAMD_EXP_N - 1)];
    double q = __builtin_fma(r, 1.0 / 120, 1.0 / 24);
    q = __builtin_fma(r, q, 1.0 / 6);
    q = __builtin_fma(r, q, 0.5);
    q = __builtin_fma(r * r, q, r);
    return ldexp(T.x + __builtin_fma(T.x, q, T.y), k >> FSAMD_EXP_LOG2N);
}

__device__ inline void load_exp_table(double2 *tab)
{
    for (int i = threadIdx.x; i < FSAMD_EXP_N; i += blockDim.x) tab[i] = reinterpret_cast<const double2 *>(d_exp)[i];
}

// Sums of t^j exp(-s t), j = 0 .. kMoments, the count of pixels with tau <=
// thresh that they are over (py_module.cpp:242-251), and of those the count
// with t < 0: [kSums][gridDim.x] partial sums.
//
// Bound: FP64 issue, 51 instructions a pixel, close above HBM (one read of the
// field).  The higher moments (two instructions each) let a pass serve the later
// steps of the iteration too (see taylor_step): 4 -> 2 passes for a forest of
// mean flux 0.68, 6 -> 4 for 0.8.  82M pixels: 218 us a pass with three sums and the
// math library's exp, 163 us now (a batch of 4 and 2048 blocks 167; moments to
// the 8th only 153, but a pass more in half of the cases).
constexpr int kMoments = 12;
constexpr int kSums = kMoments + 3;
constexpr int kMomentBlocks = 1536;   // 6 blocks a CU
constexpr int kMomentBatch = 2;       // pixels a thread loads before the first is used
// Pixels a thread has at least: a block's 15 sums over its threads cost as much as
// some 16 pixels (600000 pixels, Newton steps that each need a pass: 156 us a call
// with one, 121 with 8 and 16, 132 with 32; 3M 163, 163, 142 and 144; with three
// sums a pass it was 130 and 144).
constexpr int kMomentPixels = 16;
// Blocks whose sums the host adds up, a launch less a pass (1000 pixels 108 -> 100 us).
constexpr int kMomentFew = 32;

__global__ __launch_bounds__(kFluxThreads) void flux_moments_kernel(const double *tau, long long n, double scale,
                                                                   double thresh, double *partial)
{
    __shared__ double2 etab[FSAMD_EXP_N];
    load_exp_table(etab);
    __syncthreads();
    double v[kSums] = {};
    int used = 0;
    const auto add = [&](double t, double e) {
#pragma unroll
        for (int j = 0; j <= kMoments; ++j) {
            v[j] += e;
            e *= t;
        }
    };
    const auto add_any = [&](double t) {
        if (t > thresh) return;
        ++used;
        v[kMoments + 2] += t < 0.0 ? 1.0 : 0.0;
        add(t, flux_exp<false>(-scale * t, etab));
    };
    const long long stride = (long long)gridDim.x * kFluxThreads;
    long long i = blockIdx.x * (long long)kFluxThreads + threadIdx.x;
    const auto load = [&](double *t) {
#pragma unroll
        for (int q = 0; q < kMomentBatch; ++q) t[q] = tau[i + q * stride];
    };
    double next[kMomentBatch];   // the next batch is in flight while one is summed
    bool more = i + (kMomentBatch - 1) * stride < n;
    if (more) load(next);
    while (more) {
        double t[kMomentBatch];
        bool plain = true;
#pragma unroll
        for (int q = 0; q < kMomentBatch; ++q) t[q] = next[q];
        i += kMomentBatch * stride;
        more = i + (kMomentBatch - 1) * stride < n;
        if (more) load(next);
#pragma unroll
        for (int q = 0; q < kMomentBatch; ++q) plain = plain && t[q] >= 0.0 && t[q] <= thresh;
        if (plain) {
            used += kMomentBatch;
#pragma unroll
            for (int q = 0; q < kMomentBatch; ++q) add(t[q], flux_exp<true>(-scale * t[q], etab));
        } else {
            for (int q = 0; q < kMomentBatch; ++q) add_any(t[q]);
        }
    }
    for (; i < n; i += stride) add_any(tau[i]);
    v[kMoments + 1] = used;
    block_sum<kSums>(v);
    if (threadIdx.x == 0)
        for (int j = 0; j < kSums; ++j) partial[(size_t)j * gridDim.x + blockIdx.x] = v[j];
}

// One block a row: out[row] = sum of in[row][0 .. n)
__global__ __launch_bounds__(kFluxThreads) void row_sum_kernel(const double *in, int n, double *out)
{
    double v[1] = {0.0};
    for (int i = threadIdx.x; i < n; i += kFluxThreads) v[0] += in[(size_t)blockIdx.x * n + i];
    block_sum<1>(v);
    if (threadIdx.x == 0) out[blockIdx.x] = v[0];
}

// F(z) = sum exp(-z t) and G(z) = -F'(z) from the moments at c, by their Taylor
// polynomials.  For t >= 0 a pixel's remainder is at most
// max_t t^J exp(-x t) |z - c|^J / J! <= r^J / sqrt(2 pi J), r = |z - c| / x,
// x = min(z, c), with J = kMoments + 1 for F and (J / x) times that of |z - c|^(J-1)
// for G.  False where the Newton step (F - target) / G would be off by more than
// 1e-14 z: then the field has to be summed at z.
static bool taylor_step(const double *sum, double c, double z, double target, double &F, double &G)
{
    const double used = sum[kMoments + 1], d = z - c, x = std::min(z, c), r = std::fabs(d) / x;
    if (sum[kMoments + 2] != 0 || !(r < 0.5)) return false;
    F = G = 0;
    double f = 1;   // (-d)^j / j!
    for (int j = 0; j <= kMoments; ++j) {
        F += f * sum[j];
        if (j < kMoments) G += f * sum[j + 1];
        f *= -d / (j + 1);
    }
    if (!std::isfinite(F) || !std::isfinite(G)) return false;
    constexpr double J = kMoments + 1;
    const double rem = used * std::pow(r, J - 1) / std::sqrt(2 * M_PI * J);
    return rem * r + std::fabs((F - target) / G) * rem * J / x <= 1e-14 * z * G;
}

// Gaussian smoothing along rows with periodic wrap, weights w[0 .. nw), nw = 2r + 1
// (the correlation of scipy.ndimage.gaussian_filter1d, mode 'wrap').
//
// Bound: HBM, a read and a write.  A block stages a stretch of `cols` columns
// of a row with its taps' margin (of several rows where they are short) and the
// weights in LDS, kResTaps taps at a time; a thread has kResOut neighbouring
// outputs, so that two pixels and two weights read feed eight multiply-adds.
// 40000 rows of 2048, 9 taps: 900 -> 270 us (4.9 TB/s);
// 9765 of 2048, 57 taps, a call: 1060 -> 131 us.
constexpr int kResOut = 4;
constexpr int kResCols = kResOut * kFluxThreads;
constexpr int kResTaps = 256;   // even: only the last stretch of taps has an odd one
constexpr int kResLds = 2560;   // doubles of short rows in a block: 20 KB, with the taps seven blocks a CU

struct ResTile {
    int cols, rows, nchunk;     // a block's part: cols columns of rows rows; nchunk parts a row
    int stride;                 // of a staged row, a multiple of kResOut
};

// Parts a call has at least before short rows share a block: fewer than fill the
// chip, they would only wait for each other (1000 rows of 50, 1 and 9 taps: 21.7 and
// 22.3 us a call with 19 rows a block, 20.8 and 21.2 so).
constexpr int kResParts = 512;

static ResTile res_tile(int nrow, int ncol, int nw)
{
    ResTile t;
    t.cols = std::min(ncol, kResCols);
    t.nchunk = (ncol + t.cols - 1) / t.cols;
    t.stride = (t.cols + kResOut - 1) / kResOut * kResOut + (std::min(nw, kResTaps) + kResOut) / kResOut * kResOut;
    const int groups = (t.cols + kResOut - 1) / kResOut;
    t.rows = std::max(1, std::min(std::min(kFluxThreads / groups, kResLds / t.stride), nrow / kResParts));
    return t;
}

__global__ __launch_bounds__(kFluxThreads) void res_corr_kernel(const double *in, double *out, int nrow, int ncol,
                                                               const double *w, int nw, ResTile tile, long long nparts)
{
    extern __shared__ double2 shc[];
    double *taps = reinterpret_cast<double *>(shc), *pix = taps + (min(nw, kResTaps) + 1) / 2 * 2;
    const int groups = (tile.cols + kResOut - 1) / kResOut;
    const int myrow = threadIdx.x / groups, at = threadIdx.x % groups * kResOut;
    double *mine = pix + myrow * tile.stride + at;
    // a short row is loaded by a wavefront, a long one by the block
    const int lrow = tile.rows > 1 ? threadIdx.x / 64 : 0, lrows = tile.rows > 1 ? kFluxThreads / 64 : 1;
    const int lcol = tile.rows > 1 ? threadIdx.x % 64 : threadIdx.x, lcols = tile.rows > 1 ? 64 : kFluxThreads;
    for (long long part = blockIdx.x; part < nparts; part += gridDim.x) {
        const int row0 = (int)(part / tile.nchunk) * tile.rows, col0 = (int)(part % tile.nchunk) * tile.cols;
        const int rows = min(tile.rows, nrow - row0), cols = min(tile.cols, ncol - col0);
        double acc[kResOut] = {};
        for (int k0 = 0; k0 < nw; k0 += kResTaps) {
            const int nk = min(kResTaps, nw - k0), width = cols + nk - 1;
            int first = (col0 - nw / 2 + k0) % ncol;
            if (first < 0) first += ncol;
            __syncthreads();
            for (int k = threadIdx.x; k < nk; k += kFluxThreads) taps[k] = w[k0 + k];
            for (int r = lrow; r < rows; r += lrows) {
                const double *src = in + (size_t)(row0 + r) * ncol;
                for (int x = lcol; x < width; x += lcols) {
                    int j = first + x;
                    if (j >= ncol) j -= ncol;
                    if (j >= ncol) j %= ncol;   // more taps than columns
                    pix[r * tile.stride + x] = src[j];
                }
            }
            __syncthreads();
            if (myrow >= rows) continue;
            double2 s0 = *(const double2 *)mine, s1 = *(const double2 *)(mine + 2);
            for (int k = 0; k + 1 < nk; k += 2) {
                const double2 s2 = *(const double2 *)(mine + k + 4), t = *(const double2 *)(taps + k);
                acc[0] = fma(t.y, s0.y, fma(t.x, s0.x, acc[0]));
                acc[1] = fma(t.y, s1.x, fma(t.x, s0.y, acc[1]));
                acc[2] = fma(t.y, s1.y, fma(t.x, s1.x, acc[2]));
                acc[3] = fma(t.y, s2.x, fma(t.x, s1.y, acc[3]));
                s0 = s1;
                s1 = s2;
            }
            if (nk & 1) {
                const double t = taps[nk - 1];
                acc[0] = fma(t, s0.x, acc[0]);
                acc[1] = fma(t, s0.y, acc[1]);
                acc[2] = fma(t, s1.x, acc[2]);
                acc[3] = fma(t, s1.y, acc[3]);
            }
        }
        // through LDS, for whole lines
        __syncthreads();
        if (myrow < rows) {
            *(double2 *)mine = make_double2(acc[0], acc[1]);
            *(double2 *)(mine + 2) = make_double2(acc[2], acc[3]);
        }
        __syncthreads();
        for (int r = lrow; r < rows; r += lrows)
            for (int x = lcol; x < cols; x += lcols)
                out[(size_t)(row0 + r) * ncol + col0 + x] = pix[r * tile.stride + x];
    }
}

// ---- mixed-radix FFT power spectrum ---------------------------------------
// Self-sorting (Stockham) decimation-in-time FFT of length n = R_1 R_2 ...
// R_S in one LDS buffer.  Stage s with radix R, after the transforms of length
// p = R_1 ... R_{s-1}: for i in [0, n/R), k = i mod p,
//   u_r = a[i + r n/R] W_n^{r k n/(p R)},   a'[(i - k) R + k + q p] = sum_r u_r W_R^{r q};
// a thread holds its values of a stage in registers between the barriers.
// Two real sightlines a, b share one complex transform Z of a + i b; the sum
// of their powers at mode k is (|Z_k|^2 + |Z_{n-k}|^2) / 2, which is all the
// flux power needs (it averages the power over sightlines).
//
// Bound: LDS traffic and FP64 issue.  Radix 8 with a block of n/8 threads: four
// stages for 2048 pixels; the first reads the sightlines and stores at stride 8,
// which the swizzle spreads over the banks.  One buffer, the sums of the power
// in registers: 34 KB a block of 2048 pixels, four blocks a CU.  Powers of two
// have the next pair's pixels on their way over a pair's later stages: 395 -> 280
// us for 40000 sightlines of 2048 (598 with radix 4 and two buffers).  Other
// lengths: 13333 of 1500 510 -> 175 us, 4000 of 5000 (a direct sum before) 48 ->
// 0.20 ms, the prime 2003 6.6 -> 1.4 ms for 2000.

constexpr int kFftMaxStages = 40;
constexpr int kFftPoints = 8;          // values a thread holds, n <= kFftPoints * threads
constexpr int kFftMaxThreads = 896;
struct FftPlan {
    int nst;
    int twiddle[kFftMaxStages];   // where the stage's twiddles start in the table
    unsigned char any;            // a radix without a stage of its own
    short radix[kFftMaxStages];
};

// Radices 8, 4, 2, 3, 5, 7 first, then any remaining prime factors.
static FftPlan fft_plan(int n)
{
    FftPlan f{};
    for (int r : {8, 4, 2, 3, 5, 7})
        while (n % r == 0) { f.radix[f.nst++] = (short)r; n /= r; }
    for (int q = 11; n > 1; q += 2)
        while (n % q == 0) { f.radix[f.nst++] = (short)q; n /= q; f.any = 1; }
    int p = 1;
    for (int st = 0; st < f.nst; ++st) {
        f.twiddle[st] = p - 1;    // (R - 1) p a stage, sum over the stages before
        p *= f.radix[st];
    }
    return f;
}

__device__ inline double2 cmul(double2 a, double2 b)
{
    return make_double2(fma(a.x, b.x, -a.y * b.y), fma(a.x, b.y, a.y * b.x));
}
__device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ inline double2 cmul_mi(double2 a) { return make_double2(a.y, -a.x); }   // -i a

// exp(-2 pi i m / n)
__device__ inline double2 unit_root(int m, int n)
{
    double s, c;
    sincospi(2.0 * m / n, &s, &c);
    return make_double2(c, -s);
}

// In place: v_q = sum_r u_r W_R^{r q}
template <int R>
__device__ inline void dft(double2 (&u)[R])
{
    if constexpr (R == 2) {
        const double2 a = u[0];
        u[0] = cadd(a, u[1]);
        u[1] = csub(a, u[1]);
    } else if constexpr (R == 4) {
        const double2 s02 = cadd(u[0], u[2]), d02 = csub(u[0], u[2]);
        const double2 s13 = cadd(u[1], u[3]), d13 = cmul_mi(csub(u[1], u[3]));
        u[0] = cadd(s02, s13);
        u[1] = cadd(d02, d13);
        u[2] = csub(s02, s13);
        u[3] = csub(d02, d13);
    } else if constexpr (R == 8) {
        double2 e[4] = {u[0], u[2], u[4], u[6]}, o[4] = {u[1], u[3], u[5], u[7]};
        dft<4>(e);
        dft<4>(o);
        constexpr double h = 0.70710678118654752440;
        o[1] = make_double2(h * (o[1].x + o[1].y), h * (o[1].y - o[1].x));
        o[2] = cmul_mi(o[2]);
        o[3] = make_double2(h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            u[q] = cadd(e[q], o[q]);
            u[q + 4] = csub(e[q], o[q]);
        }
    } else {
        // cos and sin of 2 pi m / R
        constexpr double c3[] = {1.0, -0.5, -0.5}, s3[] = {0.0, 0.86602540378443864676, -0.86602540378443864676};
        constexpr double c5[] = {1.0, 0.30901699437494742410, -0.80901699437494742410, -0.80901699437494742410,
                                 0.30901699437494742410};
        constexpr double s5[] = {0.0, 0.95105651629515357212, 0.58778525229247312917, -0.58778525229247312917,
                                 -0.95105651629515357212};
        constexpr double c7[] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624,
                                 -0.90096886790241912624, -0.22252093395631440429, 0.62348980185873353053};
        constexpr double s7[] = {0.0, 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048,
                                 -0.43388373911755812048, -0.97492791218182360702, -0.78183148246802980871};
        double2 v[R];
#pragma unroll
        for (int q = 0; q < R; ++q) {
            v[q] = u[0];
#pragma unroll
            for (int r = 1; r < R; ++r) {
                const int m = (r * q) % R;
                const double c = R == 3 ? c3[m % 3] : R == 5 ? c5[m % 5] : c7[m % 7];
                const double s = R == 3 ? s3[m % 3] : R == 5 ? s5[m % 5] : s7[m % 7];
                v[q] = cadd(v[q], cmul(u[r], make_double2(c, -s)));
            }
        }
#pragma unroll
        for (int q = 0; q < R; ++q) u[q] = v[q];
    }
}

// threadIdx.x as a value of its own at each use: a stage's addresses, the same
// for every pair, are computed where they are used instead of all being kept
// (and spilled) over the loop.
__device__ inline int fft_thread()
{
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

__device__ inline int fft_swizzle(int j, int mask) { return j ^ ((j >> 3) & mask); }

// What a plan's kernel holds: the stages of radices 8, 4 and 2 and the next
// pair's pixels on their way; all stages with a radix of their own; any.
enum FftKind { kFftPow2, kFftSmall, kFftAny };

// The two sightlines' optical depths at z + r m, r < R; row1 is NULL for the
// odd one out, whose partner is zero.
template <int R>
__device__ inline void load_pair(const double *row0, const double *row1, int z, int m, double2 (&u)[R])
{
#pragma unroll
    for (int r = 0; r < R; ++r) u[r] = make_double2(row0[z + r * m], row1 ? row1[z + r * m] : 0.0);
}

// In place: exp(-s tau) / mean - 1
template <int R, bool kTable>
__device__ inline void pair_flux(double2 (&u)[R], bool two, double scale, double inv_mean, const double2 *etab)
{
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const double x = -scale * u[r].x, y = -scale * u[r].y;
        u[r].x = (kTable ? flux_exp<false>(x, etab) : exp(x)) * inv_mean - 1.0;
        u[r].y = two ? (kTable ? flux_exp<false>(y, etab) : exp(y)) * inv_mean - 1.0 : 0.0;
        if (r % 2 == 1) __builtin_amdgcn_sched_barrier(0);   // four at a time, not all in registers at once
    }
}

// The first stage for radix 8, one butterfly a thread, on pixels already loaded
__device__ inline void fft_first8(double2 *a, double2 (&u)[8], bool two, int n, double scale, double inv_mean,
                                  const double2 *etab)
{
    const int i = fft_thread();
    if (i < n / 8) {
        pair_flux<8, true>(u, two, scale, inv_mean, etab);
        dft<8>(u);
    }
    __syncthreads();
    if (i < n / 8) {
#pragma unroll
        for (int q = 0; q < 8; ++q) a[fft_swizzle(i * 8 + q, 7)] = u[q];
    }
    __syncthreads();
}

// One stage of radix R; the first one (kFirst) reads the sightlines.  mask_in,
// mask_out: the swizzle of the buffer as it is read and as it is left.
template <int R, bool kFirst, bool kTable>
__device__ inline void fft_stage(double2 *a, const double2 *tw, int n, int p, int mask_in, int mask_out,
                                 const double *row0, const double *row1, double scale, double inv_mean,
                                 const double2 *etab)
{
    constexpr int kC = (kFftPoints + R - 1) / R;
    const int m = n / R;
    const float inv_p = 1.0f / p;
    const int tid = fft_thread();
    double2 u[kC][R];
#pragma unroll
    for (int c = 0; c < kC; ++c) {
        const int i = tid + c * blockDim.x;
        if (i >= m) continue;
        if (kFirst) {
            load_pair<R>(row0, row1, i, m, u[c]);
            pair_flux<R, kTable>(u[c], row1, scale, inv_mean, etab);
        } else {
            const int k = i - p * (int)((i + 0.5f) * inv_p);
            u[c][0] = a[fft_swizzle(i, mask_in)];
#pragma unroll
            for (int r = 1; r < R; ++r) u[c][r] = cmul(a[fft_swizzle(i + r * m, mask_in)], tw[(r - 1) * p + k]);
        }
        dft<R>(u[c]);
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kC; ++c) {
        const int i = tid + c * blockDim.x;
        if (i >= m) continue;
        const int k = kFirst ? 0 : i - p * (int)((i + 0.5f) * inv_p);
        const int j = (i - k) * R + k;
#pragma unroll
        for (int q = 0; q < R; ++q) a[fft_swizzle(j + q * p, mask_out)] = u[c][q];
    }
    __syncthreads();
}

// exp(-2 pi i t / n), 0 <= t < n, from a table of t <= n/2
__device__ inline double2 half_root(const double2 *half, int t, int n)
{
    double2 w = half[min(t, n - t)];
    w.y = 2 * t > n ? -w.y : w.y;
    return w;
}

// A stage of any odd radix R, O(R) terms an output: outputs q and R - q share
// the sums C = sum u_r cos and S = sum u_r sin of 2 pi r q / R, C -+ i S.
__device__ inline void fft_stage_any(double2 *a, const double2 *half, int n, int p, int R, int mask_in)
{
    constexpr int kC = (kFftPoints * 12 / 11 + 1) / 2 + 1;   // m (R + 1) / 2 <= (n + n/11) / 2 sums over n/8 threads
    const int m = n / R, nsum = m * ((R + 1) / 2);
    const int tstep = n / (p * R), tid = fft_thread(), T = blockDim.x;
    if (p > 1) {
        for (int j = tid; j < n; j += T) {
            const int r = j / m, k = (j - r * m) % p;
            double2 &v = a[fft_swizzle(j, mask_in)];
            v = cmul(v, half_root(half, r * k * tstep, n));
        }
        __syncthreads();
    }
    double2 C[kC], S[kC];
#pragma unroll
    for (int c = 0; c < kC; ++c) {
        const int o = tid + c * T;
        C[c] = S[c] = make_double2(0.0, 0.0);
        if (o >= nsum) continue;
        const int q = o / m, i = o - q * m;
        int t = 0;
        for (int r = 0; r < R; ++r) {
            const double2 w = half_root(half, t, n), u = a[fft_swizzle(i + r * m, mask_in)];
            C[c] = make_double2(fma(u.x, w.x, C[c].x), fma(u.y, w.x, C[c].y));
            S[c] = make_double2(fma(u.x, -w.y, S[c].x), fma(u.y, -w.y, S[c].y));
            t += q * m;
            t -= t >= n ? n : 0;
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kC; ++c) {
        const int o = tid + c * T;
        if (o >= nsum) continue;
        const int q = o / m, i = o - q * m;
        const int k = i % p, j = (i - k) * R + k;
        const double2 is = cmul_mi(S[c]);   // -i S
        a[j + q * p] = cadd(C[c], is);
        if (q > 0) a[j + (R - q) * p] = csub(C[c], is);
    }
    __syncthreads();
}

// The stages' twiddles: of stage s, radix R, tw[twiddle[s] + (r - 1) p + k] = W_n^{r k n/(p R)}.
__global__ void fft_twiddle_kernel(double2 *tw, FftPlan fp)
{
    const int at = blockIdx.x * blockDim.x + threadIdx.x;
    int p = 1;
    for (int st = 0; st < fp.nst; ++st) {
        const int R = fp.radix[st], e = at - fp.twiddle[st];
        if (e < (R - 1) * p) {
            if (e >= 0) tw[at] = unit_root((e / p + 1) * (e % p), p * R);
            return;
        }
        p *= R;
    }
}

// Each block transforms sightline pairs blockIdx.x, blockIdx.x + gridDim.x, ...
// and writes the sum of their powers to part[blockIdx.x][k]; the blocks'
// rows are then summed in block order, so the result does not depend on
// scheduling.
template <FftKind kKind>
__global__ __launch_bounds__(kFftMaxThreads) void flux_fft_kernel(const double *tau, int nlos, int npix, double scale,
                                                                 double inv_mean, const double2 *tw, FftPlan fp,
                                                                 double *part)
{
    constexpr bool kTable = kKind != kFftAny;   // whose sums are far longer than the exponentials
    extern __shared__ double2 shc[];
    double2 *a = shc, *half = shc + npix, *etab = half;   // one of the two tables
    constexpr int kModes = kFftPoints / 2 + 1;   // npix/2 + 1 modes over npix/8 threads
    double acc[kModes] = {};
    const int nk = npix / 2 + 1, T = blockDim.x;
    if (kTable)
        load_exp_table(etab);
    else
        for (int m = threadIdx.x; m < nk; m += T) half[m] = unit_root(m, npix);
    __syncthreads();
    const int npair = (nlos + 1) / 2;
    double2 next[8];   // kFftPow2: this thread's pixels of the pair to come
    const auto load_next = [&](int pr) {
        const int i = fft_thread();
        if (i >= npix / 8) return;
        const double *row = tau + 2 * (size_t)pr * npix;
        load_pair<8>(row, 2 * pr + 1 < nlos ? row + npix : nullptr, i, npix / 8, next);
    };
    if (kKind == kFftPow2 && (int)blockIdx.x < npair) load_next(blockIdx.x);
    for (int pr = blockIdx.x; pr < npair; pr += gridDim.x) {
        const size_t r0 = 2 * (size_t)pr;
        const double *row0 = tau + r0 * npix, *row1 = r0 + 1 < (size_t)nlos ? row0 + npix : nullptr;
        int p = 1, mask = 0, st = 0;
        if (kKind == kFftPow2) {
            fft_first8(a, next, row1, npix, scale, inv_mean, etab);
            if (pr + (int)gridDim.x < npair) load_next(pr + gridDim.x);
            st = 1;
            p = 8;
            mask = 7;
        }
        for (; st < fp.nst; ++st) {
            const int R = fp.radix[st];
            const double2 *ts = tw + fp.twiddle[st];
            if (st == 0) {
                mask = npix % 8 == 0 ? 7 : 0;   // whole groups of 8
                const auto stage = [&](auto radix) {
                    fft_stage<decltype(radix)::value, true, kTable>(a, ts, npix, p, 0, mask, row0, row1, scale,
                                                                   inv_mean, etab);
                };
                switch (R) {
                case 2: stage(std::integral_constant<int, 2>()); break;
                case 3: stage(std::integral_constant<int, 3>()); break;
                case 4: stage(std::integral_constant<int, 4>()); break;
                case 5: stage(std::integral_constant<int, 5>()); break;
                case 7: stage(std::integral_constant<int, 7>()); break;
                case 8: stage(std::integral_constant<int, 8>()); break;
                default:
                    if (kKind != kFftAny) break;
                    __syncthreads();   // the last pair's power has been read
                    for (int j = threadIdx.x; j < npix; j += T) {
                        double2 u[1];
                        load_pair<1>(row0, row1, j, 0, u);
                        pair_flux<1, false>(u, row1, scale, inv_mean, etab);
                        a[j] = u[0];
                    }
                    mask = 0;
                    __syncthreads();
                    fft_stage_any(a, half, npix, p, R, 0);
                }
            } else {
                const auto stage = [&](auto radix) {
                    fft_stage<decltype(radix)::value, false, kTable>(a, ts, npix, p, mask, 0, row0, row1, scale,
                                                                    inv_mean, etab);
                };
                if (kKind == kFftPow2) {
                    if (R == 8)
                        stage(std::integral_constant<int, 8>());
                    else if (R == 4)
                        stage(std::integral_constant<int, 4>());
                    else
                        stage(std::integral_constant<int, 2>());
                } else {
                    switch (R) {
                    case 2: stage(std::integral_constant<int, 2>()); break;
                    case 3: stage(std::integral_constant<int, 3>()); break;
                    case 4: stage(std::integral_constant<int, 4>()); break;
                    case 5: stage(std::integral_constant<int, 5>()); break;
                    case 7: stage(std::integral_constant<int, 7>()); break;
                    case 8: stage(std::integral_constant<int, 8>()); break;
                    default:
                        if (kKind == kFftAny) fft_stage_any(a, half, npix, p, R, mask);
                    }
                }
                mask = 0;
            }
            p *= R;
        }
        if (fp.nst == 0) {   // one pixel
            double2 u[1];
            __syncthreads();
            load_pair<1>(row0, row1, 0, 0, u);
            pair_flux<1, false>(u, row1, scale, inv_mean, etab);
            if (threadIdx.x == 0) a[0] = u[0];
            __syncthreads();
        }
        // each thread owns modes threadIdx.x + c T
        const int tid = fft_thread();
#pragma unroll
        for (int c = 0; c < kModes; ++c) {
            const int k = tid + c * T;
            if (k >= nk) continue;
            const double2 z = a[fft_swizzle(k, mask)], w = a[fft_swizzle(k == 0 ? 0 : npix - k, mask)];
            acc[c] += 0.5 * ((z.x * z.x + z.y * z.y) + (w.x * w.x + w.y * w.y));
        }
    }
#pragma unroll
    for (int c = 0; c < kModes; ++c) {
        const int k = threadIdx.x + c * T;
        if (k < nk) part[(size_t)blockIdx.x * nk + k] = acc[c];
    }
}

// out[k] = norm * sum over rows of part[row][k], in a fixed order: a block has
// 16 columns (128 bytes of a row), its 16 groups of threads each a run of rows.
// One thread a column took 337 us for 1024 rows of 1025, this 6.
constexpr int kSumCols = 16;
__global__ __launch_bounds__(kFluxThreads) void column_sum_kernel(const double *part, int nrow, int nk, double norm,
                                                                 double *out)
{
    constexpr int kRuns = kFluxThreads / kSumCols;
    __shared__ double sums[kRuns][kSumCols];
    const int col = threadIdx.x % kSumCols, run = threadIdx.x / kSumCols;
    const int k = blockIdx.x * kSumCols + col;
    const int len = (nrow + kRuns - 1) / kRuns, end = min(nrow, (run + 1) * len);
    double s = 0;
    if (k < nk)
#pragma unroll 8
        for (int r = run * len; r < end; ++r) s += part[(size_t)r * nk + k];
    sums[run][col] = s;
    __syncthreads();
    if (run == 0 && k < nk) {
        for (int i = 1; i < kRuns; ++i) s += sums[i][col];
        out[k] = s * norm;
    }
}

// Histogram of exp(-s tau) over nb equal bins of [0, 1], bin edges e_k =
// k / nb as numpy.histogram places them (searchsorted on the edges, the last
// bin closed); values outside [0, 1] are not counted.  f nb is within 2e-11 of
// its value (nb <= 40960), so the edges decide only next to a whole number.
__device__ inline int flux_bin(double f, int nb)
{
    const double x = f * nb, e = rint(x);
    int b = min((int)x, nb - 1);
    if (fabs(x - e) < 1e-9 && e > 0.0 && e < (double)nb) b = f < e / (double)nb ? (int)e - 1 : (int)e;
    return b;
}

// Counts are kept per block in LDS and added to the global bins once per
// block: as many copies of a bin as there is room for, up to one a thread (a
// flux field piles up in few bins, which would serialize the atomics).
//
// Bound: HBM, one read of the field.  82M pixels, 20 bins: 230 -> 145 us, with
// the two divides a pixel and the 256 copies read by one thread a bin gone; 50
// bins, one copy before, a call on 20M pixels: 140 -> 105 us; 40000 bins, one
// copy, on 1e5 pixels 60 -> 48 us.
constexpr int kHistCounts = 10240;   // 40 KB: with the table of exponentials three blocks a CU at the most copies
constexpr int kHistBatch = 4;

// kTable: exp by flux_exp's table, where the LDS holds it beside the bins
template <bool kTable>
__global__ __launch_bounds__(kFluxThreads) void flux_hist_kernel(const double *tau, long long n, double scale, int nb,
                                                                int copies, unsigned long long *counts)
{
    extern __shared__ double2 shc[];
    double2 *etab = shc;
    unsigned int *hist = reinterpret_cast<unsigned int *>(shc + (kTable ? FSAMD_EXP_N : 0));   // [nb][copies]
    if (kTable) load_exp_table(etab);
    for (int i = threadIdx.x; i < nb * copies; i += kFluxThreads) hist[i] = 0;
    __syncthreads();
    const int copy = threadIdx.x & (copies - 1);
    const auto add = [&](double t) {
        const double f = kTable ? flux_exp<false>(-scale * t, etab) : exp(-scale * t);
        if (f >= 0.0 && f <= 1.0) atomicAdd(&hist[flux_bin(f, nb) * copies + copy], 1u);
    };
    const long long stride = (long long)gridDim.x * kFluxThreads;
    long long i = blockIdx.x * (long long)kFluxThreads + threadIdx.x;
    for (; i + (kHistBatch - 1) * stride < n; i += kHistBatch * stride) {
        double t[kHistBatch];
#pragma unroll
        for (int q = 0; q < kHistBatch; ++q) t[q] = tau[i + q * stride];
#pragma unroll
        for (int q = 0; q < kHistBatch; ++q) add(t[q]);
    }
    for (; i < n; i += stride) add(tau[i]);
    __syncthreads();
    if (copies > 1) {   // min(copies, 64) lanes a bin
        const int lanes = min(copies, 64), sub = threadIdx.x & (lanes - 1);
        for (int b = threadIdx.x / lanes; b < nb; b += kFluxThreads / lanes) {
            unsigned int c = 0;
            for (int k = sub; k < copies; k += lanes) c += hist[b * copies + k];
            for (int o = lanes / 2; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
            if (sub == 0) hist[b * copies] = c;
        }
        __syncthreads();
    }
    for (int b = threadIdx.x; b < nb; b += kFluxThreads)   // neighbouring bins in one instruction
        if (const unsigned int c = hist[b * copies]) atomicAdd(&counts[b], (unsigned long long)c);
}

}  // namespace fsamd

using namespace fsamd;

extern "C" {

int fsamd_mean_flux_scale(const double *tau, long long n, double mean_flux_desired, double tol, double thresh,
                          double *scale_out, void *stream)
{
    if (!scale_out || n < 0 || (n > 0 && !tau)) return fail(FSAMD_ERR_ARG, "NULL argument or negative size");
    if (n == 0) {
        *scale_out = 0.0;    // fluxstatistics.py:38-39
        return FSAMD_OK;
    }
    hipStream_t s = (hipStream_t)stream;
    constexpr long long kBlockPixels = (long long)kFluxThreads * kMomentPixels;
    const int nblocks = (int)std::min<long long>(kMomentBlocks, (n + kBlockPixels - 1) / kBlockPixels);
    const bool few = nblocks <= kMomentFew;
    double host[kSums * kMomentFew];
    double *partial = nullptr;
    FSAMD_HIP(hipMalloc(&partial, sizeof(double) * kSums * (nblocks + 1)));
    double *total = partial + (size_t)kSums * nblocks;
    double sum[kSums], centre = 0, scale, newscale = 1;
    int rc = FSAMD_OK;
    for (int it = 0; it < 1000; ++it) {
        scale = newscale;
        double F, G;
        if (it == 0 || !taylor_step(sum, centre, scale, mean_flux_desired * sum[kMoments + 1], F, G)) {
            flux_moments_kernel<<<nblocks, kFluxThreads, 0, s>>>(tau, n, scale, thresh, partial);
            if (!few) row_sum_kernel<<<kSums, kFluxThreads, 0, s>>>(partial, nblocks, total);
            hipError_t e = hipGetLastError();
            if (e == hipSuccess)
                e = hipMemcpyAsync(few ? host : sum, few ? partial : total, sizeof(double) * kSums * (few ? nblocks : 1),
                                   hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipStreamSynchronize(s);
            if (e != hipSuccess) {
                rc = fail(FSAMD_ERR_HIP, std::string("flux moments: ") + hipGetErrorString(e));
                break;
            }
            for (int j = 0; few && j < kSums; ++j)
                sum[j] = std::accumulate(host + j * nblocks, host + (j + 1) * nblocks, 0.0);
            centre = scale;
            F = sum[0];
            G = sum[1];
        }
        // Newton-Raphson on <exp(-s tau)> = mean_flux_desired (py_module.cpp:252-257)
        newscale = scale + (F - mean_flux_desired * sum[kMoments + 1]) / G;
        if (newscale <= 0) newscale = 1e-10;
        if (!(fabs(newscale - scale) > tol * newscale)) break;
        if (it == 999) rc = fail(FSAMD_ERR_ARG, "mean flux rescale did not converge");
    }
    (void)hipFree(partial);
    if (rc) return rc;
    *scale_out = newscale;
    return FSAMD_OK;
}

int fsamd_res_corr(const double *in, double *out, int nrow, int ncol, double sigma, void *stream)
{
    if (nrow < 0 || ncol < 1 || !(sigma > 0) || (nrow > 0 && (!in || !out)))
        return fail(FSAMD_ERR_ARG, "bad arguments to fsamd_res_corr");
    if (nrow == 0) return FSAMD_OK;
    // scipy.ndimage.gaussian_filter1d: truncate = 4, radius = int(4 sigma + 0.5)
    const int r = (int)(4.0 * sigma + 0.5);
    if (r > (1 << 20)) return fail(FSAMD_ERR_UNSUPPORTED, "smoothing radius too large");
    std::vector<double> w(2 * r + 1);
    double tot = 0;
    for (int k = -r; k <= r; ++k) tot += (w[k + r] = std::exp(-0.5 * (double)k * k / (sigma * sigma)));
    for (double &x : w) x /= tot;
    hipStream_t s = (hipStream_t)stream;
    double *dw = nullptr;
    FSAMD_HIP(hipMalloc(&dw, sizeof(double) * w.size()));
    hipError_t e = hipMemcpyAsync(dw, w.data(), sizeof(double) * w.size(), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) {
        const ResTile t = res_tile(nrow, ncol, 2 * r + 1);
        const long long nparts = ((long long)nrow + t.rows - 1) / t.rows * t.nchunk;
        const size_t shm = sizeof(double) * ((size_t)t.rows * t.stride + (std::min(2 * r + 1, kResTaps) + 1) / 2 * 2);
        res_corr_kernel<<<(int)std::min<long long>(nparts, 4096), kFluxThreads, shm, s>>>(in, out, nrow, ncol, dw,
                                                                                             2 * r + 1, t, nparts);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipFree(dw);
    if (e != hipSuccess) return fail(FSAMD_ERR_HIP, std::string("res_corr: ") + hipGetErrorString(e));
    return FSAMD_OK;
}

int fsamd_flux_power(const double *tau, int nlos, int npix, double scale, double mean_flux, double vmax,
                     double *power, void *stream)
{
    if (nlos < 1 || npix < 1 || !tau || !power || !(mean_flux != 0))
        return fail(FSAMD_ERR_ARG, "bad arguments to fsamd_flux_power");
    // a pair's row with the half table of roots beside it
    constexpr size_t kLdsBytes = 160 * 1024;
    if (sizeof(double) * 3 * (size_t)npix > kLdsBytes)
        return fail(FSAMD_ERR_UNSUPPORTED, "flux power: npix too large for the LDS buffers");
    hipStream_t s = (hipStream_t)stream;
    const int nk = npix / 2 + 1;
    const FftPlan fp = fft_plan(npix);
    const size_t shm = sizeof(double2) * ((size_t)npix + (fp.any ? nk : FSAMD_EXP_N));
    const bool pow2 = npix % 8 == 0 && (npix & (npix - 1)) == 0;
    const auto kernel = fp.any ? flux_fft_kernel<kFftAny> : pow2 ? flux_fft_kernel<kFftPow2> : flux_fft_kernel<kFftSmall>;
    const int threads = ((npix + kFftPoints - 1) / kFftPoints + 63) / 64 * 64;
    if (int rc = raise_lds_limit((const void *)kernel, shm)) return rc;
    int dev = 0, ncu = 0, percu = 0;
    FSAMD_HIP(hipGetDevice(&dev));
    FSAMD_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    FSAMD_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&percu, kernel, threads, shm));
    const int nblk = std::min((nlos + 1) / 2, std::max(1, percu) * ncu);
    double *part = nullptr;
    FSAMD_HIP(hipMalloc(&part, sizeof(double) * (size_t)nblk * nk + sizeof(double2) * (size_t)npix));
    double2 *tw = reinterpret_cast<double2 *>(part + ((size_t)nblk * nk + 1) / 2 * 2);
    fft_twiddle_kernel<<<(npix + 255) / 256, 256, 0, s>>>(tw, fp);
    kernel<<<nblk, threads, shm, s>>>(tau, nlos, npix, scale, 1.0 / mean_flux, tw, fp, part);
    // mean over sightlines of vmax |F_k|^2 / npix^2 (fluxstatistics.py:49-56, 95-102)
    const double norm = vmax / ((double)npix * (double)npix) / nlos;
    column_sum_kernel<<<(nk + kSumCols - 1) / kSumCols, kFluxThreads, 0, s>>>(part, nblk, nk, norm, power);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipFree(part);
    if (e != hipSuccess) return fail(FSAMD_ERR_HIP, std::string("flux power: ") + hipGetErrorString(e));
    return FSAMD_OK;
}

int fsamd_flux_hist(const double *tau, long long n, double scale, int nbins, unsigned long long *counts,
                    void *stream)
{
    if (n < 0 || nbins < 1 || !counts || (n > 0 && !tau)) return fail(FSAMD_ERR_ARG, "bad arguments to fsamd_flux_hist");
    hipStream_t s = (hipStream_t)stream;
    FSAMD_HIP(hipMemsetAsync(counts, 0, sizeof(unsigned long long) * nbins, s));
    if (n > 0) {
        constexpr size_t kLdsBytes = 160 * 1024, kTabBytes = sizeof(double2) * FSAMD_EXP_N;
        size_t shm = sizeof(unsigned int) * (size_t)nbins;
        if (shm > kLdsBytes) return fail(FSAMD_ERR_UNSUPPORTED, "flux histogram: too many bins for the LDS");
        const int nblocks = (int)std::min<long long>(1024, (n + kFluxThreads - 1) / kFluxThreads);
        // no more counts than a block has pixels: they are cleared and added up
        const long long room = std::min<long long>(kHistCounts, n / nblocks);
        int copies = 1;
        while (copies < kFluxThreads && 2LL * copies * nbins <= room) copies *= 2;
        const bool table = shm + kTabBytes <= kLdsBytes;
        shm = shm * copies + (table ? kTabBytes : 0);
        const auto kernel = table ? flux_hist_kernel<true> : flux_hist_kernel<false>;
        if (int rc = raise_lds_limit((const void *)kernel, shm)) return rc;
        kernel<<<nblocks, kFluxThreads, shm, s>>>(tau, n, scale, nbins, copies, counts);
        FSAMD_HIP(hipGetLastError());
    }
    FSAMD_HIP(hipStreamSynchronize(s));
    return FSAMD_OK;
}

}  // extern "C"

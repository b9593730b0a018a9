// Sightline <-> particle binning on the GPU.
//
// The reference (IndexTable, fake_spectra/index_table.cpp:7-150) sorts
// sightlines into two std::multimaps keyed by one transverse coordinate,
// range-queries them per particle, and inserts every accepted
// (sightline, particle, dr2) into per-sightline std::maps under an OpenMP
// critical section.  Here:
//   1. sightlines are bucketed into one square grid per axis over their two
//      transverse coordinates (a superset search structure only);
//   2. one thread per particle visits the grid cells its support touches and
//      applies the reference's acceptance test exactly (float key window with
//      periodic wrap, float second-coordinate window, FP64 minimum-image dr2
//      compared with the float product h*h), counting then emitting pairs
//      into a particle-major list at offsets from an exclusive scan;
//   3. a stable LSD radix sort on the sightline id (LDS digit histograms,
//      LDS prefix scans, wave-ballot ranking) turns it into per-sightline
//      rows in ascending particle order, the std::map order of the reference.
// All arithmetic that decides membership is compiled without FP contraction.
#include "fsamd_internal.h"
#include "plan.h"

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <numeric>
#include <vector>

namespace fsamd {

// ---------------------------------------------------------------------------
// Small utilities

__global__ void fill_i32_kernel(int *p, int v, long long n)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ void fill_f64_kernel(double *p, double v, long long n)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}

static int grid_for(long long n, int threads, int cap = 65536)
{
    long long b = (n + threads - 1) / threads;
    if (b < 1) b = 1;
    if (b > cap) b = cap;
    return (int)b;
}

int launch_fill_i32(int *p, int value, long long n, hipStream_t s)
{
    if (n <= 0) return FSAMD_OK;
    fill_i32_kernel<<<grid_for(n, 256), 256, 0, s>>>(p, value, n);
    FSAMD_HIP(hipGetLastError());
    return FSAMD_OK;
}

int launch_fill_f64(double *p, double value, long long n, hipStream_t s)
{
    if (n <= 0) return FSAMD_OK;
    fill_f64_kernel<<<grid_for(n, 256), 256, 0, s>>>(p, value, n);
    FSAMD_HIP(hipGetLastError());
    return FSAMD_OK;
}

__global__ void pack_records_kernel(const float *pos, const float *vel, const float *temp, const float *h,
                                    const LineDesc *lines, int nlines, long long n, PartRec *out)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += stride) {
        float4 a, b, d0, d1;
        a.x = pos[3 * i];
        a.y = pos[3 * i + 1];
        a.z = pos[3 * i + 2];
        a.w = h[i];
        b.x = vel[3 * i];
        b.y = vel[3 * i + 1];
        b.z = vel[3 * i + 2];
        b.w = temp[i];
        float d[kMaxLines];
#pragma unroll
        for (int k = 0; k < kMaxLines; ++k) d[k] = k < nlines ? lines[k].dens[i] : 0.0f;
        d0 = make_float4(d[0], d[1], d[2], d[3]);
        d1 = make_float4(d[4], d[5], d[6], d[7]);
        float4 *o = (float4 *)&out[i];
        o[0] = a;
        o[1] = b;
        o[2] = d0;
        o[3] = d1;
    }
}

int launch_pack_records(const float *pos, const float *vel, const float *temp, const float *h,
                        const LineDesc *lines, int nlines, long long n, PartRec *out, hipStream_t s)
{
    if (n <= 0) return FSAMD_OK;
    pack_records_kernel<<<grid_for(n, 256, 1 << 16), 256, 0, s>>>(pos, vel, temp, h, lines, nlines, n, out);
    FSAMD_HIP(hipGetLastError());
    return FSAMD_OK;
}

// ---------------------------------------------------------------------------
// Device-wide exclusive scan (tile reduce -> scan of tile sums -> apply).

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ inline long long wave_incl_scan(long long v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        long long t = __shfl_up(v, d, 64);
        if (lane >= d) v += t;
    }
    return v;
}

// Exclusive scan over the 256 threads of a block; *total gets the block sum.
__device__ inline long long block_excl_scan(long long v, long long *lds4, long long *total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long long inc = wave_incl_scan(v);
    if (lane == 63) lds4[w] = inc;
    __syncthreads();
    long long off = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < kScanThreads / 64; ++i) {
        if (i < w) off += lds4[i];
        tot += lds4[i];
    }
    __syncthreads();
    *total = tot;
    return off + inc - v;
}

template <typename T>
__global__ void scan_reduce_kernel(const T *in, long long n, long long *sums)
{
    __shared__ long long lds4[kScanThreads / 64];
    const long long base = (long long)blockIdx.x * kScanTile + (long long)threadIdx.x * kScanItems;
    long long s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i)
        if (base + i < n) s += (long long)in[base + i];
    long long tot;
    block_excl_scan(s, lds4, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

// out[i] = the tile's offset + exclusive prefix within the tile; out may alias
// in.  kSums: tile_off holds the tiles' sums as scan_reduce_kernel left them, at
// most kScanThreads of them, which each block adds up itself.  kEnd: out[n] = total.
template <typename T, bool kSums, bool kEnd>
__global__ void scan_apply_kernel(const T *in, long long *out, long long n, const long long *tile_off)
{
    __shared__ long long lds4[kScanThreads / 64];
    long long first = 0;
    if (kSums)
        block_excl_scan(threadIdx.x < blockIdx.x ? tile_off[threadIdx.x] : 0, lds4, &first);
    else if (tile_off)
        first = tile_off[blockIdx.x];
    const long long base = (long long)blockIdx.x * kScanTile + (long long)threadIdx.x * kScanItems;
    long long v[kScanItems];
    long long s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        v[i] = (base + i < n) ? (long long)in[base + i] : 0;
        s += v[i];
    }
    long long tot;
    long long off = block_excl_scan(s, lds4, &tot) + first;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        if (base + i < n) out[base + i] = off;
        off += v[i];
    }
    if (kEnd && base < n && base + kScanItems >= n) out[n] = off;
}

size_t exclusive_scan_ws_bytes(long long n)
{
    // every level holds ceil(n/tile)+1 tile sums and recurses on that many
    size_t total = 0;
    n += 1;
    while (n > kScanTile) {
        long long nt = (n + kScanTile - 1) / kScanTile + 1;
        total += sizeof(long long) * (size_t)nt;
        n = nt;
    }
    return total + 256;
}

// In-place exclusive scan of int64 data[0..n); ws from exclusive_scan_ws_bytes.
static int scan_i64_rec(long long *data, long long n, char *ws, size_t ws_bytes, hipStream_t s)
{
    if (n <= 0) return FSAMD_OK;
    long long nt = (n + kScanTile - 1) / kScanTile;
    if (nt == 1) {
        scan_apply_kernel<long long, false, false><<<1, kScanThreads, 0, s>>>(data, data, n, nullptr);
        FSAMD_HIP(hipGetLastError());
        return FSAMD_OK;
    }
    size_t need = sizeof(long long) * (size_t)(nt + 1);
    if (need > ws_bytes) return fail(FSAMD_ERR_ARG, "scan workspace too small");
    long long *sums = (long long *)ws;
    scan_reduce_kernel<long long><<<(int)nt, kScanThreads, 0, s>>>(data, n, sums);
    FSAMD_HIP(hipGetLastError());
    if (nt <= kScanThreads) {
        scan_apply_kernel<long long, true, false><<<(int)nt, kScanThreads, 0, s>>>(data, data, n, sums);
        FSAMD_HIP(hipGetLastError());
        return FSAMD_OK;
    }
    int rc = scan_i64_rec(sums, nt, ws + need, ws_bytes - need, s);
    if (rc) return rc;
    scan_apply_kernel<long long, false, false><<<(int)nt, kScanThreads, 0, s>>>(data, data, n, sums);
    FSAMD_HIP(hipGetLastError());
    return FSAMD_OK;
}

int exclusive_scan_i64_inplace(long long *data, long long n, void *ws, size_t ws_bytes, hipStream_t s)
{
    return scan_i64_rec(data, n, (char *)ws, ws_bytes, s);
}

// out[0..n] = exclusive scan of int32 in[0..n), out[n] = total.
int exclusive_scan_i32_to_i64(const int *in, long long *out, long long n, void *ws, size_t ws_bytes,
                              hipStream_t s)
{
    long long nt = (n + kScanTile - 1) / kScanTile;
    if (n <= 0) {
        FSAMD_HIP(hipMemsetAsync(out, 0, sizeof(long long), s));
        return FSAMD_OK;
    }
    size_t need = sizeof(long long) * (size_t)(nt + 1);
    if (need > ws_bytes) return fail(FSAMD_ERR_ARG, "scan workspace too small");
    long long *sums = (long long *)ws;
    if (nt > 1) {
        scan_reduce_kernel<int><<<(int)nt, kScanThreads, 0, s>>>(in, n, sums);
        FSAMD_HIP(hipGetLastError());
    }
    // up to 256 tiles (half a million entries): no scan of the sums between, two
    // launches in place of three, a memset and a copy (4 to 5 us each to the host)
    if (nt == 1) {
        scan_apply_kernel<int, false, true><<<1, kScanThreads, 0, s>>>(in, out, n, nullptr);
    } else if (nt <= kScanThreads) {
        scan_apply_kernel<int, true, true><<<(int)nt, kScanThreads, 0, s>>>(in, out, n, sums);
    } else {
        if (int rc = scan_i64_rec(sums, nt, (char *)ws + need, ws_bytes - need, s)) return rc;
        scan_apply_kernel<int, false, true><<<(int)nt, kScanThreads, 0, s>>>(in, out, n, sums);
    }
    FSAMD_HIP(hipGetLastError());
    return FSAMD_OK;
}

// ---------------------------------------------------------------------------
// Sightline grid

// Plane coordinates of a sightline: (key, second) as compared by the reference.
__device__ inline void los_plane(int ax, const double *c, double &k1, double &k2)
{
    if (ax == 1) {
        k1 = c[1];
        k2 = c[2];
    } else if (ax == 2) {
        k1 = c[0];
        k2 = c[2];
    } else {
        k1 = c[0];
        k2 = c[1];
    }
}

__device__ inline int wrap_cell(double k, double box, double inv_cw, int nc)
{
    double kw = k - floor(k / box) * box;
    int c = (int)floor(kw * inv_cw);
    return c < 0 ? 0 : (c >= nc ? nc - 1 : c);
}

// Sightlines of each axis.  Counted per block in LDS: one global atomic per
// sightline serializes on three addresses (150528 sightlines: 1.71 ms).
constexpr int kAxisBlocks = 64;

__global__ __launch_bounds__(256) void los_axis_count_kernel(const int *axis, int nlos, int *counts3)
{
    __shared__ int c[3];
    if (threadIdx.x < 3) c[threadIdx.x] = 0;
    __syncthreads();
    int n[3] = {0, 0, 0};
    for (int i = blockIdx.x * 256 + threadIdx.x; i < nlos; i += gridDim.x * 256) {
        const int a = axis[i];
#pragma unroll
        for (int k = 0; k < 3; ++k) n[k] += a == k + 1;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) n[k] += __shfl_xor(n[k], o, 64);
        if ((threadIdx.x & 63) == 0 && n[k]) atomicAdd(&c[k], n[k]);
    }
    __syncthreads();
    if (threadIdx.x < 3 && c[threadIdx.x]) atomicAdd(&counts3[threadIdx.x], c[threadIdx.x]);
}

// The grid cell of a sightline and its plane coordinates; -1 for one with
// non-finite coordinates, which never passes the reference's tests.
__device__ inline int los_cell(int a, const double *c, double box, const LosGrid &g, double &k1, double &k2)
{
    los_plane(a, c, k1, k2);
    if (a < 1 || a > 3 || !isfinite(k1) || !isfinite(k2)) return -1;
    const int ai = a - 1;
    const int c1 = wrap_cell(k1, box, g.inv_cw[ai], g.nc[ai]);
    const int c2 = wrap_cell(k2, box, g.inv_cw[ai], g.nc[ai]);
    return g.base[ai] + c2 * g.nc[ai] + c1;
}

// The whole grid of few sightlines by one block: counts, their scan and the
// cursors in LDS.
//
// Bound: the latency of one block's passes, 4 us for 64 sightlines and 41 us for
// 12288; the ten launches and copies in its place take about 50 us whatever the
// number, so the line lies where it still halves that.  A drop-in call on 32768
// particles and 64 sightlines: 818 -> 740 us.
constexpr int kGridThreads = 1024;
constexpr int kGridSmallCells = 8 * 1024;   // 32 KB

__global__ __launch_bounds__(kGridThreads) void grid_small_kernel(const int *axis, const double *cofm, int nlos,
                                                                  double box, LosGrid g, int ncells, int *cell_start,
                                                                  int *cell_ids, double2 *cell_kl)
{
    extern __shared__ int cursor[];   // [ncells]
    __shared__ int wsum[kGridThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int c = threadIdx.x; c < ncells; c += kGridThreads) cursor[c] = 0;
    __syncthreads();
    double k1, k2;
    for (int i = threadIdx.x; i < nlos; i += kGridThreads) {
        const int cell = los_cell(axis[i], &cofm[3 * (size_t)i], box, g, k1, k2);
        if (cell >= 0) atomicAdd(&cursor[cell], 1);
    }
    __syncthreads();
    // exclusive scan: a run of cells a thread
    const int per = (ncells + kGridThreads - 1) / kGridThreads;
    const int lo = min((int)threadIdx.x * per, ncells), hi = min(lo + per, ncells);
    int own = 0;
    for (int c = lo; c < hi; ++c) own += cursor[c];
    int incl = own;
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o, 64);
        if (lane >= o) incl += v;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int at = incl - own;
    for (int w = 0; w < wave; ++w) at += wsum[w];
    for (int c = lo; c < hi; ++c) {
        const int n = cursor[c];
        cursor[c] = at;
        cell_start[c] = at;
        at += n;
    }
    if (threadIdx.x == kGridThreads - 1) cell_start[ncells] = at;
    __syncthreads();
    for (int i = threadIdx.x; i < nlos; i += kGridThreads) {
        const int cell = los_cell(axis[i], &cofm[3 * (size_t)i], box, g, k1, k2);
        if (cell < 0) continue;
        const int to = atomicAdd(&cursor[cell], 1);
        cell_ids[to] = i;
        cell_kl[to] = make_double2(k1, k2);
    }
}

// The plan's copies of few sightlines and their number on each axis, by one
// block (2 us for 64) in place of two copies, a memset and los_axis_count_kernel,
// 4 to 5 us each to the host.
constexpr int kIntakeMax = kGridSmallCells;

__global__ __launch_bounds__(kGridThreads) void los_intake_kernel(const int *axis, const double *cofm, int nlos,
                                                                  int *axis_out, double *cofm_out, int *counts3)
{
    __shared__ int c[3];
    if (threadIdx.x < 3) c[threadIdx.x] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < nlos; i += kGridThreads) {
        const int a = axis[i];
        axis_out[i] = a;
        if (a >= 1 && a <= 3) atomicAdd(&c[a - 1], 1);
    }
    for (int i = threadIdx.x; i < 3 * nlos; i += kGridThreads) cofm_out[i] = cofm[i];
    __syncthreads();
    if (threadIdx.x < 3) counts3[threadIdx.x] = c[threadIdx.x];
}

__global__ void los_cell_kernel(const int *axis, const double *cofm, int nlos, double box, LosGrid g,
                                int *cell_of, int *cell_count)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nlos) return;
    double k1, k2;
    const int cell = los_cell(axis[i], &cofm[3 * (size_t)i], box, g, k1, k2);
    cell_of[i] = cell;
    if (cell >= 0) atomicAdd(&cell_count[cell], 1);
}

__global__ void los_scatter_kernel(const int *axis, const double *cofm, int nlos, const int *cell_of,
                                   int *cursor, int *cell_ids, double2 *cell_kl)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nlos) return;
    int cell = cell_of[i];
    if (cell < 0) return;
    int at = atomicAdd(&cursor[cell], 1);
    double k1, k2;
    los_plane(axis[i], &cofm[3 * (size_t)i], k1, k2);
    cell_ids[at] = i;
    cell_kl[at] = make_double2(k1, k2);
}

__global__ void i64_to_i32_kernel(const long long *in, int *out, long long n)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        out[i] = (int)in[i];
}

// ---------------------------------------------------------------------------
// The reference acceptance test (index_table.cpp:22-113), exact.
//   first/second: the particle's float coordinates along the sightline's key
//   and second axes; key/lproj2: the sightline's coordinates; hh: float h.
__device__ inline bool los_accept(float first, float second, float hh, double key, double lproj2,
                                  double box, double &dr2)
{
    // get_nearby: half-open key window [ffm, ffp) with periodic wrap (93-112)
    float ffp = first + hh;
    if ((double)ffp > box) ffp = (float)((double)ffp - box);
    float ffm = first - hh;
    if (ffm < 0) ffm = (float)((double)ffm + box);
    const bool inwin = (ffm <= ffp) ? (key >= (double)ffm && key < (double)ffp)
                                    : (key < (double)ffp || key >= (double)ffm);
    if (!inwin) return false;
    // second_close (52-68)
    bool close = false;
    float sp = second + hh;
    if ((double)sp > box && lproj2 < (double)sp - box) close = true;
    float sm = second - hh;
    if (!close && sm < 0 && lproj2 > (double)sm + box) close = true;
    if (!close && lproj2 > (double)sm && lproj2 < (double)sp) close = true;
    if (!close) return false;
    // calc_dr2 (70-87) and the acceptance dr2 <= hh*hh with a float product (45)
    double dr = fabs((double)first - key);
    if (dr > 0.5 * box) dr = box - dr;
    double d2 = dr * dr;
    dr = fabs((double)second - lproj2);
    if (dr > 0.5 * box) dr = box - dr;
    d2 += dr * dr;
    dr2 = d2;
    const float hh2 = hh * hh;
    return d2 <= (double)hh2;
}

// Particle coordinates (first, second) for a sightline axis (index_table.cpp:33-40, 117-127).
__device__ inline void particle_plane(int ax, const float *p, float &first, float &second)
{
    if (ax == 1) {
        first = p[1];
        second = p[2];
    } else if (ax == 2) {
        first = p[0];
        second = p[2];
    } else {
        first = p[0];
        second = p[1];
    }
}

// The cells (of nc, periodic) within hr of x: n of them from lo on, 0 <= lo < nc;
// all of them from 0 if the window is as wide as the box.  False if none can
// hold a sightline within hr: x is a NaN, or so many boxes away that no
// distance the reference forms is below the support.
__device__ inline bool cell_window(double x, double hr, double inv, int nc, int &lo, int &n)
{
    const double a = floor((x - hr) * inv), width = floor((x + hr) * inv) - a + 1.0;
    if (width >= (double)nc) {
        lo = 0;
        n = nc;
        return true;
    }
    if (!(fabs(a) < 1e9)) return false;
    lo = (int)a;
    n = (int)width;
    if (lo < 0) lo += nc;
    if (lo < 0 || lo >= nc) lo = (lo % nc + nc) % nc;
    return true;
}

// Supports that reach no sightline: no number, or infinite (los_accept, like the
// reference's windows, is empty or undefined for them).
__device__ inline bool finite_support(float hh) { return __builtin_fabsf(hh) < __builtin_inff(); }

// Visit every sightline accepted for particle p; f(sightline, dr2) returns
// false to stop the visit early.
//
// Bound: divergence (a wavefront goes through the longest of its lanes' rows and
// runs; a quarter of the lanes are active).  Runs of a row's cells in place of
// cell by cell, windows in 32-bit integers: 512^3 particles, 8000 sightlines, count
// and emit 11.0 and 12.5 -> 8.1 and 9.1 ms.  The grid in LDS (11.1 and 14.4 with
// a preselection in FP32) and cells four times as narrow along a row (7.0 and
// 8.7, but bin_any_kernel 763 -> 861 us) did not pay.
template <class F>
__device__ inline void visit_accepted(const BinArgs &A, const float *p, float hh, F &&f)
{
    if (!finite_support(hh)) return;
    const double ah = fabs((double)hh);
    for (int ai = 0; ai < 3; ++ai) {
        if (A.grid.nlos_axis[ai] == 0) continue;
        const int ax = ai + 1;
        float first, second;
        particle_plane(ax, p, first, second);
        const int nc = A.grid.nc[ai];
        const double inv = A.grid.inv_cw[ai];
        const double hr = ah * (1.0 + 1e-5) + 1e-3 * A.grid.cw[ai];
        int lo1, n1, lo2, n2;
        if (!cell_window((double)first, hr, inv, nc, lo1, n1) || !cell_window((double)second, hr, inv, nc, lo2, n2))
            continue;
        // a row's cells follow each other: one run of sightlines, two where it wraps
        const int over = max(lo1 + n1 - nc, 0);
        for (int r = 0; r < n2; ++r) {
            const int w2 = lo2 + r < nc ? lo2 + r : lo2 + r - nc;
            const int *row = A.grid.cell_start + A.grid.base[ai] + w2 * nc;
            int k = row[lo1], e = row[lo1 + n1 - over];
            for (int part = 0;; ++part) {
                for (; k < e; ++k) {
                    const double2 kl = A.grid.cell_kl[k];
                    double dr2;
                    if (los_accept(first, second, hh, kl.x, kl.y, A.box, dr2) && !f(A.grid.cell_ids[k], dr2))
                        return;
                }
                if (part || over == 0) break;
                k = row[0];
                e = row[over];
            }
        }
    }
}

__global__ void bin_count_kernel(BinArgs A, int *cnt)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < A.npart;
         i += (long long)gridDim.x * blockDim.x) {
        const float p[3] = {A.pos[3 * i], A.pos[3 * i + 1], A.pos[3 * i + 2]};
        int c = 0;
        visit_accepted(A, p, A.h[i], [&](int, double) {
            ++c;
            return true;
        });
        cnt[i] = c;
    }
}

__global__ void bin_emit_kernel(BinArgs A, const long long *poff, int *keys, int *vals)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < A.npart;
         i += (long long)gridDim.x * blockDim.x) {
        const float p[3] = {A.pos[3 * i], A.pos[3 * i + 1], A.pos[3 * i + 2]};
        long long at = poff[i];
        visit_accepted(A, p, A.h[i], [&](int s, double) {
            keys[at] = s;
            vals[at] = (int)i;
            ++at;
            return true;
        });
    }
}

// Whether one of the sightlines of the cell that holds the particle's own
// point of the plane accepts it, on any axis.
// (An infinite support is accepted here: finite_support, asked after this in the
// kernel, costs nothing, and 2.5% of the call where a cell's reads wait for it.)
__device__ inline bool own_cell_accepts(const BinArgs &A, const float *p, float hh)
{
    for (int ai = 0; ai < 3; ++ai) {
        if (A.grid.nlos_axis[ai] == 0) continue;
        float first, second;
        particle_plane(ai + 1, p, first, second);
        const int nc = A.grid.nc[ai];
        const double c1 = floor((double)first * A.grid.inv_cw[ai]), c2 = floor((double)second * A.grid.inv_cw[ai]);
        if (!(c1 >= 0 && c1 < nc && c2 >= 0 && c2 < nc)) continue;   // outside the box: the full visit decides
        const int cell = A.grid.base[ai] + (int)c2 * nc + (int)c1;
        const int e = A.grid.cell_start[cell + 1];
        for (int k = A.grid.cell_start[cell]; k < e; ++k) {
            const double2 kl = A.grid.cell_kl[k];
            double dr2;
            if (los_accept(first, second, hh, kl.x, kl.y, A.box, dr2)) return true;
        }
    }
    return false;
}

// Bit i of mask[w] = 1 if particle 64 w + i reaches at least one sightline
// (the _near_lines test, py_module.cpp:58-76), cnt[w] its number of bits.
//
// Bound: the latency of the dependent reads (cell start, then its entries) of
// the cells a support touches, not the 16 bytes a particle.  Where sightlines
// are dense most particles are accepted by one next to them, while a visit
// begins at a corner of the support's square, out of the circle's reach: a
// particle's own cell is tried first, and the block's particles that it does
// not settle (some of nearly every wavefront) are then visited packed
// together.  16.8M particles, 150528 gridded sightlines: 1565 us a visit
// each, 1379 us with the own cell first, 1042 us packed, 763 us with runs of cells.
constexpr int kAnyWords = 32;            // mask words (64 particles each) of a block

__global__ __launch_bounds__(256) void bin_any_kernel(BinArgs A, unsigned long long *mask, int *cnt)
{
    __shared__ unsigned long long bits[kAnyWords];
    __shared__ unsigned short queue[kAnyWords * 64];
    __shared__ int nq;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long nw = (A.npart + 63) / 64;
    for (long long w0 = blockIdx.x * (long long)kAnyWords; w0 < nw; w0 += (long long)gridDim.x * kAnyWords) {
        if (threadIdx.x == 0) nq = 0;
        __syncthreads();
        for (int k = wave; k < kAnyWords; k += 4) {
            const long long i = (w0 + k) * 64 + lane;
            const bool have = i < A.npart;
            bool any = false;
            if (have) {
                const float p[3] = {A.pos[3 * i], A.pos[3 * i + 1], A.pos[3 * i + 2]};
                const float hh = A.h[i];
                any = own_cell_accepts(A, p, hh) && finite_support(hh);
            }
            const unsigned long long m = __ballot(any), open = __ballot(have && !any);
            int at = 0;
            if (lane == 0) {
                bits[k] = m;
                if (open) at = atomicAdd(&nq, __popcll(open));
            }
            at = __shfl(at, 0, 64);
            if ((open >> lane) & 1ull)
                queue[at + __popcll(open & ((1ull << lane) - 1ull))] = (unsigned short)(k * 64 + lane);
        }
        __syncthreads();
        const int n = nq;
        for (int q = threadIdx.x; q < n; q += 256) {
            const int l = queue[q];
            const long long i = w0 * 64 + l;
            const float p[3] = {A.pos[3 * i], A.pos[3 * i + 1], A.pos[3 * i + 2]};
            bool any = false;
            visit_accepted(A, p, A.h[i], [&](int, double) {
                any = true;
                return false;
            });
            if (any) atomicOr(&bits[l >> 6], 1ull << (l & 63));
        }
        __syncthreads();
        if (threadIdx.x < kAnyWords && w0 + threadIdx.x < nw) {
            mask[w0 + threadIdx.x] = bits[threadIdx.x];
            cnt[w0 + threadIdx.x] = __popcll(bits[threadIdx.x]);
        }
        __syncthreads();
    }
}

// Ids of the set bits, word w's at off[w].
__global__ __launch_bounds__(256) void mask_scatter_kernel(const unsigned long long *mask, const long long *off,
                                                           long long nw, int *out)
{
    const int lane = threadIdx.x & 63;
    const long long step = (long long)gridDim.x * 4;
    for (long long w = blockIdx.x * 4ll + (threadIdx.x >> 6); w < nw; w += step) {
        const unsigned long long m = mask[w];
        if ((m >> lane) & 1ull) out[off[w] + __popcll(m & ((1ull << lane) - 1ull))] = (int)(w * 64 + lane);
    }
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort of (key, value) int32 pairs by key digits.

constexpr int kRsThreads = 256;
constexpr int kRsItems = 16;
constexpr long long kRsTile = (long long)kRsThreads * kRsItems;
constexpr int kRsMaxBits = 8;
constexpr int kRsWaves = kRsThreads / 64;

__global__ void rs_upsweep_kernel(const int *keys, long long n, int shift, int bits, long long ntiles,
                                  long long *table)
{
    __shared__ int hist[1 << kRsMaxBits];
    const int nb = 1 << bits;
    for (int d = threadIdx.x; d < nb; d += kRsThreads) hist[d] = 0;
    __syncthreads();
    const long long base = blockIdx.x * kRsTile;
    const unsigned mask = (unsigned)nb - 1;
    for (int r = 0; r < kRsItems; ++r) {
        const long long e = base + r * kRsThreads + threadIdx.x;
        if (e < n) atomicAdd(&hist[((unsigned)keys[e] >> shift) & mask], 1);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < nb; d += kRsThreads) table[(long long)d * ntiles + blockIdx.x] = hist[d];
}

// Bound: HBM, 8 bytes a pair in and out.  A wavefront ranks its quarter of the
// tile in registers against running counts of its own (no block barrier a
// round), the tile is put in order in LDS, and a digit's run leaves as whole
// lines; written pair by pair from the ranking rounds, three barriers each,
// 125M pairs took 1.96 ms a pass, this 0.63 (3.2 TB/s).
__global__ __launch_bounds__(kRsThreads) void rs_downsweep_kernel(const int *kin, const int *vin, int *kout, int *vout,
                                                                 long long n, int shift, int bits, long long ntiles,
                                                                 const long long *table)
{
    __shared__ long long base_off[1 << kRsMaxBits];
    __shared__ int start[1 << kRsMaxBits];             // of a digit in the ordered tile
    __shared__ int wcnt[kRsWaves][1 << kRsMaxBits];    // counts, then a wavefront's place in the tile
    __shared__ long long lds4[kScanThreads / 64];
    __shared__ int2 ordered[kRsTile];
    static_assert(kRsThreads == kScanThreads && (1 << kRsMaxBits) <= kRsThreads, "one digit a thread");
    const int nb = 1 << bits;
    const unsigned mask = (unsigned)nb - 1;
    for (int d = threadIdx.x; d < nb; d += kRsThreads) {
        base_off[d] = table[(long long)d * ntiles + blockIdx.x];
        for (int w = 0; w < kRsWaves; ++w) wcnt[w][d] = 0;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const long long tbase = blockIdx.x * kRsTile;
    const int count = (int)min((long long)kRsTile, n - tbase);
    const int first = wave * (int)(kRsTile / kRsWaves) + lane;
    int k[kRsItems], v[kRsItems], pos[kRsItems];
#pragma unroll
    for (int r = 0; r < kRsItems; ++r) {
        const int e = first + r * 64;
        k[r] = e < count ? kin[tbase + e] : 0;
        v[r] = e < count ? vin[tbase + e] : 0;
    }
#pragma unroll
    for (int r = 0; r < kRsItems; ++r) {
        const bool valid = first + r * 64 < count;
        const unsigned d = ((unsigned)k[r] >> shift) & mask;
        unsigned long long peers = __ballot(valid);
        for (int b = 0; b < bits; ++b) {
            const bool bit = (d >> b) & 1u;
            const unsigned long long bb = __ballot(bit);
            peers &= bit ? bb : ~bb;
        }
        const int rank = __popcll(peers & lt);
        const int before = wcnt[wave][d];
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (valid && rank == 0) wcnt[wave][d] = before + __popcll(peers);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        pos[r] = before + rank;
    }
    __syncthreads();
    {
        const int d = threadIdx.x;
        int c[kRsWaves] = {}, sum = 0;
        if (d < nb)
            for (int w = 0; w < kRsWaves; ++w) sum += c[w] = wcnt[w][d];
        long long total;
        int at = (int)block_excl_scan(sum, lds4, &total);
        if (d < nb) {
            start[d] = at;
            for (int w = 0; w < kRsWaves; ++w) {
                wcnt[w][d] = at;
                at += c[w];
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRsItems; ++r)
        if (first + r * 64 < count)
            ordered[wcnt[wave][((unsigned)k[r] >> shift) & mask] + pos[r]] = make_int2(k[r], v[r]);
    __syncthreads();
    for (int i = threadIdx.x; i < count; i += kRsThreads) {
        const int2 kv = ordered[i];
        const unsigned d = ((unsigned)kv.x >> shift) & mask;
        const long long off = base_off[d] + (i - start[d]);
        kout[off] = kv.x;
        vout[off] = kv.y;
    }
}

// offsets[s] = first position of key >= s in the sorted keys (s = 0..nlos)
__global__ void row_offsets_kernel(const int *keys, long long n, int nlos, long long *offsets)
{
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s > nlos) return;
    long long lo = 0, hi = n;
    while (lo < hi) {
        long long mid = (lo + hi) >> 1;
        if (keys[mid] < s) lo = mid + 1;
        else hi = mid;
    }
    offsets[s] = lo;
}

__global__ void near_flag_kernel(const long long *poff, long long n, int *flag)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        flag[i] = poff[i + 1] > poff[i] ? 1 : 0;
}

__global__ void near_scatter_kernel(const long long *poff, const long long *fscan, long long n, int *out)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        if (poff[i + 1] > poff[i]) out[fscan[i]] = (int)i;
}

// ---------------------------------------------------------------------------
// Voronoi mesh (kernel 2): IndexTable::assign_cells (index_table.cpp:152-223).
// Each sightline is cut into npts = int(box/RESO) points at (i + 1/2) reso;
// point i goes to the nearest particle of the sightline's neighbour list
// (periodic distance, the first of the ascending row on ties), and a
// particle's segment runs from its first to its last point, +- reso/2.  The
// reference walks the points in order; here the same result comes from
// three parallel passes:
//   A: over the points past the middle of the box (xp > box/2 + reso/2), the
//      first one owned by the owner of point 0 (the periodic wrap, where the
//      reference restarts that particle's segment and stops the walk);
//   B: over the points before it, each particle's first and last point and
//      count (atomics);
//   C: per particle, the segment in FP32 with the reference's roundings; a
//      particle whose points are not contiguous marks the sightline in
//      error, where the reference exits (index_table.cpp:199-206).

struct VorArgs {
    double box, reso;
    int npts;                  // int(box / RESO)
    int imin;                  // first point with xp > box/2 + reso/2
    const float *pos;
    const int *axis;
    const double *cofm;
    const long long *line_off;
    const int *pair_part;
    int nlos;
    int *nn0;                  // [L] owner of point 0 (row index)
    int *istar;                // [L] first point >= imin owned by nn0; npts if none
    int *first, *last, *count; // [M] per pair
    int *err;                  // [L]
    float2 *seg;               // [M] segment ends
};

constexpr double kReso = 0.1;     // index_table.h:8
constexpr int kVorThreads = 256;
constexpr int kVorWaves = kVorThreads / 64;
constexpr int kVorStrips = 8;                              // strips of 64 points per wavefront
constexpr int kVorPts = kVorThreads * kVorStrips;          // points per block
constexpr int kVorCand = 512;                              // candidates held in LDS at a time

// Separation of one coordinate as the reference measures it (periodic box).
__device__ inline double vor_sep(double q, double p, double half, double box)
{
    double d = fabs(q - p);
    if (d > half) d = box - d;
    return d;
}

// A particle that may own one of a block's points: its coordinate along the
// sightline, its squared separations across it, and its row index.
struct VorCand {
    double x, y2, z2;
    int j, pad;
};

struct VorRow {
    int ax;
    double yp, zp, half;
    long long p0, n;
};

__device__ inline VorRow vor_row(const VorArgs &V, int s)
{
    VorRow R;
    R.ax = V.axis[s];
    const double *c = &V.cofm[3 * (size_t)s];
    R.yp = c[R.ax % 3];
    R.zp = c[(R.ax + 1) % 3];
    R.half = V.box / 2.;
    R.p0 = V.line_off[s];
    R.n = V.line_off[s + 1] - R.p0;
    return R;
}

__device__ inline VorCand vor_load(const VorArgs &V, const VorRow &R, long long j)
{
    const float *pp = &V.pos[3 * (size_t)V.pair_part[R.p0 + j]];
    const double dy = vor_sep((double)pp[R.ax % 3], R.yp, R.half, V.box);
    const double dz = vor_sep((double)pp[(R.ax + 1) % 3], R.zp, R.half, V.box);
    VorCand c;
    c.x = (double)pp[R.ax - 1];
    c.y2 = dy * dy;
    c.z2 = dz * dz;
    c.j = (int)j;
    c.pad = 0;
    return c;
}

__device__ inline double vor_d2(const VorArgs &V, const VorRow &R, const VorCand &c, double xp)
{
    const double dx = vor_sep(c.x, xp, R.half, V.box);
    return dx * dx + c.y2 + c.z2;
}

// Owner of each of the block's points i0 .. i0 + npt - 1 (npt <= kVorPts):
// owner[r] of point i0 + (wave * kVorStrips + r) * 64 + lane is the first
// particle of the ascending row at the smallest distance (the reference's
// scan, index_table.cpp:172-186), 0 if none is nearer than a box length.
//
// Bound: FP64 VALU.  Testing every particle of the row at every point costs
// points x row; but a distance changes by at most the distance moved along
// the sightline, so a particle farther from the middle of a stretch of points
// than the nearest one there plus the stretch's length owns none of them.
// The block drops those for its 2048 points (205 length units; some tens of
// a row of ~1000 remain), each wavefront again for its strips of 64 (one
// candidate per lane, 2-3 remain).  The candidates keep the row's order and
// the distances are the same expression, so ties fall as before.  64000
// particles, 200 sightlines of 200000 points (~850 particles a row): lists,
// cells and tau together 70.9 ms with every particle at every point, 1.36 ms so.
__device__ inline void vor_owners(const VorArgs &V, const VorRow &R, int i0, int npt, int (&owner)[kVorStrips])
{
    __shared__ VorCand cand[kVorCand];
    __shared__ double s_min[kVorWaves];
    __shared__ int s_cnt[kVorWaves];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const double slack = 1e-9 * V.box;       // far above the rounding of the distances
    const double xc = (i0 + 0.5 * npt) * V.reso, len = npt * V.reso;
    double dmin = 1e300;
    for (long long j = threadIdx.x; j < R.n; j += kVorThreads) {
        const double d2 = vor_d2(V, R, vor_load(V, R, j), xc);
        if (d2 < dmin) dmin = d2;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) dmin = fmin(dmin, __shfl_xor(dmin, o, 64));
    if (lane == 0) s_min[wave] = dmin;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kVorWaves; ++w) dmin = fmin(dmin, s_min[w]);
    const double thr = sqrt(dmin) + len + slack;
    const double thr2 = thr * thr * (1.0 + 1e-12);
    double best[kVorStrips], best2[kVorStrips];
#pragma unroll
    for (int r = 0; r < kVorStrips; ++r) {
        best[r] = V.box;
        best2[r] = V.box * V.box;
        owner[r] = 0;
    }
    int held = 0;
    for (long long t0 = 0; t0 < R.n; t0 += kVorThreads) {
        const long long j = t0 + threadIdx.x;
        VorCand c;
        bool in = false;
        if (j < R.n) {
            c = vor_load(V, R, j);
            in = !(vor_d2(V, R, c, xc) > thr2);
        }
        const unsigned long long m = __ballot(in);
        if (lane == 0) s_cnt[wave] = __popcll(m);
        __syncthreads();
        int at = held;
#pragma unroll
        for (int w = 0; w < kVorWaves; ++w) {
            if (w < wave) at += s_cnt[w];
            held += s_cnt[w];
        }
        if (in) cand[at + __popcll(m & ((1ull << lane) - 1ull))] = c;
        __syncthreads();
        if (held + kVorThreads <= kVorCand && t0 + kVorThreads < R.n) continue;
        for (int c0 = 0; c0 < held; c0 += 64) {
            const bool have = c0 + lane < held;
            const VorCand mine = cand[have ? c0 + lane : c0];
#pragma unroll
            for (int r = 0; r < kVorStrips; ++r) {
                const int f = (wave * kVorStrips + r) * 64;
                if (f >= npt) break;
                // the nearest of these 64 candidates and of the earlier ones
                // (whose best is at least as near at some point of the strip)
                const double xs = (i0 + f + 32) * V.reso;
                const double ds2 = have ? vor_d2(V, R, mine, xs) : 1e300;
                double lo = ds2;
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) lo = fmin(lo, __shfl_xor(lo, o, 64));
                const double ts = sqrt(lo) + 64 * V.reso + slack;
                unsigned long long todo = __ballot(have && !(ds2 > ts * ts * (1.0 + 1e-12)));
                const double xp = (i0 + f + lane + 0.5) * V.reso;
                while (todo) {
                    const int q = __builtin_ctzll(todo);
                    todo &= todo - 1;
                    const VorCand k = cand[c0 + q];
                    const double d2 = vor_d2(V, R, k, xp);
                    // sqrt is monotonic: only a smaller d2 can give a smaller distance
                    if (d2 < best2[r]) {
                        const double d = sqrt(d2);
                        if (d < best[r]) {
                            best[r] = d;
                            best2[r] = d2;
                            owner[r] = k.j;
                        }
                    }
                }
            }
        }
        held = 0;
        __syncthreads();
    }
}

// Owner of point 0 of each sightline (one block per sightline): the first
// particle of the row at the smallest distance, the threads over the row.
__global__ __launch_bounds__(kVorThreads) void vor_first_kernel(VorArgs V)
{
    __shared__ double s_d[kVorWaves];
    __shared__ int s_j[kVorWaves];
    const int s = blockIdx.x;
    if (V.line_off[s + 1] == V.line_off[s]) {
        if (threadIdx.x == 0) V.nn0[s] = -1;
        return;
    }
    const VorRow R = vor_row(V, s);
    double best = V.box;
    int bi = 0x7fffffff;
    for (long long j = threadIdx.x; j < R.n; j += kVorThreads) {
        const double d = sqrt(vor_d2(V, R, vor_load(V, R, j), 0.5 * V.reso));
        if (d < best) {
            best = d;
            bi = (int)j;
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double d = __shfl_xor(best, o, 64);
        const int j = __shfl_xor(bi, o, 64);
        if (d < best || (d == best && j < bi)) {
            best = d;
            bi = j;
        }
    }
    if (lane == 0) {
        s_d[wave] = best;
        s_j[wave] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kVorWaves; ++w)
            if (s_d[w] < best || (s_d[w] == best && s_j[w] < bi)) {
                best = s_d[w];
                bi = s_j[w];
            }
        V.nn0[s] = bi == 0x7fffffff ? 0 : bi;   // none nearer than a box length: the first of the row
        V.istar[s] = V.npts;
    }
}

// Pass A: blocks over (chunk of points from imin, sightline).
__global__ __launch_bounds__(kVorThreads) void vor_wrap_kernel(VorArgs V)
{
    __shared__ int s_skip;
    const int s = blockIdx.y;
    const int i0 = V.imin + blockIdx.x * kVorPts;
    if (V.nn0[s] < 0 || i0 >= V.npts) return;
    // an earlier point already wraps: read once for the whole block
    if (threadIdx.x == 0) s_skip = __atomic_load_n(&V.istar[s], __ATOMIC_RELAXED) < i0;
    __syncthreads();
    if (s_skip) return;
    const int npt = min(kVorPts, V.npts - i0);
    int owner[kVorStrips];
    vor_owners(V, vor_row(V, s), i0, npt, owner);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nn0 = V.nn0[s];
    int first = V.npts;
#pragma unroll
    for (int r = kVorStrips - 1; r >= 0; --r) {
        const int i = (wave * kVorStrips + r) * 64 + lane;
        const unsigned long long m = __ballot(i < npt && owner[r] == nn0);
        if (m) first = i0 + (wave * kVorStrips + r) * 64 + __builtin_ctzll(m);
    }
    if (lane == 0 && first < V.npts) atomicMin(&V.istar[s], first);
}

// Pass B: blocks over (chunk of points from 0, sightline), points before
// istar.  A strip's points belong to one or two particles: one lane per run
// of equal owners updates its first and last point and its count.
__global__ __launch_bounds__(kVorThreads) void vor_cells_kernel(VorArgs V)
{
    const int s = blockIdx.y;
    const int i0 = blockIdx.x * kVorPts;
    if (V.nn0[s] < 0 || i0 >= V.istar[s]) return;
    const int npt = min(kVorPts, V.istar[s] - i0);
    const VorRow R = vor_row(V, s);
    int owner[kVorStrips];
    vor_owners(V, R, i0, npt, owner);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int r = 0; r < kVorStrips; ++r) {
        const int f = (wave * kVorStrips + r) * 64;
        unsigned long long left = __ballot(f + lane < npt);
        while (left) {
            const int lead = __builtin_ctzll(left);
            const int own = __shfl(owner[r], lead, 64);
            const unsigned long long m = __ballot(owner[r] == own) & left;
            left &= ~m;
            if (lane == lead) {
                const long long k = R.p0 + own;
                atomicMin(&V.first[k], i0 + f + lead);
                atomicMax(&V.last[k], i0 + f + 63 - __builtin_clzll(m));
                atomicAdd(&V.count[k], __popcll(m));
            }
        }
    }
}

// Pass C: one block per sightline, threads over its particles.
__global__ __launch_bounds__(kVorThreads) void vor_segments_kernel(VorArgs V)
{
    const int s = blockIdx.x;
    const long long p0 = V.line_off[s], n = V.line_off[s + 1] - p0;
    const double reso = V.reso, box = V.box;
    for (long long j = threadIdx.x; j < n; j += kVorThreads) {
        const long long k = p0 + j;
        const int c = V.count[k];
        float lo = (float)(3 * box), hi = (float)(3 * box);
        if (c > 0) {
            const int f = V.first[k], l = V.last[k];
            if (c != l - f + 1) atomicOr(&V.err[s], 1);   // two separate runs: the reference exits
            lo = (float)((f + 0.5) * reso);
            hi = (float)((l + 0.5) * reso);
            if (j == V.nn0[s] && V.istar[s] < V.npts) {
                // the wrap (index_table.cpp:187-196): the segment restarts at
                // istar and its end moves on by one box length
                lo = (float)((V.istar[s] + 0.5) * reso);
                hi = (float)((double)hi + box);
            }
        }
        // index_table.cpp:218-221
        V.seg[k] = make_float2((float)((double)lo - 0.5 * reso), (float)((double)hi + 0.5 * reso));
    }
}

int plan_assign_cells(fsamd_plan *P, const float *pos, hipStream_t s)
{
    int rc;
    const long long M = P->npairs;
    const int L = P->nlos;
    if ((rc = P->seg.alloc(sizeof(float2) * (size_t)std::max<long long>(M, 1), P->arena))) return rc;
    P->seg_ready = false;
    if (L == 0 || M == 0) {
        P->seg_ready = true;
        return FSAMD_OK;
    }
    const int npts = (int)(P->box / kReso);
    if (npts < 1) return fail(FSAMD_ERR_ARG, "the box is shorter than the Voronoi grid spacing (0.1)");
    VorArgs V;
    V.box = P->box;
    V.reso = P->box / npts;
    V.npts = npts;
    // first point past the middle of the box (the wrap test of index_table.cpp:187)
    int imin = 0;
    while (imin < npts && !((imin + 0.5) * V.reso > P->box / 2. + 0.5 * V.reso)) ++imin;
    V.imin = imin;
    V.pos = pos;
    V.axis = P->axis.as<int>();
    V.cofm = P->cofm.as<double>();
    V.line_off = P->line_off.as<long long>();
    V.pair_part = P->pair_part.as<int>();
    V.nlos = L;
    DevBuf nn0, istar, first, last, count, err;
    if ((rc = nn0.alloc(sizeof(int) * (size_t)L, P->arena)) || (rc = istar.alloc(sizeof(int) * (size_t)L, P->arena)) ||
        (rc = err.alloc(sizeof(int) * (size_t)L, P->arena)) ||
        (rc = first.alloc(sizeof(int) * (size_t)M, P->arena)) || (rc = last.alloc(sizeof(int) * (size_t)M, P->arena)) ||
        (rc = count.alloc(sizeof(int) * (size_t)M, P->arena)))
        return rc;
    V.nn0 = nn0.as<int>();
    V.istar = istar.as<int>();
    V.err = err.as<int>();
    V.first = first.as<int>();
    V.last = last.as<int>();
    V.count = count.as<int>();
    V.seg = P->seg.as<float2>();
    if ((rc = launch_fill_i32(V.err, 0, L, s)) || (rc = launch_fill_i32(V.first, INT32_MAX, M, s)) ||
        (rc = launch_fill_i32(V.last, -1, M, s)) || (rc = launch_fill_i32(V.count, 0, M, s)))
        return rc;
    vor_first_kernel<<<L, kVorThreads, 0, s>>>(V);
    FSAMD_HIP(hipGetLastError());
    const int chunks_a = (npts - imin + kVorPts - 1) / kVorPts;
    if (chunks_a > 0) {
        vor_wrap_kernel<<<dim3(chunks_a, L), kVorThreads, 0, s>>>(V);
        FSAMD_HIP(hipGetLastError());
    }
    vor_cells_kernel<<<dim3((npts + kVorPts - 1) / kVorPts, L), kVorThreads, 0, s>>>(V);
    FSAMD_HIP(hipGetLastError());
    vor_segments_kernel<<<L, kVorThreads, 0, s>>>(V);
    FSAMD_HIP(hipGetLastError());
    std::vector<int> herr(L);
    FSAMD_HIP(hipMemcpyAsync(herr.data(), V.err, sizeof(int) * L, hipMemcpyDeviceToHost, s));
    FSAMD_HIP(hipStreamSynchronize(s));
    for (int i = 0; i < L; ++i)
        if (herr[i])
            return fail(FSAMD_ERR_ARG, "Voronoi cell assignment: a particle owns two separate runs of sightline " +
                                           std::to_string(i) + " (the reference exits here, index_table.cpp:199-206)");
    P->seg_ready = true;
    return FSAMD_OK;
}

// ---------------------------------------------------------------------------
// Host side

// Device memory kept across plans.  Buffers recycled where no queued work can
// still use them (after a synchronization: a plan's own buffers when it is
// destroyed, the binning's temporaries at its end) go to a per-device free
// list instead of hipFree, so that plans of one shape made one after another
// (the drop-in's plan per call, a loop over snapshots) reuse the same blocks
// instead of allocating and freeing some 20 GB of pair buffers each time.
// Sizes are rounded (256 B, or 2 MiB above 2 MiB); a request takes the
// smallest pooled block that fits with at most 1/4 + 2 MiB to spare.  The
// pool keeps at most kPoolCap bytes per device; a hipMalloc that fails
// empties the calling device's pool and tries again.
namespace {
constexpr size_t kPoolCap = 64ull << 30;
constexpr size_t kBig = 2ull << 20;
std::mutex g_pool_mu;
std::map<int, std::multimap<size_t, void *>> g_pool;
std::map<int, size_t> g_pool_bytes;

size_t pool_round(size_t n) { return n >= kBig ? (n + kBig - 1) & ~(kBig - 1) : (n + 255) & ~(size_t)255; }

bool pool_take(int dev, size_t n, void *&p, size_t &bytes)
{
    std::lock_guard<std::mutex> g(g_pool_mu);
    auto &m = g_pool[dev];
    auto it = m.lower_bound(n);
    if (it == m.end() || it->first > n + n / 4 + kBig) return false;
    p = it->second;
    bytes = it->first;
    g_pool_bytes[dev] -= bytes;
    m.erase(it);
    return true;
}

bool pool_put(int dev, void *p, size_t bytes)
{
    std::lock_guard<std::mutex> g(g_pool_mu);
    if (g_pool_bytes[dev] + bytes > kPoolCap) return false;
    g_pool[dev].emplace(bytes, p);
    g_pool_bytes[dev] += bytes;
    return true;
}

void pool_flush(int dev)
{
    std::multimap<size_t, void *> m;
    {
        std::lock_guard<std::mutex> g(g_pool_mu);
        m.swap(g_pool[dev]);
        g_pool_bytes[dev] = 0;
    }
    for (auto &e : m) (void)hipFree(e.second);
}
}  // namespace

}  // namespace fsamd

extern "C" int fsamd_pool_release(void)
{
    int d = 0;
    FSAMD_HIP(hipGetDevice(&d));
    FSAMD_HIP(hipDeviceSynchronize());
    fsamd::pool_flush(d);
    return FSAMD_OK;
}

namespace fsamd {

DevBuf::~DevBuf() { release(); }

void DevBuf::release()
{
    if (ptr && !borrowed) (void)hipFree(ptr);
    ptr = nullptr;
    bytes = 0;
    borrowed = false;
    dev = -1;
}

void DevBuf::recycle()
{
    if (ptr && !borrowed && dev >= 0 && pool_put(dev, ptr, bytes)) {
        ptr = nullptr;
        bytes = 0;
        dev = -1;
        return;
    }
    release();
}

int DevBuf::alloc(size_t n, Arena *arena)
{
    release();
    if (n == 0) n = 16;
    if (arena) {
        const size_t at = (arena->used + 255) & ~(size_t)255;
        if (at > arena->cap || n > arena->cap - at)
            return fail(FSAMD_ERR_UNSUPPORTED, "this call needs more device memory than the " +
                                                   std::to_string(arena->cap >> 20) +
                                                   " MiB scratch of the allocation-free entry; "
                                                   "use the allocating entry point");
        ptr = arena->base + at;
        bytes = n;
        borrowed = true;
        arena->used = at + n;
        return FSAMD_OK;
    }
    int d = 0;
    FSAMD_HIP(hipGetDevice(&d));
    n = pool_round(n);
    if (pool_take(d, n, ptr, bytes)) {
        dev = d;
        return FSAMD_OK;
    }
    hipError_t e = hipMalloc(&ptr, n);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        pool_flush(d);
        e = hipMalloc(&ptr, n);
    }
    if (e != hipSuccess) {
        ptr = nullptr;
        (void)hipGetLastError();
        return fail(FSAMD_ERR_OOM, "hipMalloc of " + std::to_string(n) + " bytes failed");
    }
    bytes = n;
    dev = d;
    return FSAMD_OK;
}

static int choose_cells(int n)
{
    if (n <= 0) return 1;
    int c = (int)std::ceil(std::sqrt((double)n));
    return std::max(1, std::min(c, 4096));
}

// The sightline grid of a plan (IndexTable ctor, index_table.cpp:7-18):
// copies of axis/cofm, per-axis cell counts, cell starts, sightline ids and
// (key, second) coordinates in cell order.
static int grid_build(fsamd_plan *P, double box, const int *axis, const double *cofm, int nlos, hipStream_t s)
{
    int rc;
    P->box = box;
    P->nlos = nlos;
    if ((rc = P->axis.alloc(sizeof(int) * (size_t)nlos, P->arena))) return rc;
    if ((rc = P->cofm.alloc(sizeof(double) * 3 * (size_t)nlos, P->arena))) return rc;
    DevBuf counts3;
    if ((rc = counts3.alloc(sizeof(int) * 4, P->arena))) return rc;
    if (nlos <= kIntakeMax) {
        los_intake_kernel<<<1, kGridThreads, 0, s>>>(axis, cofm, nlos, P->axis.as<int>(), P->cofm.as<double>(),
                                                     counts3.as<int>());
        FSAMD_HIP(hipGetLastError());
    } else {
        FSAMD_HIP(hipMemcpyAsync(P->axis.ptr, axis, sizeof(int) * nlos, hipMemcpyDeviceToDevice, s));
        FSAMD_HIP(hipMemcpyAsync(P->cofm.ptr, cofm, sizeof(double) * 3 * nlos, hipMemcpyDeviceToDevice, s));
        FSAMD_HIP(hipMemsetAsync(counts3.ptr, 0, sizeof(int) * 4, s));
        los_axis_count_kernel<<<std::min((nlos + 255) / 256, kAxisBlocks), 256, 0, s>>>(P->axis.as<int>(), nlos, counts3.as<int>());
        FSAMD_HIP(hipGetLastError());
    }
    // --- sightline grid
    int hc[4] = {0, 0, 0, 0};
    FSAMD_HIP(hipMemcpyAsync(hc, counts3.ptr, sizeof(int) * 3, hipMemcpyDeviceToHost, s));
    FSAMD_HIP(hipStreamSynchronize(s));
    LosGrid &g = P->grid;
    int ncells = 0;
    for (int a = 0; a < 3; ++a) {
        g.nlos_axis[a] = hc[a];
        g.nc[a] = choose_cells(hc[a]);
        g.cw[a] = box / g.nc[a];
        g.inv_cw[a] = g.nc[a] / box;
        g.base[a] = ncells;
        ncells += g.nc[a] * g.nc[a];
    }
    P->ncells = ncells;
    if ((rc = P->cell_start.alloc(sizeof(int) * (size_t)(ncells + 1), P->arena))) return rc;
    if ((rc = P->cell_ids.alloc(sizeof(int) * (size_t)std::max(nlos, 1), P->arena))) return rc;
    if ((rc = P->cell_kl.alloc(sizeof(double2) * (size_t)std::max(nlos, 1), P->arena))) return rc;
    g.cell_start = P->cell_start.as<int>();
    g.cell_ids = P->cell_ids.as<int>();
    g.cell_kl = P->cell_kl.as<double2>();
    if (ncells <= kGridSmallCells) {
        grid_small_kernel<<<1, kGridThreads, sizeof(int) * (size_t)ncells, s>>>(
            P->axis.as<int>(), P->cofm.as<double>(), nlos, box, g, ncells, P->cell_start.as<int>(),
            P->cell_ids.as<int>(), P->cell_kl.as<double2>());
        FSAMD_HIP(hipGetLastError());
        return FSAMD_OK;
    }
    DevBuf cell_of, cell_count, cell_cursor, scan_ws, cell_start64;
    if ((rc = cell_of.alloc(sizeof(int) * (size_t)std::max(nlos, 1), P->arena))) return rc;
    if ((rc = cell_count.alloc(sizeof(int) * (size_t)(ncells + 1), P->arena))) return rc;
    if ((rc = cell_start64.alloc(sizeof(long long) * (size_t)(ncells + 1), P->arena))) return rc;
    if ((rc = scan_ws.alloc(exclusive_scan_ws_bytes((long long)ncells + 1), P->arena))) return rc;
    if ((rc = launch_fill_i32(cell_count.as<int>(), 0, ncells + 1, s))) return rc;
    if (nlos > 0) {
        los_cell_kernel<<<(nlos + 255) / 256, 256, 0, s>>>(P->axis.as<int>(), P->cofm.as<double>(), nlos, box, g,
                                                           cell_of.as<int>(), cell_count.as<int>());
        FSAMD_HIP(hipGetLastError());
    }
    if ((rc = exclusive_scan_i32_to_i64(cell_count.as<int>(), cell_start64.as<long long>(), ncells,
                                        scan_ws.ptr, scan_ws.bytes, s)))
        return rc;
    i64_to_i32_kernel<<<grid_for(ncells + 1, 256), 256, 0, s>>>(cell_start64.as<long long>(),
                                                                P->cell_start.as<int>(), ncells + 1);
    FSAMD_HIP(hipGetLastError());
    if ((rc = cell_cursor.alloc(sizeof(int) * (size_t)(ncells + 1), P->arena))) return rc;
    FSAMD_HIP(hipMemcpyAsync(cell_cursor.ptr, P->cell_start.ptr, sizeof(int) * (ncells + 1),
                             hipMemcpyDeviceToDevice, s));
    if (nlos > 0) {
        los_scatter_kernel<<<(nlos + 255) / 256, 256, 0, s>>>(P->axis.as<int>(), P->cofm.as<double>(), nlos,
                                                              cell_of.as<int>(), cell_cursor.as<int>(),
                                                              P->cell_ids.as<int>(), P->cell_kl.as<double2>());
        FSAMD_HIP(hipGetLastError());
    }
    return FSAMD_OK;
}

int plan_build(fsamd_plan *P, double box, const float *pos, const float *h, long long npart,
               const int *axis, const double *cofm, int nlos, hipStream_t s)
{
    int rc;
    P->npart = npart;
    if ((rc = grid_build(P, box, axis, cofm, nlos, s))) return rc;
    const LosGrid &g = P->grid;
    DevBuf scan_ws;
    if ((rc = scan_ws.alloc(exclusive_scan_ws_bytes(npart + 1), P->arena))) return rc;

    // --- count, scan, emit
    BinArgs A;
    A.box = box;
    A.pos = pos;
    A.h = h;
    A.npart = npart;
    A.grid = g;
    DevBuf cnt;
    if ((rc = cnt.alloc(sizeof(int) * (size_t)std::max<long long>(npart, 1), P->arena))) return rc;
    if ((rc = P->poff.alloc(sizeof(long long) * (size_t)(npart + 1), P->arena))) return rc;
    if (npart > 0) {
        bin_count_kernel<<<grid_for(npart, 256, 1 << 20), 256, 0, s>>>(A, cnt.as<int>());
        FSAMD_HIP(hipGetLastError());
    }
    if ((rc = exclusive_scan_i32_to_i64(cnt.as<int>(), P->poff.as<long long>(), npart, scan_ws.ptr,
                                        scan_ws.bytes, s)))
        return rc;
    long long M = 0;
    FSAMD_HIP(hipMemcpyAsync(&M, P->poff.as<long long>() + npart, sizeof(long long), hipMemcpyDeviceToHost, s));
    FSAMD_HIP(hipStreamSynchronize(s));
    cnt.recycle();
    P->npairs = M;
    DevBuf k0, v0, k1, v1;
    const size_t mbytes = sizeof(int) * (size_t)std::max<long long>(M, 1);
    if ((rc = k0.alloc(mbytes, P->arena)) || (rc = v0.alloc(mbytes, P->arena)) || (rc = k1.alloc(mbytes, P->arena)) || (rc = v1.alloc(mbytes, P->arena)))
        return rc;
    if (npart > 0 && M > 0) {
        bin_emit_kernel<<<grid_for(npart, 256, 1 << 20), 256, 0, s>>>(A, P->poff.as<long long>(), k0.as<int>(),
                                                                      v0.as<int>());
        FSAMD_HIP(hipGetLastError());
    }
    // --- stable radix sort by sightline id, ping-pong between (k0,v0) and (k1,v1)
    int total_bits = 1;
    while ((1ll << total_bits) < (long long)nlos) ++total_bits;
    const int passes = (total_bits + kRsMaxBits - 1) / kRsMaxBits;
    const int bits_per = (total_bits + passes - 1) / passes;
    DevBuf *kin = &k0, *vin = &v0, *kout = &k1, *vout = &v1;
    DevBuf table, tws;
    if (M > 0) {
        const long long ntiles = (M + kRsTile - 1) / kRsTile;
        if ((rc = table.alloc(sizeof(long long) * (size_t)((1 << bits_per) * ntiles + 1), P->arena))) return rc;
        if ((rc = tws.alloc(exclusive_scan_ws_bytes((1 << bits_per) * ntiles + 1), P->arena))) return rc;
        for (int ps = 0; ps < passes; ++ps) {
            const int shift = ps * bits_per;
            const int bits = std::min(bits_per, total_bits - shift);
            rs_upsweep_kernel<<<(int)ntiles, kRsThreads, 0, s>>>(kin->as<int>(), M, shift, bits, ntiles,
                                                                 table.as<long long>());
            FSAMD_HIP(hipGetLastError());
            if ((rc = exclusive_scan_i64_inplace(table.as<long long>(), (1ll << bits) * ntiles, tws.ptr,
                                                 tws.bytes, s)))
                return rc;
            rs_downsweep_kernel<<<(int)ntiles, kRsThreads, 0, s>>>(kin->as<int>(), vin->as<int>(), kout->as<int>(),
                                                                   vout->as<int>(), M, shift, bits, ntiles,
                                                                   table.as<long long>());
            FSAMD_HIP(hipGetLastError());
            std::swap(kin, kout);
            std::swap(vin, vout);
        }
    }
    // (kin, vin) hold the sorted sightline ids and particle ids
    P->pair_part.take(*vin);
    if ((rc = P->line_off.alloc(sizeof(long long) * (size_t)(nlos + 1), P->arena))) return rc;
    row_offsets_kernel<<<(nlos + 1 + 255) / 256, 256, 0, s>>>(kin->as<int>(), M, nlos,
                                                             P->line_off.as<long long>());
    FSAMD_HIP(hipGetLastError());

    // --- work order: sightlines by descending pair count (stable)
    std::vector<long long> off(nlos + 1);
    FSAMD_HIP(hipMemcpyAsync(off.data(), P->line_off.ptr, sizeof(long long) * (nlos + 1),
                             hipMemcpyDeviceToHost, s));
    FSAMD_HIP(hipStreamSynchronize(s));
    // the binning's temporaries are idle now
    for (DevBuf *b : {&scan_ws, kin, kout, vout, &table, &tws}) b->recycle();
    P->max_row = 0;
    for (int i = 0; i < nlos; ++i) P->max_row = std::max(P->max_row, off[i + 1] - off[i]);
    std::vector<int> order(nlos);
    if (P->max_row <= 4 * (long long)nlos + (1 << 20)) {
        // counting sort on the pair count, descending, stable
        std::vector<int> first((size_t)P->max_row + 2, 0);
        for (int i = 0; i < nlos; ++i) ++first[(size_t)(P->max_row - (off[i + 1] - off[i])) + 1];
        for (size_t c = 1; c < first.size(); ++c) first[c] += first[c - 1];
        for (int i = 0; i < nlos; ++i) order[first[(size_t)(P->max_row - (off[i + 1] - off[i]))]++] = i;
    } else {
        std::iota(order.begin(), order.end(), 0);
        std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
            return off[a + 1] - off[a] > off[b + 1] - off[b];
        });
    }
    P->order_host = std::move(order);
    P->off_host = std::move(off);
    return FSAMD_OK;
}

int near_lines_direct(double box, const float *pos, const float *h, long long npart, const int *axis,
                      const double *cofm, int nlos, int *out, long long *n_out, hipStream_t s)
{
    int rc;
    *n_out = 0;
    if (npart == 0 || nlos == 0) return FSAMD_OK;
    fsamd_plan G;   // holds the grid's buffers for this call
    G.npart = npart;
    if ((rc = grid_build(&G, box, axis, cofm, nlos, s))) return rc;
    BinArgs A;
    A.box = box;
    A.pos = pos;
    A.h = h;
    A.npart = npart;
    A.grid = G.grid;
    // one mask word and one count per 64 particles: the scan and the ids'
    // placement then read 20 bytes a word instead of 12 a particle
    const long long nw = (npart + 63) / 64;
    DevBuf mask, cnt, off, ws;
    if ((rc = mask.alloc(sizeof(unsigned long long) * (size_t)nw))) return rc;
    if ((rc = cnt.alloc(sizeof(int) * (size_t)nw))) return rc;
    if ((rc = off.alloc(sizeof(long long) * (size_t)(nw + 1)))) return rc;
    if ((rc = ws.alloc(exclusive_scan_ws_bytes(nw + 1)))) return rc;
    bin_any_kernel<<<grid_for(nw, kAnyWords, 1 << 20), 256, 0, s>>>(A, mask.as<unsigned long long>(), cnt.as<int>());
    FSAMD_HIP(hipGetLastError());
    if ((rc = exclusive_scan_i32_to_i64(cnt.as<int>(), off.as<long long>(), nw, ws.ptr, ws.bytes, s))) return rc;
    mask_scatter_kernel<<<grid_for(nw, 4, 1 << 16), 256, 0, s>>>(mask.as<unsigned long long>(), off.as<long long>(), nw,
                                                                 out);
    FSAMD_HIP(hipGetLastError());
    long long found = 0;
    FSAMD_HIP(hipMemcpyAsync(&found, off.as<long long>() + nw, sizeof(long long), hipMemcpyDeviceToHost, s));
    FSAMD_HIP(hipStreamSynchronize(s));
    for (DevBuf *b : {&mask, &cnt, &off, &ws}) b->recycle();
    *n_out = found;
    return FSAMD_OK;
}

int plan_near_lines(const fsamd_plan *P, int *out, long long *n_out, hipStream_t s)
{
    int rc;
    const long long n = P->npart;
    if (n == 0) {
        *n_out = 0;
        return FSAMD_OK;
    }
    DevBuf flag, fscan, ws;
    if ((rc = flag.alloc(sizeof(int) * (size_t)n))) return rc;
    if ((rc = fscan.alloc(sizeof(long long) * (size_t)(n + 1)))) return rc;
    if ((rc = ws.alloc(exclusive_scan_ws_bytes(n + 1)))) return rc;
    near_flag_kernel<<<grid_for(n, 256), 256, 0, s>>>(P->poff.as<long long>(), n, flag.as<int>());
    FSAMD_HIP(hipGetLastError());
    if ((rc = exclusive_scan_i32_to_i64(flag.as<int>(), fscan.as<long long>(), n, ws.ptr, ws.bytes, s)))
        return rc;
    near_scatter_kernel<<<grid_for(n, 256), 256, 0, s>>>(P->poff.as<long long>(), fscan.as<long long>(), n, out);
    FSAMD_HIP(hipGetLastError());
    long long cnt = 0;
    FSAMD_HIP(hipMemcpyAsync(&cnt, fscan.as<long long>() + n, sizeof(long long), hipMemcpyDeviceToHost, s));
    FSAMD_HIP(hipStreamSynchronize(s));
    for (DevBuf *b : {&flag, &fscan, &ws}) b->recycle();
    *n_out = cnt;
    return FSAMD_OK;
}

}  // namespace fsamd

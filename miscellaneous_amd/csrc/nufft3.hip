// nufft3.hip -- the type-3 2-D NUFFT (non-uniform to non-uniform, FP64) on
// gfx950:
//     F_j = sum_k f_k e^{-i (s_j x_k + t_j y_k)},
// the GPU counterpart of NUFFT_2D_CPU (NFFT/NFFT3/C/NFFT3_2D_C.cpp:199-312):
// Gaussian gridding with the reference's parameters (R = 2.2, the tap
// half-width msp from eps, an Mry x Mrx grid sized by the data extents).
//
// One call:
//   1. k3_extent / k3_extent_final: min and max of x, y, s, t (and whether all
//      are finite).  The host reads them back -- the call's one
//      synchronisation -- and derives every parameter exactly as :214-267, and
//      from the extremes' own cells the part of the grid that the inputs reach
//      and the part of the spectrum that the outputs read (about half and two
//      fifths per side: the reference's grid holds R = 2.2 times the band, the
//      inputs lie in its middle half).  Everything below works on those parts.
//   2. k3_prep: per input its pre-modulated sample and grid cell, per output
//      its cell and post-compensation factor; both are counted into bins
//      (inputs 8 x 8 cells, outputs 16 x 16 cells and 8 x 2 blocks of them) and
//      sorted (k3_scan_local, k3_scan_totals, k3_scatter).
//   3. k3_spread: one block per 16 x 16 tile of the reached cells sums
//      c_k ey_k(j) ex_k(i) over the inputs within reach of the tile, four
//      inputs per v_mfma_f64_16x16x4f64 (the Gaussian of :76 is separable);
//      the cell factor fact e^{b (Dx^2 dsi^2 + Dy^2 dsj^2)} multiplies the
//      finished tile.  Each cell is written once: no atomics, no zero fill.
//   4. The forward 2-D DFT of the grid (:280-292) from the reached rows and
//      cells to the read frequencies, as two chirp-z passes (nfft2d_czt.hpp):
//      P inputs and Q outputs of a line are a convolution of P + Q - 1 points,
//      a grid side of 1,638 takes 2,048 instead of the 4,096 of a full
//      Bluestein transform, on half and two fifths of the lines.  The first
//      pass writes its lines side by side: no transpose.  The circular and FFT
//      shifts and the checkerboard sign of circAndFFTShiftsFunction (:135-151)
//      are the passes' output offset and a sign in their output factors.
//   5. k3_interp: one block per output bin stages the bin's patch of the
//      spectrum in LDS; one wave per 16 outputs sums the (2 R + 1)^2
//      separable Gaussian taps and applies the post-compensation of
//      spectralConvolutionFunctionCompensation (:156-194).
// 300,000 -> 300,000, X1 S = Y1 T = 500, eps 1e-6 (grid 1,638^2): 835 -> 288 us.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <chrono>
#include <cmath>
#include <map>
#include <mutex>

#include "../../include/nfft2d.h"
#include "nfft2d_czt.hpp"
#include "nfft2d_internal.hpp"

namespace nufft3 {

constexpr int kTile = 16;              // grid tile and output bin edge, cells
constexpr int kInBin = 8;              // input bin edge, cells (finer: fewer out-of-reach candidates per tile)
constexpr int kMaxMsp = 42;            // LDS patch (16 + 2 msp)^2 x 16 B <= 160 000 B
constexpr int kMaxFft = 8192;          // longest FFT of a chirp-z line (139 KB of LDS)
constexpr int kExtentBlocks = 1024;
typedef double d4 __attribute__((ext_vector_type(4)));

struct Par {
    double xb, yb, sb, tb, kkx, kky, Dx, Dy, b, t1, fact;
    int reach, Mrx, Mry;      // taps per side in use (at most msp, see tap_reach)
    int ci, cj, ni, nj;       // input cells [ci, ci + ni) x [cj, cj + nj); 8 x 8-cell bins from (ci, cj)
    int oi, oj, mi, mj;       // output cells [oi, oi + mi) x [oj, oj + mj); 16 x 16-cell bins from (oi, oj)
    int ibx, iby, nbx, nby;   // input bins, output bins
    int gi, gj, Px, Py;       // reached cells [gi, gi + Px) x [gj, gj + Py)
    int qi, qj, Qx, Qy;       // read frequencies qi + [0, Qx), qj + [0, Qy) (mod Mrx, Mry)
};

struct alignas(16) InRec {     // one input, in bin order
    double xt, yt, re, im;     // scaled offsets (x - xb) / Dx, (y - yb) / Dy; pre-modulated sample
};
struct alignas(16) OutRec {    // one output, in bin order
    double difs, dift;         // fractional cell offsets
    double pr, pi;             // post-compensation factor
    int nsn, ntn, idx, pad;
};

// ------------------------------------------------------------ 1. extents
// 9 values per block: max x, min x, max y, min y, max s, min s, max t, min t,
// and 1.0 if any coordinate is not finite.  The start values are -FLT_MAX /
// FLT_MAX, as the reference's thrust::reduce calls (:214-231).
__device__ __forceinline__ double wmax(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ double wmin(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
    return v;
}

__global__ __launch_bounds__(256) void k3_extent(const double *__restrict__ x, const double *__restrict__ y,
                                                 const double *__restrict__ s, const double *__restrict__ t,
                                                 int len_in, int len_out, double *__restrict__ part)
{
    __shared__ double red[4][9];
    double v[9];
    for (int q = 0; q < 8; q += 2) {
        v[q] = -(double)FLT_MAX;
        v[q + 1] = (double)FLT_MAX;
    }
    v[8] = 0.0;
    const int stride = gridDim.x * 256;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < len_in; i += stride) {
        const double a = x[i], c = y[i];
        if (!isfinite(a) || !isfinite(c)) v[8] = 1.0;
        if (a > v[0]) v[0] = a;
        if (a < v[1]) v[1] = a;
        if (c > v[2]) v[2] = c;
        if (c < v[3]) v[3] = c;
    }
    for (int i = blockIdx.x * 256 + threadIdx.x; i < len_out; i += stride) {
        const double a = s[i], c = t[i];
        if (!isfinite(a) || !isfinite(c)) v[8] = 1.0;
        if (a > v[4]) v[4] = a;
        if (a < v[5]) v[5] = a;
        if (c > v[6]) v[6] = c;
        if (c < v[7]) v[7] = c;
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < 9; ++q) {
        const double r = (q & 1) && q < 8 ? wmin(v[q]) : wmax(v[q]);
        if (lane == 0) red[w][q] = r;
    }
    __syncthreads();
    if (threadIdx.x < 9) {
        const int q = threadIdx.x;
        double r = red[0][q];
        for (int ww = 1; ww < 4; ++ww) r = (q & 1) && q < 8 ? fmin(r, red[ww][q]) : fmax(r, red[ww][q]);
        part[blockIdx.x * 9 + q] = r;
    }
}

// One wave per quantity, its loads in flight together (one wave for all nine
// in turn took 26 us); the results go straight to the host's buffer (pinned memory), then the call's number, for which the host polls: a stream
// synchronisation returns about 10 us later.
__global__ __launch_bounds__(64 * 9) void k3_extent_final(const double *__restrict__ part, int nblk, double call,
                                                          double *__restrict__ out)
{
    const int q = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const bool mn = (q & 1) && q < 8;
    const double none = q == 8 ? 0.0 : mn ? (double)FLT_MAX : -(double)FLT_MAX;
    double v[kExtentBlocks / 64];
#pragma unroll
    for (int k = 0; k < kExtentBlocks / 64; ++k) v[k] = 64 * k + lane < nblk ? part[(64 * k + lane) * 9 + q] : none;
    double r = none;
#pragma unroll
    for (int k = 0; k < kExtentBlocks / 64; ++k) r = mn ? fmin(r, v[k]) : fmax(r, v[k]);
    r = mn ? wmin(r) : wmax(r);
    if (lane == 0) __hip_atomic_store(&out[q], r, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(&out[9], call, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ------------------------------------------------------------ 2. points and bins
// Keys: inputs their 8 x 8-cell bin; outputs their 16 x 16-cell bin and the
// 8 x 2 block inside it (8 rows, 2 columns), so that 16 outputs in a row share
// most of their windows: 39 taps cover 46 rows (three MFMA tiles, as one window
// does) and about 41 columns.  Key nki / nko (never read) takes cells outside the grid,
// which the extents rule out but for rounding at huge offsets.
__device__ __forceinline__ void prep_in(int k, const double *__restrict__ x0, const double *__restrict__ y0,
                                        const double2 *__restrict__ f, const Par &p, InRec *__restrict__ rec,
                                        int2 *__restrict__ kr, int *__restrict__ cnt)
{
#pragma clang fp contract(off)
    // spatialConvolutionFunction (:38-63), on the rescaled x / kk_x, y / kk_y (:247-248)
    const double x = x0[k] / p.kkx, y = y0[k] / p.kky;
    const double2 v = f[k];
    InRec r;
    r.xt = (x - p.xb) / p.Dx;
    r.yt = (y - p.yb) / p.Dy;
    const int i = (int)floor((double)(p.Mrx / 2) + r.xt) - p.ci, j = (int)floor((double)(p.Mry / 2) + r.yt) - p.cj;
    const bool ok = i >= 0 && i < p.ni && j >= 0 && j < p.nj;
    const int bin = ok ? (j / kInBin) * p.ibx + i / kInBin : p.ibx * p.iby;
    const int rank = atomicAdd(&cnt[bin], 1);
    const double arg = p.sb * x + p.tb * y;
    double sn, cs;
    sincos(arg, &sn, &cs);
    r.re = v.x * cs + v.y * sn;
    r.im = v.y * cs - v.x * sn;
    rec[k] = r;
    kr[k] = make_int2(bin, rank);
}

__device__ __forceinline__ void prep_out(int k, const double *__restrict__ s0, const double *__restrict__ t0,
                                         const Par &p, OutRec *__restrict__ rec, int2 *__restrict__ kr,
                                         int *__restrict__ cnt, double2 *__restrict__ F)
{
#pragma clang fp contract(off)
    // spectralConvolutionFunctionCompensation (:164-167), s * kk_x, t * kk_y (:249-250), Ds = Dt = 1
    const double s = s0[k] * p.kkx, t = t0[k] * p.kky;
    const double sd = s - p.sb, td = t - p.tb;
    OutRec r;
    r.nsn = (int)floor((double)(p.Mrx / 2) + sd);
    r.difs = ((double)(p.Mrx / 2) + sd) - r.nsn;
    r.ntn = (int)floor((double)(p.Mry / 2) + td);
    r.dift = ((double)(p.Mry / 2) + td) - r.ntn;
    r.idx = k;
    r.pad = 0;
    const int i = r.nsn - p.oi, j = r.ntn - p.oj;
    const bool ok = i >= 0 && i < p.mi && j >= 0 && j < p.mj;
    const int bin = ok ? ((j / kTile) * p.nbx + i / kTile) * kTile + (j % kTile) / 8 * 8 + (i % kTile) / 2
                       : p.nbx * p.nby * kTile;
    const int rank = atomicAdd(&cnt[bin], 1);
    if (!ok) F[k] = make_double2(NAN, NAN);
    const double a1 = p.Dy * td, a2 = p.Dx * sd;
    const double temp = exp(p.b * (a1 * a1 + a2 * a2));
    const double arg = sd * p.xb + td * p.yb;
    double sn, cs;
    sincos(arg, &sn, &cs);
    r.pr = cs * temp;
    r.pi = sn * temp;
    rec[k] = r;
    kr[k] = make_int2(bin, rank);
}

// Blocks below gin take inputs, the others outputs: one launch, so that the
// two sides' atomics and arithmetic run beside each other.
__global__ __launch_bounds__(256) void k3_prep(const double *__restrict__ x, const double *__restrict__ y,
                                               const double2 *__restrict__ f, int len_in, int gin, Par p,
                                               InRec *__restrict__ rin, int2 *__restrict__ kin, int *__restrict__ cin,
                                               const double *__restrict__ s, const double *__restrict__ t, int len_out,
                                               OutRec *__restrict__ rout, int2 *__restrict__ kout,
                                               int *__restrict__ cout, double2 *__restrict__ F)
{
    if ((int)blockIdx.x < gin) {
        const int k = blockIdx.x * 256 + threadIdx.x;
        if (k < len_in) prep_in(k, x, y, f, p, rin, kin, cin);
    } else {
        const int k = (blockIdx.x - gin) * 256 + threadIdx.x;
        if (k < len_out) prep_out(k, s, t, p, rout, kout, cout, F);
    }
}

// One dimension's chirp-z tables (nfft2d_czt.hpp): lines of P cells from p0 on
// to Q frequencies from q0 on of a side of n, c[k] = e^{-i pi k^2 / n} (k^2
// reduced mod 2n exactly).
struct AxisTables {
    double2 *cin, *cout, *hhat, *tw;   // P, Q, m, m
    int n, P, Q, p0, q0, m;
};
__device__ __forceinline__ double2 chirp3(long long k, int n)
{
    double sn, cs;
    sincospi((double)((k * k) % (2LL * n)) / n, &sn, &cs);
    return make_double2(cs, -sn);
}
// Entry e of the tables; hhat gets the kernel conj(c[d + q0 - p0]) at d mod m,
// d in (-P, Q), which k3_kernel_fft transforms.  The output factors carry the
// checkerboard sign (-1)^k of circAndFFTShiftsFunction (:135-151).
__device__ __forceinline__ void axis_entry(const AxisTables &t, int e)
{
    if (e < t.P) t.cin[e] = chirp3((long long)e + t.p0, t.n);
    if (e < t.Q) {
        const double2 c = chirp3((long long)e + t.q0, t.n);
        t.cout[e] = ((e + t.q0) & 1) ? make_double2(-c.x, -c.y) : c;
    }
    if (e < t.m) {
        double sn, cs;
        sincospi(2.0 * nfft2d::czt_tw_index(t.m, e) / t.m, &sn, &cs);
        t.tw[e] = make_double2(cs, -sn);
        double2 h = make_double2(0.0, 0.0);
        const int d = e < t.Q ? e : e - t.m;
        if (d > -t.P) {
            h = chirp3((long long)d + t.q0 - t.p0, t.n);
            h.y = -h.y;
        }
        t.hhat[e] = h;
    }
}

// Exclusive scan of the key counts in two steps: k3_scan_local scans each
// 1024-key segment and writes the segment totals, k3_scan_totals scans those;
// key i starts at start[i] + tot[i >> 10].  Side 0 the inputs, side 1 the
// outputs; the scan's launch also fills the chirp-z tables (its last blocks).
struct ScanSide {
    int *cnt, *start, *tot;
    int n, segs;   // keys (the out-of-grid one and the end among them), segments
};
__global__ __launch_bounds__(1024) void k3_scan_local(ScanSide a, ScanSide b, AxisTables tx, AxisTables ty)
{
    __shared__ int wsum[16];
    int seg = blockIdx.x;
    if (seg >= a.segs + b.segs) {
        const int e = (seg - a.segs - b.segs) * 1024 + threadIdx.x;
        axis_entry(tx, e);
        axis_entry(ty, e);
        return;
    }
    const ScanSide &s = seg < a.segs ? a : b;
    if (seg >= a.segs) seg -= a.segs;
    const int i = seg * 1024 + threadIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int v = i < s.n ? s.cnt[i] : 0;
    int inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(inc, o, 64);
        if (lane >= o) inc += u;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    int before = 0;
    for (int k = 0; k < w; ++k) before += wsum[k];
    if (i < s.n) s.start[i] = before + inc - v;
    if (threadIdx.x == 1023) s.tot[seg] = before + inc;
}

__global__ __launch_bounds__(1024) void k3_scan_totals(ScanSide a, ScanSide b)
{
    __shared__ int sums[1024];
    const ScanSide &s = blockIdx.x ? b : a;
    const int per = (s.segs + 1023) / 1024;
    const int lo = min(s.segs, (int)threadIdx.x * per), hi = min(s.segs, lo + per);
    int acc = 0;
    for (int i = lo; i < hi; ++i) acc += s.tot[i];
    sums[threadIdx.x] = acc;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        const int u = threadIdx.x >= o ? sums[threadIdx.x - o] : 0;
        __syncthreads();
        sums[threadIdx.x] += u;
        __syncthreads();
    }
    int run = sums[threadIdx.x] - acc;
    for (int i = lo; i < hi; ++i) {
        const int v = s.tot[i];
        s.tot[i] = run;
        run += v;
    }
}

__device__ __forceinline__ int key_start(const int *__restrict__ st, const int *__restrict__ tot, int i)
{
    return st[i] + tot[i >> 10];
}

__global__ __launch_bounds__(256) void k3_scatter(const InRec *__restrict__ rin, const int2 *__restrict__ kin,
                                                  int len_in, int gin, ScanSide a, InRec *__restrict__ sin_,
                                                  const OutRec *__restrict__ rout, const int2 *__restrict__ kout,
                                                  int len_out, ScanSide b, OutRec *__restrict__ sout)
{
    if ((int)blockIdx.x < gin) {
        const int k = blockIdx.x * 256 + threadIdx.x;
        if (k >= len_in) return;
        const int2 e = kin[k];
        sin_[key_start(a.start, a.tot, e.x) + e.y] = rin[k];
    } else {
        const int k = (blockIdx.x - gin) * 256 + threadIdx.x;
        if (k >= len_out) return;
        const int2 e = kout[k];
        sout[key_start(b.start, b.tot, e.x) + e.y] = rout[k];
    }
}

// ------------------------------------------------------------ 3. Gaussian gridding
// Block per 16 x 16 tile (tx, ty) of the reached cells: i in [i0, i0 + 16),
// i0 = gi + 16 tx, j likewise.  An input k reaches cell (i, j) when
// |i - nno_k| <= R and |j - mmo_k| <= R, R = msp (:65-72) or less (tap_reach).
// The 4 waves take turns over the 64-input chunks of the 8 x 8-cell input bins that can reach the
// tile, the next chunk's records in flight.  The inputs within reach (about
// two thirds) go to a queue in LDS, and each full batch of 32 is spread: lane l
// of the lower half takes input l of the batch and writes its 16 row factors
// ey to a slot, lane l + 32 its 16 column factors ex, from two exponentials
// and one product each (fast Gaussian gridding, Greengard & Lee, SIAM Rev. 46
// (2004)): with u = yt - (j0 - Mry/2),
//     e^{-t1 (u - r)^2} = e^{-t1 u^2} (e^{2 t1 u})^r e^{-t1 r^2},
// the last factor, the same for every input, taken into the finished cell's.
// (e^{2 t1 u r} stays below e^{2 t1 (R + 16) 15}, far inside the range.)
// The slots are then taken four per MFMA step: lane l supplies
// A[r][k] = c_k ey_k(j0 + r) and B[k][r] = ex_k(i0 + r) at r = l % 16,
// k = l / 16, and accumulator element q of lane l is cell
// (j0 + 4 q + l / 16, i0 + l % 16).
// MASK: factors outside an input's reach are set to zero.  Without it an input
// that reaches the tile adds its tails there too; beyond R cells a factor is
// below e^{-t1 R^2}, which the host finds to be under 2^-54 of the input's
// largest, and the two selects per factor would cost more than its product.
// What bounds it is FP64 arithmetic: this GPU's FP64 matrix rate is its vector
// rate, and the counters add up as if both shared one pipe (112K matrix and
// about 80K vector cycles of 245K with R = 19).  So the batches keep every lane
// of the factors' work busy (one lane per candidate left a third idle, and its
// slots held LDS for two blocks a CU only), and tails that change nothing are
// not formed.  300,000 inputs, msp 19: 229 us; in batches 119, with one product
// a factor and without the floors in the reach test 116, with R = 16 90.
constexpr int kSpreadWaves = 4;
constexpr int kChunk = 64;        // candidate inputs per wave and round
constexpr int kBatch = 32;        // inputs spread at a time
constexpr int kQueue = kBatch - 1 + kChunk;
constexpr int kRow = kTile + 2;   // padded slot row (doubles, 16-byte aligned)
constexpr int kMaxBinRows = (kTile + 2 * kMaxMsp) / kInBin + 2;   // bin rows that can reach a tile
static_assert(kMaxBinRows <= 64, "one lane per bin row");

struct SpreadLds {
    InRec q[kQueue];
    double ey[kBatch][kRow], ex[kBatch][kRow];
};

__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool MASK>
__global__ __launch_bounds__(64 * kSpreadWaves) void k3_spread(const InRec *__restrict__ pts,
                                                                const int *__restrict__ st,
                                                                const int *__restrict__ tot, Par p, int ntx,
                                                                double2 *__restrict__ G)
{
    __shared__ union {
        SpreadLds s[kSpreadWaves];
        double2 part[kSpreadWaves][kTile * kTile];
    } sh;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    SpreadLds &L = sh.s[w];
    const int tx = blockIdx.x % ntx, ty = blockIdx.x / ntx;
    const int i0 = p.gi + tx * kTile, j0 = p.gj + ty * kTile;
    const int r = lane & 15, ks = lane >> 4;
    const bool rows_half = lane < 32;                     // this lane's factors: rows (ey) or columns (ex)
    const int sl = lane & 31;
    const double org = rows_half ? (double)(j0 - p.Mry / 2) : (double)(i0 - p.Mrx / 2);
    const int half_grid = rows_half ? p.Mry / 2 : p.Mrx / 2, cell0 = rows_half ? j0 : i0;
    const int R = p.reach;
    d4 accr = {0.0, 0.0, 0.0, 0.0}, acci = {0.0, 0.0, 0.0, 0.0};
    const int by0 = max(0, j0 - R - p.cj) / kInBin, by1 = min(p.iby - 1, (j0 + kTile - 1 + R - p.cj) / kInBin);
    const int bx0 = max(0, i0 - R - p.ci) / kInBin, bx1 = min(p.ibx - 1, (i0 + kTile - 1 + R - p.ci) / kInBin);
    // a bin row's inputs are contiguous; lane l holds row by0 + l's range
    int lo_l = 0, hi_l = 0;
    if (by0 + lane <= by1 && bx0 <= bx1) {
        const int k0 = (by0 + lane) * p.ibx + bx0;
        lo_l = key_start(st, tot, k0);
        hi_l = key_start(st, tot, k0 + bx1 - bx0 + 1);
    }

    // inputs whose cell is in [i0 - R, i0 + 16 + R) x [j0 - R, j0 + 16 + R) reach the tile
    const double ilo = i0 - R, ihi = i0 + kTile + R, jlo = j0 - R, jhi = j0 + kTile + R;
    int n = 0;                                            // queued inputs
    auto batch = [&](int q0) {
        // factors of the batch's inputs q0 .. q0 + 31
        const InRec &e = L.q[q0 + sl];
        const double d = rows_half ? e.yt : e.xt, u = d - org;
        double g = exp(-p.t1 * (u * u));
        const double e1 = exp(2.0 * p.t1 * u);
        int lo = 0, hi = kTile - 1;
        if (MASK) {
            const int c = (int)floor((double)half_grid + d) - cell0;
            lo = c - R;
            hi = c + R;
        }
        double *o = rows_half ? L.ey[sl] : L.ex[sl];
#pragma unroll
        for (int k = 0; k < kTile; k += 2) {
            double2 v;
            v.x = !MASK || (k >= lo && k <= hi) ? g : 0.0;
            g *= e1;
            v.y = !MASK || (k + 1 >= lo && k + 1 <= hi) ? g : 0.0;
            g *= e1;
            *reinterpret_cast<double2 *>(o + k) = v;
        }
        wave_lds_sync();
#pragma unroll
        for (int q = 0; q < kBatch; q += 4) {
            const int b = q + ks;
            const double2 c = *reinterpret_cast<const double2 *>(&L.q[q0 + b].re);
            const double wy = L.ey[b][r], wx = L.ex[b][r];
            accr = __builtin_amdgcn_mfma_f64_16x16x4f64(c.x * wy, wx, accr, 0, 0, 0);
            acci = __builtin_amdgcn_mfma_f64_16x16x4f64(c.y * wy, wx, acci, 0, 0, 0);
        }
        wave_lds_sync();                                  // slots and queue entries are free again
    };

    // this wave's chunks, row after row: chunk k of a row is wave (turn + k) % 4's
    int by = by0 - 1, base = 0, s1 = 0, turn = 0;
    auto advance = [&]() {
        base += kChunk * kSpreadWaves;
        while (base >= s1 && ++by <= by1) {
            const int s0 = __builtin_amdgcn_readlane(lo_l, by - by0);
            s1 = __builtin_amdgcn_readlane(hi_l, by - by0);
            base = s0 + kChunk * ((w - turn) & (kSpreadWaves - 1));
            turn += (s1 - s0 + kChunk - 1) / kChunk;
        }
    };
    auto fetch = [&]() {
        InRec v;
        v.xt = v.yt = 1e300;                              // reaches nothing
        v.re = v.im = 0.0;
        if (by <= by1 && base + lane < s1) v = pts[base + lane];
        return v;
    };
    advance();
    InRec cur = fetch();
    while (by <= by1) {
        advance();
        const InRec nxt = fetch();
        // the cell is the floor of these, as k3_prep found it
        const double vi = (double)(p.Mrx / 2) + cur.xt, vj = (double)(p.Mry / 2) + cur.yt;
        const bool in = vi >= ilo && vi < ihi && vj >= jlo && vj < jhi;
        const unsigned long long mask = __ballot(in);
        if (in) {
            const int pos = __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                                      __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
            L.q[n + pos] = cur;
        }
        n += __popcll(mask);
        wave_lds_sync();
        while (n >= kBatch) {
            n -= kBatch;
            batch(n);
        }
        cur = nxt;
    }
    if (n > 0) {                                          // the rest, zero samples behind it
        if (lane >= n && lane < kBatch) {
            InRec z;
            z.xt = (double)(i0 - p.Mrx / 2);
            z.yt = (double)(j0 - p.Mry / 2);
            z.re = z.im = 0.0;
            L.q[lane] = z;
        }
        wave_lds_sync();
        batch(0);
    }
    __syncthreads();   // every wave's slot reads are done: the partial tiles may overwrite them
#pragma unroll
    for (int q = 0; q < 4; ++q) sh.part[w][(4 * q + ks) * kTile + r] = make_double2(accr[q], acci[q]);
    __syncthreads();
    {
        const int cell = threadIdx.x, ii = i0 + cell % kTile, jj = j0 + cell / kTile;
        double sr = 0.0, si = 0.0;
#pragma unroll
        for (int ww = 0; ww < kSpreadWaves; ++ww) {   // fixed order
            const double2 v = sh.part[ww][cell];
            sr += v.x;
            si += v.y;
        }
        if (jj < p.gj + p.Py && ii < p.gi + p.Px) {
            const double ddi = (double)(ii - p.Mrx / 2), ddj = (double)(jj - p.Mry / 2);
            const double ri = (double)(ii - i0), rj = (double)(jj - j0);
            const double sc = p.fact * exp(p.b * (p.Dy * p.Dy * ddj * ddj) + p.b * (p.Dx * p.Dx * ddi * ddi)) *
                              exp(-p.t1 * (ri * ri + rj * rj));
            G[(size_t)(jj - p.gj) * p.Px + (ii - p.gi)] = make_double2(sr * sc, si * sc);
        }
    }
}
static_assert(64 * kSpreadWaves == kTile * kTile, "one cell per thread in the sum");

// ------------------------------------------------------------ 4. FFTs of the grid lines
// The convolution kernels' transforms in place, block 0 for x, 1 for y (a
// block whose side has another length leaves at once).
template <int LOGM>
__global__ __launch_bounds__((1 << LOGM) / 8) void k3_kernel_fft(AxisTables tx, AxisTables ty)
{
    extern __shared__ double2 X[];
    const AxisTables &t = blockIdx.x ? ty : tx;
    if (t.m != 1 << LOGM) return;
    constexpr int TPL = (1 << LOGM) / 8;
    const bool act[1] = {true};
    const int line[1] = {0}, j[1] = {(int)threadIdx.x};
    double2 v[1][8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[0][q] = t.hhat[j[0] + q * TPL];
    nfft2d::czt_fft<double, LOGM, 1>(v, X, t.tw, act, line, j, line, j, line, j);
#pragma unroll
    for (int q = 0; q < 8; ++q) t.hhat[j[0] + q * TPL] = v[0][q];
}

// ------------------------------------------------------------ 5. interpolation at the outputs
// Block per output bin (by, bx), 8 waves.  The patch of the spectrum for mm in
// [m0 - R, m0 + 16 + R), m0 = oj + 16 by, and nn likewise goes to LDS as
// P[c][a] (c = nn offset, a = mm offset, W = 16 + 2 R per side; entries past
// the read frequencies are loaded from the edge and never weighted).  The
// outputs of the bin come sorted by 8 x 2-cell blocks.  A wave takes 16 of
// them at a time and contracts, for each output j, H_j[a] = sum_c P[c][a]
// ex_j[c] on v_mfma_f64_16x16x4f64 (A[a][k] = P[c0 + k][a0 + a] from LDS,
// B[k][j] = ex_j[c0 + k], accumulator element q of lane l = H_{l % 16}[a0 + 4 q
// + l / 16]) over the rows and columns that the 16 windows cover, then
// F_j = sum_a ey_j[a] H_j[a] and the post-compensation.  The taps follow
// e^{-t1 (d - c - 4)^2} = e^{-t1 (d - c)^2} rho_c, rho_{c+4} = rho_c e^{-32 t1}
// along both c and a (two multiplications per step).
// Bound by FP64 arithmetic, most of it two 64-cycle products per 16 rows, 4
// columns and 16 outputs.  Outputs sorted by rows covered 54 columns a group,
// sorted by blocks about 41.  300,000 outputs, msp 19: 136 us; by blocks, with
// recurrences along both sides and the compensation in k3_prep 96, without the
// masks 81, with R = 16 69.
// MASK as in the spread: past its window an output's tails are below 2^-54 of
// its largest tap.
constexpr int kInterpWaves = 8;

// Minimum over the 16 lanes of a row.
__device__ __forceinline__ int row_min(int v)
{
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xf, 0xf, false));    // lanes 1 0 3 2
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xf, 0xf, false));    // lanes 2 3 0 1
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xf, 0xf, false));   // mirrored in 8
    return min(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xf, 0xf, false));   // mirrored in 16
}

template <bool MASK>
__global__ __launch_bounds__(64 * kInterpWaves) void k3_interp(const double2 *__restrict__ S,
                                                                const OutRec *__restrict__ outs,
                                                                const int *__restrict__ st,
                                                                const int *__restrict__ tot, Par p,
                                                                double2 *__restrict__ F)
{
    extern __shared__ double2 P[];
    const int bin = blockIdx.x;
    const int s0 = key_start(st, tot, bin * kTile), s1 = key_start(st, tot, bin * kTile + kTile);   // its 16 keys
    if (s0 == s1) return;
    const int bx = bin % p.nbx, by = bin / p.nbx;
    const int R = p.reach, W = kTile + 2 * R, taps = 2 * R + 1;
    const int mm0 = p.oj + by * kTile - R, nn0 = p.oi + bx * kTile - R;
    // S[i][j]: frequency qi + i, qj + j; cell nn is frequency nn - Mrx/2
    for (int e = threadIdx.x; e < W * W; e += 64 * kInterpWaves) {
        const int a = e % W, c = e / W;   // a: mm offset (contiguous in S), c: nn offset
        int i = nn0 + c - p.Mrx / 2 - p.qi, j = mm0 + a - p.Mry / 2 - p.qj;
        i = i >= p.Qx && p.Qx == p.Mrx ? i - p.Mrx : i;   // the whole side is held: periodic
        j = j >= p.Qy && p.Qy == p.Mry ? j - p.Mry : j;
        P[c * W + a] = S[(size_t)min(i, p.Qx - 1) * p.Qy + min(j, p.Qy - 1)];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int jo = lane & 15, kq = lane >> 4;
    const double kappa = exp(-32.0 * p.t1);
    for (int g = s0 + kTile * w; g < s1; g += kTile * kInterpWaves) {
        const int o = g + jo;
        const bool valid = o < s1;
        const OutRec rec = outs[valid ? o : s1 - 1];
        const int ra = rec.ntn - R - mm0, ca = rec.nsn - R - nn0;   // window origin in the patch, in [0, 16)
        const int rlo = row_min(valid ? ra : 1 << 20), rhi = taps - 1 - row_min(valid ? -ra : 1 << 20);
        const int clo = row_min(valid ? ca : 1 << 20), chi = taps - 1 - row_min(valid ? -ca : 1 << 20);
        const double dxc = rec.difs + ca + R;   // ex_j[c] = e^{-t1 (dxc - c)^2} on c in [ca, ca + 2 R]
        const double dya = rec.dift + ra + R;   // ey_j[a] = e^{-t1 (dya - a)^2} on a in [ra, ra + 2 R]
        // columns cs .. cs + 4 steps - 1 cover clo .. chi and end inside the patch; where they begin before it
        // (W not a multiple of 4), the entries before column 0 are column 0's and weigh nothing
        const int steps = (chi - clo + 4) / 4, cs = min(clo, W - 4 * steps);
        const double dc = dxc - (double)(cs + kq), da = dya - (double)(rlo + kq);
        const double ev0 = exp(-p.t1 * (dc * dc)), rho0 = exp(8.0 * p.t1 * dc - 16.0 * p.t1);
        double ey = exp(-p.t1 * (da * da)), sig = exp(8.0 * p.t1 * da - 16.0 * p.t1);
        double sr = 0.0, si = 0.0;
        for (int a0 = rlo; a0 <= rhi; a0 += 16) {
            d4 hr = {0.0, 0.0, 0.0, 0.0}, hi = {0.0, 0.0, 0.0, 0.0};
            const double2 *col = P + min(a0 + jo, W - 1);             // rows past W: never weighted
            double ev = ev0, rho = rho0;
            int c = cs + kq;
            col += max(c, 0) * W;
            auto step = [&](const double2 av) {
                const double bv = !MASK || (c >= ca && c < ca + taps) ? ev : 0.0;
                hr = __builtin_amdgcn_mfma_f64_16x16x4f64(av.x, bv, hr, 0, 0, 0);
                hi = __builtin_amdgcn_mfma_f64_16x16x4f64(av.y, bv, hi, 0, 0, 0);
                c += 4;
                ev *= rho;
                rho *= kappa;
            };
            step(*col);
            col = P + min(a0 + jo, W - 1) + c * W;                    // c >= 0 from the second step on
#pragma unroll 4
            for (int k = 1; k < steps; ++k) {
                step(*col);
                col += 4 * W;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int a = a0 + 4 * q + kq;
                const double wy = a >= ra && a < ra + taps ? ey : 0.0;
                sr = fma(wy, hr[q], sr);
                si = fma(wy, hi[q], si);
                ey *= sig;
                sig *= kappa;
            }
        }
        sr += __shfl_xor(sr, 16, 64);
        si += __shfl_xor(si, 16, 64);
        sr += __shfl_xor(sr, 32, 64);
        si += __shfl_xor(si, 32, 64);
        if (kq == 0 && valid)
            F[rec.idx] = make_double2(sr * rec.pr + si * rec.pi, si * rec.pr - sr * rec.pi);
    }
}

}  // namespace nufft3

using namespace nufft3;

// ============================================================== host side
namespace {

constexpr double kPi3 = 3.141592653589793238462643383279502884;

bool is_pow2(int n) { return n > 0 && (n & (n - 1)) == 0; }
int next_pow2(int n)
{
    int m = 1;
    while (m < n) m <<= 1;
    return m;
}
int fft_len(int n) { return is_pow2(n) ? n : next_pow2(2 * n - 1); }

// NUFFT_2D_CPU's parameters from the extents (:214-267), in its order of
// operations.  ext: max/min of x, y, s, t.
#pragma clang fp contract(off)
void derive(const double *ext, double eps, double *out)
{
    double Mx = ext[0], mx = ext[1], My = ext[2], my = ext[3];
    double Ms = ext[4], ms = ext[5], Mt = ext[6], mt = ext[7];
    double xb = (Mx + mx) / 2, X1 = fabs(Mx - xb);
    double yb = (My + my) / 2, Y1 = fabs(My - yb);
    double sb = (Ms + ms) / 2, S = fabs(Ms - sb);
    double tb = (Mt + mt) / 2, T = fabs(Mt - tb);
    const double R = 2.2;
    double msp = 2 + 2 * (R * R) * (-log(eps / 76)) / (kPi3 * (R * R - 2));
    const double mrx = 2 * ceil((X1 * S / kPi3) * R * R + R * msp);
    const double mry = 2 * ceil((Y1 * T / kPi3) * R * R + R * msp);
    double kkx = X1 / (kPi3 / 2), kky = Y1 / (kPi3 / 2);
    Mx /= kkx; mx /= kkx; xb = (Mx + mx) / 2;
    Ms *= kkx; ms *= kkx; sb = (Ms + ms) / 2;
    My /= kky; my /= kky; yb = (My + my) / 2;
    Mt *= kky; mt *= kky; tb = (Mt + mt) / 2;
    const double b = (msp - 2) / (4 * kPi3), t1 = 1 / (4 * b);
    msp = floor(msp - 2);
    double fact = 1. / (4. * kPi3 * b);
    out[0] = xb; out[1] = yb; out[2] = sb; out[3] = tb; out[4] = kkx; out[5] = kky;
    out[6] = 2 * kPi3 / mrx; out[7] = 2 * kPi3 / mry; out[8] = b; out[9] = t1; out[10] = fact * fact;
    out[11] = msp; out[12] = mrx; out[13] = mry;
}
#pragma clang fp contract(on)

// Cells that the coordinates between mn and mx fall into, first and count,
// inside a side of M.  cell(v) must be k3_prep's own operations: each is
// monotone in v, rounding included, so the extremes' cells bound all others.
#pragma clang fp contract(off)
template <typename Cell>
void cell_range(double mn, double mx, int M, Cell cell, int &first, int &count)
{
    const double lo = std::min(std::max(cell(mn), 0.0), M - 1.0), hi = std::min(std::max(cell(mx), lo), M - 1.0);
    first = (int)lo;
    count = (int)hi - (int)lo + 1;
}
void in_cells(double mn, double mx, double kk, double base, double D, int M, int &first, int &count)
{
    auto cell = [&](double v) {
        const double u = v / kk;
        const double o = (u - base) / D;
        return std::floor((double)(M / 2) + o);
    };
    cell_range(mn, mx, M, cell, first, count);
}
void out_cells(double mn, double mx, double kk, double base, int M, int &first, int &count)
{
    auto cell = [&](double v) {
        const double u = v * kk;
        const double o = u - base;
        return std::floor((double)(M / 2) + o);
    };
    cell_range(mn, mx, M, cell, first, count);
}
#pragma clang fp contract(on)

// Taps per side that change a sum: at distance d a Gaussian factor is
// e^{-t1 d^2} of its point's largest, below 2^-58 beyond d = sqrt(58 ln 2 / t1),
// where msp (the reference's, chosen for eps at the grid's band edge) goes on:
// msp 19 -> 16, 27 -> 19, 34 -> 22.  Each side's work falls with the square of
// (2 R + 16).
int tap_reach(int msp, double t1)
{
    const double d = std::ceil(std::sqrt(58.0 * 0.69314718055994531 / t1));
    return d < msp ? (int)d : msp;
}

struct Workspace {
    unsigned char *ptr = nullptr;
    size_t size = 0;
};
std::mutex g_mu;
std::map<int, Workspace> g_ws;
double *g_ext = nullptr;   // pinned: the nine extents of the running call and its number (under g_mu)
double g_call = 0.0;

int ensure(Workspace &ws, size_t bytes)
{
    if (ws.size >= bytes) return NFFT2D_OK;
    if (ws.ptr) {
        (void)hipDeviceSynchronize();
        (void)hipFree(ws.ptr);
        ws.ptr = nullptr;
        ws.size = 0;
    }
    const size_t want = bytes + bytes / 4;
    if (nfft2d_malloc(&ws.ptr, want) != hipSuccess) {
        (void)hipGetLastError();
        ws.ptr = nullptr;
        return nfft2d_fail(NFFT2D_ERR_ALLOC, "type-3 workspace of %zu bytes", want);
    }
    ws.size = want;
    return NFFT2D_OK;
}

size_t al(size_t b) { return (b + 255) & ~(size_t)255; }

struct Carve {
    unsigned char *base;
    size_t off = 0;
    template <typename T>
    T *take(size_t n)
    {
        T *p = reinterpret_cast<T *>(base + off);
        off += al(n * sizeof(T));
        return p;
    }
};

int check_args(const void *x, const void *y, const void *s, const void *t, const void *f, const void *F,
               double eps, int len_in, int len_out)
{
    if (len_in < 0 || len_out < 0) return nfft2d_fail(NFFT2D_ERR_ARG, "len_in = %d, len_out = %d", len_in, len_out);
    if (len_in > kMaxPoints || len_out > kMaxPoints)
        return nfft2d_fail(NFFT2D_ERR_ARG, "at most %d inputs and outputs", kMaxPoints);
    if (!(eps > 0.0 && eps < 1.0)) return nfft2d_fail(NFFT2D_ERR_ARG, "eps = %g: 0 < eps < 1 required", eps);
    if (len_out > 0 && (!s || !t || !F)) return nfft2d_fail(NFFT2D_ERR_ARG, "null output-side pointer");
    if (len_in > 0 && (!x || !y || !f)) return nfft2d_fail(NFFT2D_ERR_ARG, "null input-side pointer");
    return NFFT2D_OK;
}

// Extents on the device, parameters on the host; ext[9] as k3_extent_final
// leaves them, out[14] as orc_nufft3_params.
int params(Workspace &ws, const double *x, const double *y, const double *s, const double *t, double eps,
           int len_in, int len_out, double *ext, double *out)
{
    const int L = std::max(len_in, len_out);
    const int nblk = std::max(1, std::min(kExtentBlocks, (L + 255) / 256));
    int rc = ensure(ws, al(sizeof(double) * 9 * kExtentBlocks));
    if (rc) return rc;
    if (!g_ext && hipHostMalloc((void **)&g_ext, sizeof(double) * 10, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        g_ext = nullptr;
        return nfft2d_fail(NFFT2D_ERR_ALLOC, "type-3: pinned buffer of the extents");
    }
    if (g_call == 0.0) g_ext[9] = 0.0;
    g_call += 1.0;
    double *part = reinterpret_cast<double *>(ws.ptr), *fin = nullptr;
    NFFT2D_HIP_TRY(hipHostGetDevicePointer((void **)&fin, g_ext, 0));
    hipLaunchKernelGGL(k3_extent, dim3(nblk), dim3(256), 0, nullptr, x, y, s, t, len_in, len_out, part);
    NFFT2D_LAUNCH_CHECK();
    hipLaunchKernelGGL(k3_extent_final, dim3(1), dim3(64 * 9), 0, nullptr, part, nblk, g_call, fin);
    NFFT2D_LAUNCH_CHECK();
    // poll for at most a millisecond (longer work ahead on the stream, or an error, goes to the runtime)
    const auto t0 = std::chrono::steady_clock::now();
    while (__atomic_load_n(reinterpret_cast<const unsigned long long *>(g_ext + 9), __ATOMIC_ACQUIRE) !=
           __builtin_bit_cast(unsigned long long, g_call)) {
        if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(1)) {
            NFFT2D_HIP_TRY(hipStreamSynchronize(nullptr));
            break;
        }
    }
    for (int q = 0; q < 9; ++q) ext[q] = g_ext[q];
    if (ext[8] != 0.0) return nfft2d_fail(NFFT2D_ERR_ARG, "a coordinate is not finite");
    if (!(ext[0] > ext[1]) || !(ext[2] > ext[3]))
        return nfft2d_fail(NFFT2D_ERR_ARG,
                           "the inputs span no extent in x or y (all equal): the type-3 scaling divides by it");
    derive(ext, eps, out);
    return NFFT2D_OK;
}

template <int LOGM>
int kernel_fft(int m, const AxisTables &tx, const AxisTables &ty, hipStream_t st)
{
    if (m == 1 << LOGM) {
        constexpr int bytes = (int)sizeof(double2) * nfft2d::lds_line<1 << LOGM>();
        NFFT2D_HIP_TRY(hipFuncSetAttribute((const void *)k3_kernel_fft<LOGM>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
        hipLaunchKernelGGL(k3_kernel_fft<LOGM>, dim3(2), dim3(m / 8), bytes, st, tx, ty);
        NFFT2D_LAUNCH_CHECK();
        return NFFT2D_OK;
    }
    if constexpr (LOGM < nfft2d::kCztMaxLog<double>) return kernel_fft<LOGM + 1>(m, tx, ty, st);
    return nfft2d_fail(NFFT2D_ERR_SIZE, "no chirp-z transform of %d points", m);
}

nfft2d::CztTables<double> lines_of(const AxisTables &t)
{
    nfft2d::CztTables<double> c;
    c.cin = t.cin;
    c.cout = t.cout;
    c.hhat = t.hhat;
    c.tw = t.tw;
    c.P = t.P;
    c.Q = t.Q;
    c.m = t.m;
    return c;
}

int run(const double *x, const double *y, const double *s, const double *t, const nfft2d_c128 *f,
        nfft2d_c128 *F, double eps, int len_in, int len_out)
{
    int rc = check_args(x, y, s, t, f, F, eps, len_in, len_out);
    if (rc) return rc;
    if (len_out == 0) return NFFT2D_OK;
    if (len_in == 0) {   // the empty sum
        NFFT2D_HIP_TRY(hipMemsetAsync(F, 0, sizeof(nfft2d_c128) * (size_t)len_out, nullptr));
        return NFFT2D_OK;
    }
    std::lock_guard<std::mutex> lk(g_mu);
    int dev = 0;
    NFFT2D_HIP_TRY(hipGetDevice(&dev));
    Workspace &ws = g_ws[dev];
    double ext[9], pv[14];
    if ((rc = params(ws, x, y, s, t, eps, len_in, len_out, ext, pv))) return rc;
    if (!(pv[12] <= kMaxFft && pv[13] <= kMaxFft))
        return nfft2d_fail(NFFT2D_ERR_SIZE,
                           "grid %.0f x %.0f (Mrx x Mry): at most 4096 (8192 for powers of two) per side; reduce the "
                           "products of the extents X1 S and Y1 T",
                           pv[12], pv[13]);
    Par p;
    p.xb = pv[0]; p.yb = pv[1]; p.sb = pv[2]; p.tb = pv[3]; p.kkx = pv[4]; p.kky = pv[5];
    p.Dx = pv[6]; p.Dy = pv[7]; p.b = pv[8]; p.t1 = pv[9]; p.fact = pv[10];
    p.Mrx = (int)pv[12]; p.Mry = (int)pv[13];
    const int msp = (int)pv[11];
    if (msp < 0 || msp > kMaxMsp)
        return nfft2d_fail(NFFT2D_ERR_SIZE, "eps = %g gives %d taps per side; at most %d (eps >= ~1e-14)", eps, msp,
                           kMaxMsp);
    p.reach = tap_reach(msp, p.t1);
    const bool mask = !(p.t1 * p.reach * p.reach > 54.0 * 0.69314718055994531);   // tails of 2^-54 and more
    if (fft_len(p.Mrx) > kMaxFft || fft_len(p.Mry) > kMaxFft)
        return nfft2d_fail(NFFT2D_ERR_SIZE,
                           "grid %d x %d (Mrx x Mry) needs FFTs of %d and %d points; at most %d (Mrx, Mry <= 4096, "
                           "or 8192 for powers of two): reduce the products of the extents X1 S and Y1 T",
                           p.Mrx, p.Mry, fft_len(p.Mrx), fft_len(p.Mry), kMaxFft);
    // the reached part of the grid and the read part of the spectrum
    in_cells(ext[1], ext[0], p.kkx, p.xb, p.Dx, p.Mrx, p.ci, p.ni);
    in_cells(ext[3], ext[2], p.kky, p.yb, p.Dy, p.Mry, p.cj, p.nj);
    out_cells(ext[5], ext[4], p.kkx, p.sb, p.Mrx, p.oi, p.mi);
    out_cells(ext[7], ext[6], p.kky, p.tb, p.Mry, p.oj, p.mj);
    p.gi = std::max(0, p.ci - p.reach);
    p.gj = std::max(0, p.cj - p.reach);
    p.Px = std::min(p.Mrx, p.ci + p.ni + p.reach) - p.gi;
    p.Py = std::min(p.Mry, p.cj + p.nj + p.reach) - p.gj;
    p.qi = p.oi - p.reach - p.Mrx / 2;
    p.qj = p.oj - p.reach - p.Mry / 2;
    p.Qx = std::min(p.mi + 2 * p.reach, p.Mrx);
    p.Qy = std::min(p.mj + 2 * p.reach, p.Mry);
    const int mx = std::max(1 << nfft2d::kCztMinLog, next_pow2(p.Px + p.Qx - 1));
    const int my = std::max(1 << nfft2d::kCztMinLog, next_pow2(p.Py + p.Qy - 1));
    if (mx > kMaxFft || my > kMaxFft)   // only coordinates rounded far off their cells (huge offsets) get here
        return nfft2d_fail(NFFT2D_ERR_SIZE, "grid %d x %d (Mrx x Mry): the inputs reach %d x %d cells", p.Mrx, p.Mry,
                           p.Px, p.Py);
    p.nbx = (p.mi + kTile - 1) / kTile;
    p.nby = (p.mj + kTile - 1) / kTile;
    p.ibx = (p.ni + kInBin - 1) / kInBin;
    p.iby = (p.nj + kInBin - 1) / kInBin;
    const int nbo = p.nbx * p.nby;                              // output bins
    const int nki = p.ibx * p.iby + 1, nko = nbo * kTile + 1;   // keys, the out-of-grid ones last
    ScanSide a, b;
    a.n = nki;
    b.n = nko;
    a.segs = (nki + 1023) / 1024;
    b.segs = (nko + 1023) / 1024;

    // workspace: counts, starts, records, the grid parts, the chirp-z tables
    const size_t cells = (size_t)p.Px * p.Py, mixed = (size_t)p.Qx * p.Py, spec = (size_t)p.Qx * p.Qy;
    size_t need = 0;
    {
        const size_t sz[] = {(al(sizeof(int) * nki) + al(sizeof(int) * nko)) * 2,
                             al(sizeof(int) * a.segs) + al(sizeof(int) * b.segs),
                             al(sizeof(InRec) * len_in) * 2, al(sizeof(int2) * len_in),
                             al(sizeof(OutRec) * len_out) * 2, al(sizeof(int2) * len_out),
                             al(sizeof(double2) * cells) + al(sizeof(double2) * mixed) + al(sizeof(double2) * spec),
                             al(sizeof(double2) * mx) * 2 + al(sizeof(double2) * p.Px) + al(sizeof(double2) * p.Qx),
                             al(sizeof(double2) * my) * 2 + al(sizeof(double2) * p.Py) + al(sizeof(double2) * p.Qy)};
        for (size_t v : sz) need += v;
    }
    if ((rc = ensure(ws, need))) return rc;
    Carve cv{ws.ptr};
    a.cnt = cv.take<int>(nki);
    b.cnt = cv.take<int>(nko);
    a.start = cv.take<int>(nki);
    b.start = cv.take<int>(nko);
    a.tot = cv.take<int>(a.segs);
    b.tot = cv.take<int>(b.segs);
    InRec *rin = cv.take<InRec>(len_in), *sin_ = cv.take<InRec>(len_in);
    int2 *kin = cv.take<int2>(len_in);
    OutRec *rout = cv.take<OutRec>(len_out), *sout = cv.take<OutRec>(len_out);
    int2 *kout = cv.take<int2>(len_out);
    double2 *G = cv.take<double2>(cells), *T = cv.take<double2>(mixed), *S = cv.take<double2>(spec);
    auto axis = [&](int n, int P, int Q, int p0, int q0, int m) {
        AxisTables t;
        t.cin = cv.take<double2>(P);
        t.cout = cv.take<double2>(Q);
        t.hhat = cv.take<double2>(m);
        t.tw = cv.take<double2>(m);
        t.n = n; t.P = P; t.Q = Q; t.p0 = p0; t.q0 = q0; t.m = m;
        return t;
    };
    const AxisTables tx = axis(p.Mrx, p.Px, p.Qx, p.gi, p.qi, mx), ty = axis(p.Mry, p.Py, p.Qy, p.gj, p.qj, my);

    hipStream_t st = nullptr;
    NFFT2D_HIP_TRY(hipMemsetAsync(a.cnt, 0, al(sizeof(int) * nki) + al(sizeof(int) * nko), st));
    const int gin = (len_in + 255) / 256, gout = (len_out + 255) / 256;
    hipLaunchKernelGGL(k3_prep, dim3(gin + gout), dim3(256), 0, st, x, y, reinterpret_cast<const double2 *>(f), len_in,
                       gin, p, rin, kin, a.cnt, s, t, len_out, rout, kout, b.cnt, reinterpret_cast<double2 *>(F));
    NFFT2D_LAUNCH_CHECK();
    hipLaunchKernelGGL(k3_scan_local, dim3(a.segs + b.segs + (std::max(mx, my) + 1023) / 1024), dim3(1024), 0, st, a, b,
                       tx, ty);
    NFFT2D_LAUNCH_CHECK();
    hipLaunchKernelGGL(k3_scan_totals, dim3(2), dim3(1024), 0, st, a, b);
    NFFT2D_LAUNCH_CHECK();
    if ((rc = kernel_fft<nfft2d::kCztMinLog>(mx, tx, ty, st))) return rc;
    if (my != mx && (rc = kernel_fft<nfft2d::kCztMinLog>(my, tx, ty, st))) return rc;
    hipLaunchKernelGGL(k3_scatter, dim3(gin + gout), dim3(256), 0, st, rin, kin, len_in, gin, a, sin_, rout, kout,
                       len_out, b, sout);
    NFFT2D_LAUNCH_CHECK();

    // spread
    const int ntx = (p.Px + kTile - 1) / kTile, nty = (p.Py + kTile - 1) / kTile;
    hipLaunchKernelGGL((mask ? k3_spread<true> : k3_spread<false>), dim3(ntx * nty),
                       dim3(64 * kSpreadWaves), 0, st, sin_, a.start, a.tot, p, ntx, G);
    NFFT2D_LAUNCH_CHECK();

    // 2-D DFT: G's rows (j) to the read x frequencies, written side by side: T[qi][j]; then T's rows: S[qi][qj]
    const double *none = nullptr;
    if ((rc = nfft2d::czt_launch<double, 2>(lines_of(tx), p.Py, (const double2 *)G, p.Px, 1, T, 1, p.Py, none, none,
                                            false, false, st)))
        return rc;
    if ((rc = nfft2d::czt_launch<double, 0>(lines_of(ty), p.Qx, (const double2 *)T, p.Py, 1, S, p.Qy, 1, none, none,
                                            false, false, st)))
        return rc;

    // interpolation at the outputs
    const int W = kTile + 2 * p.reach;
    const size_t lds = sizeof(double2) * (size_t)W * W;
    auto interp = mask ? k3_interp<true> : k3_interp<false>;
    NFFT2D_HIP_TRY(hipFuncSetAttribute((const void *)interp, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(interp, dim3(nbo), dim3(64 * kInterpWaves), lds, st, S, sout, b.start, b.tot, p,
                       reinterpret_cast<double2 *>(F));
    NFFT2D_LAUNCH_CHECK();
    return NFFT2D_OK;
}

}  // namespace

extern "C" int NUFFT_2D_GPU(const double *x, const double *y, const double *s, const double *t,
                            const nfft2d_c128 *f, nfft2d_c128 *F, double eps, int len_in, int len_out)
{
    return run(x, y, s, t, f, F, eps, len_in, len_out);
}

extern "C" int NUFFT_2D_GPU_params(const double *x, const double *y, const double *s, const double *t, double eps,
                                   int len_in, int len_out, double *out)
{
    int rc = check_args(x, y, s, t, (const void *)1, (const void *)1, eps, len_in, len_out);
    if (rc) return rc;
    if (!out) return nfft2d_fail(NFFT2D_ERR_ARG, "null output array");
    if (len_in == 0 || len_out == 0) return nfft2d_fail(NFFT2D_ERR_ARG, "no inputs or no outputs");
    std::lock_guard<std::mutex> lk(g_mu);
    int dev = 0;
    NFFT2D_HIP_TRY(hipGetDevice(&dev));
    double ext[9];
    return params(g_ws[dev], x, y, s, t, eps, len_in, len_out, ext, out);
}

extern "C" int NUFFT_2D_GPU_host(const double *x, const double *y, const double *s, const double *t,
                                 const nfft2d_c128 *f, nfft2d_c128 *F, double eps, int len_in, int len_out)
{
    int rc = check_args(x, y, s, t, f, F, eps, len_in, len_out);
    if (rc) return rc;
    if (len_out == 0) return NFFT2D_OK;
    const size_t ni = (size_t)len_in, no = (size_t)len_out;
    void *buf = nullptr;
    const size_t bytes = al(16 * ni) + al(16 * ni) + al(16 * no) * 2;
    if (nfft2d_malloc(&buf, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return nfft2d_fail(NFFT2D_ERR_ALLOC, "NUFFT_2D_GPU_host: %zu bytes", bytes);
    }
    unsigned char *b = static_cast<unsigned char *>(buf);
    double *dx = reinterpret_cast<double *>(b), *dy = dx + ni;
    nfft2d_c128 *df = reinterpret_cast<nfft2d_c128 *>(b + al(16 * ni));
    double *ds = reinterpret_cast<double *>(b + al(16 * ni) * 2), *dt = ds + no;
    nfft2d_c128 *dF = reinterpret_cast<nfft2d_c128 *>(b + al(16 * ni) * 2 + al(16 * no));
    hipError_t e = hipSuccess;
    if (ni) {
        if (e == hipSuccess) e = hipMemcpy(dx, x, 8 * ni, hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMemcpy(dy, y, 8 * ni, hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMemcpy(df, f, 16 * ni, hipMemcpyHostToDevice);
    }
    if (e == hipSuccess) e = hipMemcpy(ds, s, 8 * no, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dt, t, 8 * no, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(buf);
        return nfft2d_fail(NFFT2D_ERR_HIP, "NUFFT_2D_GPU_host: copy in: %s", hipGetErrorString(e));
    }
    rc = run(ni ? dx : nullptr, ni ? dy : nullptr, ds, dt, ni ? df : nullptr, dF, eps, len_in, len_out);
    if (rc == NFFT2D_OK) {
        e = hipMemcpy(F, dF, 16 * no, hipMemcpyDeviceToHost);
        if (e != hipSuccess) rc = nfft2d_fail(NFFT2D_ERR_HIP, "NUFFT_2D_GPU_host: copy out: %s", hipGetErrorString(e));
    }
    (void)hipFree(buf);
    return rc;
}

// ndft2d.hip -- the 2D NDFT.  Part 1: NDFT2_2D_GPU, the reference's direct
// sum in FP64 (NFFT/NDFT2_2D.cu:15-32,37-72):
//   out[n] = sum_{m<M} in[m] exp(-2 pi i (u[n] X[m] / Nu + v[n] Y[m] / Nv)).
// The reference fills an explicit M x N FP64 kernel matrix (:44-50; 64 GiB at
// M = N = 65536), writes it to a text file (:56) and calls cublasZgemv (:67).
// Here nothing of that size is materialised: on the integer meshgrid the
// reference's caller passes, the sum is an FP64 complex GEMM on the matrix
// cores (k_ndft_grid + k_ndft_finish, with a cached workspace of at most 256
// partial output arrays); for other (u, v) each thread takes one output over a
// range of the points, accumulating in FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <new>

#include "../../include/nfft2d.h"
#include "ndft2d_mfma.hpp"
#include "nfft2d_internal.hpp"

namespace {

constexpr int kThreads = 256;

// ---------------------------------------------------------------------------
// Output grids.  The reference's only caller passes (u, v) = the integer
// meshgrid of the far-field plane (Synthesis/PSO/Synthesis.cu:85-90,397):
// N = nu nv outputs with u and v arithmetic progressions.  Then
//     out[i, j] = sum_m in_m e^{-2 pi i a_i X_m / Nu} e^{-2 pi i b_j Y_m / Nv},
//     a_i = u0 + i du, b_j = v0 + j dv,
// is the complex product (nu x M) . (M x nv) of two phasor matrices: a GEMM on
// the FP64 matrix cores instead of M N separate kernel evaluations.
// k_grid_detect recognises the two flattenings of such a grid (u constant
// over runs of nv outputs, or v constant over runs of nu) and k_grid_verify
// checks every output against it by exact FP64 comparison; the finding stays
// in g_grid (one per device, as every __device__ variable); k_ndft_grid takes
// the matrix cores when it is a grid and the direct sum (any u, v) when it is
// not.  It reads the flag on the device, so the call stays asynchronous and
// capturable.  Two NDFT2_2D_GPU calls that overlap on
// one device (different streams) race on g_grid.
struct GridInfo {
    int ok;          // 1: (u, v) is a grid of nu x nv outputs
    int vmajor;      // 0: n = i nv + j (u constant over runs of nv); 1: n = j nu + i
    int nu, nv;
    double u0, du, v0, dv;
};
__device__ GridInfo g_grid;

constexpr int kDetThreads = 1024;
__global__ __launch_bounds__(kDetThreads) void k_grid_detect(const double *__restrict__ u,
                                                             const double *__restrict__ v, int N)
{
    __shared__ int s_run[2];
    const int t = threadIdx.x;
    if (t == 0) {
        s_run[0] = N;
        s_run[1] = N;
    }
    __syncthreads();
    const double u0 = u[0], v0 = v[0];
    // first change of u and of v, block-wide over chunks of kDetThreads
    // outputs: each wave's first hit is the lowest set bit of its ballot, one
    // LDS atomic per wave and value takes the block's minimum, and the block
    // stops at the first chunk after which both are found (later chunks hold
    // only larger indices).  An atomic per element serialised on one address
    // (425 us at 65,536 outputs); threads scanning on their own until their
    // own first hits ran the whole array where a stride of kDetThreads never
    // meets a change (29 us on a 256 x 256 grid).
    const int lane = t & 63;
    for (int base = 1; base < N; base += kDetThreads) {
        const int n = base + t;
        const bool in = n < N;
        const unsigned long long bu = __ballot(in && u[n] != u0);
        const unsigned long long bv = __ballot(in && v[n] != v0);
        if (lane == 0) {   // n is the wave's first index
            if (bu) atomicMin(&s_run[0], n + __ffsll((long long)bu) - 1);
            if (bv) atomicMin(&s_run[1], n + __ffsll((long long)bv) - 1);
        }
        __syncthreads();
        const bool done = s_run[0] < N && s_run[1] < N;
        __syncthreads();   // every thread has read before the next chunk's atomics
        if (done) break;
    }
    const int ru = s_run[0], rv = s_run[1];
    // u-major: v changes at once and u after nv = ru outputs; v-major: the converse
    int vmajor = -1, nu = 1, nv = 1;
    if (N == 1) {
        vmajor = 0;
    } else if (rv == 1 && ru > 1 && N % ru == 0) {
        vmajor = 0;
        nv = ru;
        nu = N / ru;
    } else if (ru == 1 && rv > 1 && N % rv == 0) {
        vmajor = 1;
        nu = rv;
        nv = N / rv;
    }
    double du = 0.0, dv = 0.0;
    if (vmajor == 0) {
        du = nu > 1 ? u[nv] - u0 : 0.0;
        dv = nv > 1 ? v[1] - v0 : 0.0;
    } else if (vmajor == 1) {
        du = nu > 1 ? u[1] - u0 : 0.0;
        dv = nv > 1 ? v[nu] - v0 : 0.0;
    }
    // every output is then checked against the grid by k_grid_verify (all of
    // the chip: one block's loop over N outputs took 76 us at N = 65,536)
    if (t == 0) {
        GridInfo g;
        g.ok = vmajor >= 0 && nu * nv == N;
        g.vmajor = vmajor > 0;
        g.nu = nu;
        g.nv = nv;
        g.u0 = u0;
        g.du = du;
        g.v0 = v0;
        g.dv = dv;
        g_grid = g;
    }
}

__device__ __forceinline__ double2 phasor(double t)   // e^{-2 pi i t}
{
    t -= floor(t);
    double s, c;
    sincospi(2.0 * t, &s, &c);
    return make_double2(c, -s);
}

__device__ __forceinline__ double2 zmul(double2 a, double2 b)
{
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// One point of the grid case: its sample times the phasor of the grid's
// centre, its 16-row and 16-column phasor steps, and X / Nu, Y / Nv.
struct alignas(16) GridPt {
    double2 d, step[2];
    double xy[2];
};

// Two independent jobs on the detector's finding.  Blocks below nver clear
// g_grid.ok when an output is not the grid's: u[n] = u0 + i du and v[n] =
// v0 + j dv, exactly, for n's (i, j) in the detected flattening.  The others
// prepare the points (what they write is unused when the check fails).
__global__ __launch_bounds__(kThreads) void k_grid_verify(const double *__restrict__ u, const double *__restrict__ v,
                                                          int N, int nver, const double *__restrict__ X,
                                                          const double *__restrict__ Y,
                                                          const double2 *__restrict__ in, double inv_Nu,
                                                          double inv_Nv, int M, GridPt *__restrict__ pts)
{
    const GridInfo g = g_grid;
    if (!g.ok) return;
    if ((int)blockIdx.x < nver) {
        const int n = blockIdx.x * kThreads + threadIdx.x;
        if (n >= N) return;
        const int i = g.vmajor ? n % g.nu : n / g.nv, j = g.vmajor ? n / g.nu : n % g.nv;
        if (u[n] != g.u0 + i * g.du || v[n] != g.v0 + j * g.dv) g_grid.ok = 0;
        return;
    }
    const int m = (blockIdx.x - nver) * kThreads + threadIdx.x;
    if (m >= M) return;
    const double xm = X[m] * inv_Nu, ym = Y[m] * inv_Nv;
    const double uc = g.u0 + 0.5 * (g.nu - 1) * g.du, vc = g.v0 + 0.5 * (g.nv - 1) * g.dv;
    GridPt p;
    p.d = zmul(zmul(in[m], phasor(uc * xm)), phasor(vc * ym));
    p.step[0] = phasor(16.0 * g.du * xm);
    p.step[1] = phasor(16.0 * g.dv * ym);
    p.xy[0] = xm;
    p.xy[1] = ym;
    pts[m] = p;
}

// The grid case by conjugate pairs.  About the grid's centre (uc, vc) its rows
// are uc +- delta_p, delta_p = (p + 1/2) du (nu even) or p du (nu odd), and so
// are its columns, so with d_m the sample times the centre's phasor
//     out[uc + s1 delta1, vc + s2 delta2] = sum_m d_m (c1 + i s1 t1) (c2 + i s2 t2),
//     (c, t) = (cos, -sin) of the pair's phase, s1, s2 = +-1,
// are four combinations of the real-phasor sums CC = sum d c1 c2, TC = sum d
// t1 c2, CT and TT: 8 real products per 4 outputs and point, half of a complex
// product for every output.
//
// Products on v_mfma_f64_16x16x4f64 (4 points per instruction): lane l
// supplies A[i][k] at i = l % 16, k = l / 16 and B[k][j] at j = l % 16;
// accumulator element r of lane l is C[4 r + l / 16][l % 16].  A block takes a
// tile of 64 x 64 pairs (128 x 128 outputs) over one range of the points: wave
// w the 16 x 32 pairs of row tile w / 2, column tiles 2 (w % 2) and + 1 (16
// accumulator tiles, 128 VGPRs; 2 waves per SIMD); where only one row or column
// tile is in use, wave w < 4 its w-th (1 x 20,000 outputs from M = 65,536: 6.5 ->
// 3.8 ms; two waves of two tiles each left two SIMDs idle).  FP64 VALU work does
// not run under FP64 MFMAs, so the phasors are evaluated once per block: for a
// chunk of 16 points each of the 512 threads takes one (point, row or column
// index mod 16) by an FP64 phase reduction and sincospi, advances it three
// times by the point's 16-step phasor, and leaves the four in LDS (two
// buffers) while the previous chunk's products run.
// 256 x 256 outputs from M = 65,536: 0.30 ms a call, 0.22 at the FP64 matrix rate
// (one wave per 32 x 64 outputs with its own phasors and complex products: 0.69).
// The partial sums go to range r's slice of a workspace; k_ndft_finish adds
// the ranges in a fixed order (the result does not depend on the launch).
// Work items are walked persistently (their count is known on the device only).
constexpr int kTilePairs = 64;                    // pairs per block tile and dimension
constexpr int kGridThreads = 512;
constexpr int kGridBlocks = 256;                  // one per CU
constexpr int kGridChunk = 16;                    // points per LDS buffer
typedef double d4 __attribute__((ext_vector_type(4)));

// Any other (u, v): the direct sum, one output per thread over one range of the
// points (every thread of a block at the same point, so the point's values are
// scalar loads), the partial sums going the same way.  One thread per output
// over all points left most of the chip idle: 4,200 outputs from M = 4,000
// points, 656 us; in ranges 62 us.
__device__ __forceinline__ void direct_item(const double *__restrict__ X, const double *__restrict__ Y, double un,
                                            double vn, const double2 *__restrict__ in, int m_lo, int m_hi,
                                            double2 &acc)
{
    double ar = 0.0, ai = 0.0;
    auto add = [&](double xm, double ym, double2 d) {
        double t = un * xm + vn * ym;
        t -= floor(t);
        double s, c;
        sincospi(2.0 * t, &s, &c);   // e^{-2 pi i t} = c - i s
        ar += d.x * c + d.y * s;
        ai += d.y * c - d.x * s;
    };
    // 8 points' loads ahead of their sums (2 waves per SIMD hide little of a load's latency)
    constexpr int B = 8;
    int m = m_lo;
    for (; m + B <= m_hi; m += B) {
        double xm[B], ym[B];
        double2 d[B];
#pragma unroll
        for (int b = 0; b < B; ++b) {
            xm[b] = X[m + b];
            ym[b] = Y[m + b];
            d[b] = in[m + b];
        }
#pragma unroll
        for (int b = 0; b < B; ++b) add(xm[b], ym[b], d[b]);
    }
    for (; m < m_hi; ++m) add(X[m], Y[m], in[m]);
    acc = make_double2(ar, ai);
}

// Point ranges in use on a grid.  A thin grid has far more tiles than a square
// one of as many outputs, and every item has its fixed cost (its first chunk,
// its partial sums written and added): where the ranges given would be shorter
// than 16 chunks, no more than four items per block.
// Outputs 1 x 4,096 from M = 5,000, 32 tiles: 256 ranges 215 us, 32 120 (75 with
// one tile per wave); 1 x 20,000 1,001 -> 555 (328); 2 x 2,000 118 -> 68 (47).
__device__ __forceinline__ int grid_ranges(const GridInfo &g, int M, int ranges)
{
    const int tiles = ((g.nu + 1) / 2 + kTilePairs - 1) / kTilePairs * (((g.nv + 1) / 2 + kTilePairs - 1) / kTilePairs);
    return min(ranges, max(max(1, 4 * kGridBlocks / tiles), M / (16 * kGridChunk)));
}

__global__ __launch_bounds__(kGridThreads) void k_ndft_grid(const GridPt *__restrict__ pts,
                                                            double2 *__restrict__ part, int M, int ranges, int chunk,
                                                            const double *__restrict__ X, const double *__restrict__ Y,
                                                            const double *__restrict__ u, const double *__restrict__ v,
                                                            const double2 *__restrict__ in, double inv_Nu,
                                                            double inv_Nv, int nout)
{
    const GridInfo g = g_grid;
    if (!g.ok) {
        const long long nblk = ((long long)nout + kGridThreads - 1) / kGridThreads;
        for (long long item = blockIdx.x; item < nblk * ranges; item += gridDim.x) {
            const int r = (int)(item / nblk);
            const long long n = (item % nblk) * kGridThreads + threadIdx.x;
            const int m_lo = min(M, r * chunk), m_hi = min(M, m_lo + chunk);
            const bool have = n < nout;
            double2 acc;
            direct_item(X, Y, have ? u[n] * inv_Nu : 0.0, have ? v[n] * inv_Nv : 0.0, in, m_lo, m_hi, acc);
            if (have) part[(size_t)r * nout + n] = acc;
        }
        return;
    }
    __shared__ double2 s_ph[2][2][kGridChunk][kTilePairs];   // [buffer][row, column][point][pair]
    __shared__ double2 s_d[2][kGridChunk];
    const int t = threadIdx.x, lane = t & 63, q = lane & 15, k = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nu2 = (g.nu + 1) / 2, nv2 = (g.nv + 1) / 2;    // pairs (an odd length's centre is a pair of its own)
    const int tcols = (nv2 + kTilePairs - 1) / kTilePairs;
    ranges = grid_ranges(g, M, ranges);
    chunk = ((M + ranges - 1) / ranges + kGridChunk - 1) / kGridChunk * kGridChunk;
    const int items = (nu2 + kTilePairs - 1) / kTilePairs * tcols * ranges;
    const long long N = (long long)g.nu * g.nv;
    // phasor role of this thread: side, point of the chunk, index mod 16
    const int side = w >> 2, pt = (t >> 4) & 15, pq = t & 15;
    // rounds of one item per block; where a round spans tiles every other one goes
    // backwards, so that a block that took a whole tile's share gets an edge tile's next
    for (int i0 = 0, back = 0; i0 < items; i0 += gridDim.x, back ^= ranges < (int)gridDim.x) {
        const int item = i0 + (int)(back ? gridDim.x - 1 - blockIdx.x : blockIdx.x);
        if (item >= items) continue;
        const int r = item % ranges, st = item / ranges;
        const int p1 = (st / tcols) * kTilePairs, p2 = (st % tcols) * kTilePairs;   // first pairs of the tile
        const int m_lo = min(M, r * chunk), m_hi = min(M, m_lo + chunk);
        const double idx = side ? p2 + pq + (g.nv & 1 ? 0.0 : 0.5) : p1 + pq + (g.nu & 1 ? 0.0 : 0.5);
        const double off = idx * (side ? g.dv : g.du);
        // the tile's 16-pair rows and columns in use; a single one of either lies on
        // four waves of four SIMDs, not on two
        const int nrt = min(4, (nu2 - p1 + 15) / 16), nct = min(4, (nv2 - p2 + 15) / 16);
        const int rt = nrt == 1 ? 0 : nct == 1 ? w : w >> 1, ct = nrt == 1 ? w : nct == 1 ? 0 : 2 * (w & 1);
        const bool act0 = rt < nrt && ct < nct, act1 = nrt > 1 && rt < nrt && ct + 1 < nct;
        const int nst = side ? nct : nrt;
        struct Pt {
            double2 d, step;
            double x;
        };
        auto load = [&](int m) {
            Pt o;
            o.d = make_double2(0.0, 0.0);   // a point past the range adds nothing
            o.step = make_double2(1.0, 0.0);
            o.x = 0.0;
            if (m < m_hi) {
                const GridPt *p = pts + m;
                o.d = p->d;
                o.step = p->step[side];
                o.x = p->xy[side];
            }
            return o;
        };
        auto stage = [&](const Pt &p, int b) {
            double2 z = phasor(off * p.x);
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                if (h >= nst) break;
                if (h > 0) z = zmul(z, p.step);
                s_ph[b][side][pt][16 * h + pq] = z;
            }
            if (side == 0 && pq == 0) s_d[b][pt] = p.d;
        };
        // [column tile][CC, TC, CT, TT]
        d4 ar[2][4], ai[2][4];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) ar[c][e] = ai[c][e] = d4{0.0, 0.0, 0.0, 0.0};
        __syncthreads();                    // the previous item's reads are done
        stage(load(m_lo + pt), 0);
        Pt nxt = load(m_lo + kGridChunk + pt);
        __syncthreads();
        int b = 0;
        for (int m0 = m_lo; m0 < m_hi; m0 += kGridChunk, b ^= 1) {
            const Pt cur = nxt;
            nxt = load(m0 + 2 * kGridChunk + pt);
            if (m0 + kGridChunk < m_hi) stage(cur, b ^ 1);
            if (act0)
#pragma unroll
                for (int s = 0; s < kGridChunk / 4; ++s) {
                    const double2 d = s_d[b][4 * s + k], a = s_ph[b][0][4 * s + k][16 * rt + q];
                    const double cr = d.x * a.x, ci = d.y * a.x, tr = d.x * a.y, ti = d.y * a.y;
#pragma unroll
                    for (int c = 0; c < 2; ++c) {
                        if (c && !act1) continue;
                        const double2 v = s_ph[b][1][4 * s + k][16 * (ct + c) + q];
                        ar[c][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(cr, v.x, ar[c][0], 0, 0, 0);
                        ai[c][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(ci, v.x, ai[c][0], 0, 0, 0);
                        ar[c][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(tr, v.x, ar[c][1], 0, 0, 0);
                        ai[c][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(ti, v.x, ai[c][1], 0, 0, 0);
                        ar[c][2] = __builtin_amdgcn_mfma_f64_16x16x4f64(cr, v.y, ar[c][2], 0, 0, 0);
                        ai[c][2] = __builtin_amdgcn_mfma_f64_16x16x4f64(ci, v.y, ai[c][2], 0, 0, 0);
                        ar[c][3] = __builtin_amdgcn_mfma_f64_16x16x4f64(tr, v.y, ar[c][3], 0, 0, 0);
                        ai[c][3] = __builtin_amdgcn_mfma_f64_16x16x4f64(ti, v.y, ai[c][3], 0, 0, 0);
                    }
                }
            __syncthreads();
        }
        // the four outputs of each pair of pairs: rows nu / 2 + p and nu - 1 - (nu / 2 + p)
        double2 *dst = part + (size_t)r * N;
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (!(c ? act1 : act0)) continue;
                const int i = g.nu / 2 + p1 + 16 * rt + 4 * e + k, j = g.nv / 2 + p2 + 16 * (ct + c) + q;
                if (i >= g.nu || j >= g.nv) continue;
#pragma unroll
                for (int sg = 0; sg < 4; ++sg) {
                    const double s1 = sg & 2 ? -1.0 : 1.0, s2 = sg & 1 ? -1.0 : 1.0;
                    const double re = ar[c][0][e] - s1 * s2 * ar[c][3][e] - (s1 * ai[c][1][e] + s2 * ai[c][2][e]);
                    const double im = ai[c][0][e] - s1 * s2 * ai[c][3][e] + (s1 * ar[c][1][e] + s2 * ar[c][2][e]);
                    const int ii = sg & 2 ? g.nu - 1 - i : i, jj = sg & 1 ? g.nv - 1 - j : j;
                    dst[(size_t)ii * g.nv + jj] = make_double2(re, im);   // an odd length's centre: the same value twice
                }
            }
    }
}

// The partial sums' workspace, one per device, grown as needed (the
// drop-in's calls run on the null stream, so consecutive calls are ordered).
struct GridWs {
    double2 *ptr = nullptr;
    size_t count = 0;
};
std::mutex g_ws_mu;
std::map<int, GridWs> g_ws;

// out[n] = sum over the ranges (in a fixed order) of the partial sums, in the
// caller's flattening: 64 outputs per block, 4 threads each over every fourth
// range.
constexpr int kSumOut = 64;
__global__ __launch_bounds__(kThreads) void k_ndft_finish(const double2 *__restrict__ part, int M, int ranges,
                                                          double2 *__restrict__ out, int N)
{
    const GridInfo g = g_grid;
    __shared__ double2 s_sum[kThreads / kSumOut - 1][kSumOut];
    const int o = threadIdx.x % kSumOut, sl = threadIdx.x / kSumOut, n = blockIdx.x * kSumOut + o;
    double sr = 0.0, si = 0.0;
    if (n < N) {
        size_t e = n;
        if (g.ok) {
            const int i = g.vmajor ? n % g.nu : n / g.nv, j = g.vmajor ? n / g.nu : n % g.nv;
            e = (size_t)i * g.nv + j;
            ranges = grid_ranges(g, M, ranges);
        }
        const double2 *src = part + e;
#pragma unroll 4
        for (int r = sl; r < ranges; r += kThreads / kSumOut) {
            const double2 p = src[(size_t)r * N];
            sr += p.x;
            si += p.y;
        }
    }
    if (sl > 0) s_sum[sl - 1][o] = make_double2(sr, si);
    __syncthreads();
    if (sl > 0 || n >= N) return;
    for (int h = 0; h < kThreads / kSumOut - 1; ++h) {
        sr += s_sum[h][o].x;
        si += s_sum[h][o].y;
    }
    out[n] = make_double2(sr, si);
}

// Point ranges: a work item per CU at the tile count that a square grid of N
// outputs has at least, each range at least one chunk of points.
int point_ranges(int M, int N)
{
    const int ranges = std::max(1, kGridBlocks / std::max(1, N / (4 * kTilePairs * kTilePairs)));
    return std::max(1, std::min(ranges, (M + kGridChunk - 1) / kGridChunk));
}
// The workspace, in complex values: ranges N partial sums (256 N below two
// tiles' outputs, then at most 1 + 1 / k times 256 tiles' for N / 16,384 = k, or
// N), then the prepared points.
size_t workspace_values(int M, int N)
{
    return (size_t)point_ranges(M, N) * (size_t)N + sizeof(GridPt) / sizeof(double2) * (size_t)M;
}

}  // namespace

extern "C" long long nfft2d_ndft_workspace_bytes(int M, int N)
{
    if (M < 0 || N < 0) return nfft2d_fail(NFFT2D_ERR_ARG, "nfft2d_ndft_workspace_bytes: M = %d, N = %d", M, N);
    return N == 0 ? 0 : (long long)(sizeof(double2) * workspace_values(M, N));
}

extern "C" int NDFT2_2D_GPU(void *handle, const double *X, const double *Y, const double *u, const double *v,
                            const nfft2d_c128 *in, nfft2d_c128 *out, int Nu, int Nv, int M, int N)
{
    (void)handle;
    if (M < 0 || N < 0) return nfft2d_fail(NFFT2D_ERR_ARG, "NDFT2_2D_GPU: negative size");
    if (Nu == 0 || Nv == 0) return nfft2d_fail(NFFT2D_ERR_ARG, "NDFT2_2D_GPU: Nu and Nv must be non-zero");
    if (N == 0) return NFFT2D_OK;
    if (!u || !v || !out || (M > 0 && (!X || !Y || !in)))
        return nfft2d_fail(NFFT2D_ERR_ARG, "NDFT2_2D_GPU: null pointer");
    // (u, v) a grid: FP64 MFMA contraction; otherwise the direct sum (k_ndft_grid
    // reads the detector's finding and does one or the other).
    const int ranges = point_ranges(M, N);
    const int chunk = ((M + ranges - 1) / ranges + kGridChunk - 1) / kGridChunk * kGridChunk;
    const int dev = [] { int d = 0; (void)hipGetDevice(&d); return d; }();
    double2 *part = nullptr;
    // held until the launches are queued: a call from another host thread that
    // grows the workspace frees the old one only after a device synchronise
    std::lock_guard<std::mutex> lk(g_ws_mu);
    {
        GridWs &ws = g_ws[dev];
        const size_t need = workspace_values(M, N);
        if (ws.count < need) {
            if (ws.ptr) {
                (void)hipDeviceSynchronize();
                (void)hipFree(ws.ptr);
                ws.ptr = nullptr;
                ws.count = 0;
            }
            if (nfft2d_malloc(&ws.ptr, sizeof(double2) * need) != hipSuccess) {
                (void)hipGetLastError();
                ws.ptr = nullptr;
                return nfft2d_fail(NFFT2D_ERR_ALLOC, "NDFT2_2D_GPU: workspace of %zu bytes", sizeof(double2) * need);
            }
            ws.count = need;
        }
        part = ws.ptr;
    }
    GridPt *pts = reinterpret_cast<GridPt *>(part + (size_t)ranges * (size_t)N);
    const double2 *din = reinterpret_cast<const double2 *>(in);
    hipLaunchKernelGGL(k_grid_detect, dim3(1), dim3(kDetThreads), 0, nullptr, u, v, N);
    NFFT2D_LAUNCH_CHECK();
    const int nver = (N + kThreads - 1) / kThreads;
    hipLaunchKernelGGL(k_grid_verify, dim3(nver + (M + kThreads - 1) / kThreads), dim3(kThreads), 0, nullptr, u, v, N,
                       nver, X, Y, din, 1.0 / Nu, 1.0 / Nv, M, pts);
    NFFT2D_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_ndft_grid, dim3(kGridBlocks), dim3(kGridThreads), 0, nullptr, pts, part, M, ranges, chunk, X, Y,
                       u, v, din, 1.0 / Nu, 1.0 / Nv, N);
    NFFT2D_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_ndft_finish, dim3((N + kSumOut - 1) / kSumOut), dim3(kThreads), 0, nullptr, part, M, ranges,
                       reinterpret_cast<double2 *>(out), N);
    NFFT2D_LAUNCH_CHECK();
    return NFFT2D_OK;
}

extern "C" int nfft2d_ndft_grid_info(int *is_grid, int *nu, int *nv, int *vmajor)
{
    if (!is_grid || !nu || !nv || !vmajor) return nfft2d_fail(NFFT2D_ERR_ARG, "nfft2d_ndft_grid_info: null pointer");
    GridInfo g;
    if (hipDeviceSynchronize() != hipSuccess ||
        hipMemcpyFromSymbol(&g, HIP_SYMBOL(g_grid), sizeof(g), 0, hipMemcpyDeviceToHost) != hipSuccess)
        return nfft2d_fail(NFFT2D_ERR_HIP, "nfft2d_ndft_grid_info: reading the detector's finding failed");
    *is_grid = g.ok;
    *nu = g.nu;
    *nv = g.nv;
    *vmajor = g.vmajor;
    return NFFT2D_OK;
}

// ============================================================================
// Part 2: the type-2 direct sum as a split-precision MFMA contraction
// (kernels in ndft2d_mfma.hpp).  A plan holds the mode operand.
namespace {

constexpr int kNdftMaxN = 8192;
constexpr int kNdftC = ndft::kChunkTiles;  // MFMA column tiles per chunk

// Bytes of the mode operand of `tiles` tiles.
size_t ndft_operand_bytes(int prec, long long tiles)
{
    switch (prec) {
    case NFFT2D_NDFT_FP32: return ndft::operand_bytes<ndft::kNdftFp32>(tiles);
    case NFFT2D_NDFT_BF16X3: return ndft::operand_bytes<ndft::kNdftBf16x3>(tiles);
    default: return ndft::operand_bytes<ndft::kNdftFp16>(tiles);
    }
}

}  // namespace

struct nfft2d_ndft_plan_s {
    int N1, N2, prec, device;
    int nch, nks;
    void *G;              // mode operand, nch * nks * C * 64 slices
    float *scale;         // FP16: N1 per-row scales and their inverses
    float *inv_scale;
};

extern "C" int nfft2d_ndft_plan_create(nfft2d_ndft_plan **plan, int N1, int N2, int precision)
{
    if (!plan) return nfft2d_fail(NFFT2D_ERR_ARG, "nfft2d_ndft_plan_create: null plan pointer");
    *plan = nullptr;
    if (N1 <= 0 || N2 <= 0 || (N1 & 1) || (N2 & 1) || N1 > kNdftMaxN || N2 > kNdftMaxN)
        return nfft2d_fail(NFFT2D_ERR_SIZE, "nfft2d_ndft_plan_create: N1=%d N2=%d must be even, in [2, %d]", N1, N2,
                           kNdftMaxN);
    if (precision != NFFT2D_NDFT_FP32 && precision != NFFT2D_NDFT_BF16X3 && precision != NFFT2D_NDFT_FP16)
        return nfft2d_fail(NFFT2D_ERR_ARG, "nfft2d_ndft_plan_create: unknown precision %d", precision);
    nfft2d_ndft_plan_s *p = new (std::nothrow) nfft2d_ndft_plan_s();
    if (!p) return nfft2d_fail(NFFT2D_ERR_ALLOC, "nfft2d_ndft_plan_create: host allocation failed");
    p->N1 = N1;
    p->N2 = N2;
    p->prec = precision;
    NFFT2D_HIP_TRY(hipGetDevice(&p->device));
    // K indices: pairs of modes, or (FP16) single modes
    const int kn = precision == NFFT2D_NDFT_FP16 ? N2 : N2 / 2;
    p->nch = (N1 + ndft::kChunkK1 - 1) / ndft::kChunkK1;
    p->nks = (kn + 8 * ndft::kKsPad - 1) / (8 * ndft::kKsPad) * ndft::kKsPad;
    const size_t gbytes = ndft_operand_bytes(precision, (long long)p->nch * p->nks * kNdftC);
    if (nfft2d_malloc(&p->G, gbytes) != hipSuccess || nfft2d_malloc(&p->scale, sizeof(float) * N1) != hipSuccess ||
        nfft2d_malloc(&p->inv_scale, sizeof(float) * N1) != hipSuccess) {
        (void)hipGetLastError();
        nfft2d_ndft_plan_destroy(p);
        return nfft2d_fail(NFFT2D_ERR_ALLOC, "nfft2d_ndft_plan_create: device allocation of %zu bytes failed", gbytes);
    }
    *plan = p;
    return NFFT2D_OK;
}

extern "C" int nfft2d_ndft_plan_destroy(nfft2d_ndft_plan *p)
{
    if (!p) return nfft2d_fail(NFFT2D_ERR_ARG, "nfft2d_ndft_plan_destroy: null plan");
    if (p->G) (void)hipFree(p->G);
    if (p->scale) (void)hipFree(p->scale);
    if (p->inv_scale) (void)hipFree(p->inv_scale);
    delete p;
    return NFFT2D_OK;
}

extern "C" int nfft2d_ndft_set_modes(nfft2d_ndft_plan *p, const nfft2d_c64 *data, void *stream)
{
    if (!p || !data) return nfft2d_fail(NFFT2D_ERR_ARG, "nfft2d_ndft_set_modes: null argument");
    int rc = nfft2d_check_device(p->device);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    const float2 *F = reinterpret_cast<const float2 *>(data);
    if (p->prec == NFFT2D_NDFT_FP16) {   // the other precisions take their operands unscaled
        hipLaunchKernelGGL(ndft::k_ndft_rowscale, dim3(p->N1), dim3(256), 0, s, F, p->scale, p->inv_scale, p->N2);
        NFFT2D_LAUNCH_CHECK();
    }
    const long long total = (long long)p->nch * p->nks * kNdftC * 64;
    const dim3 grid((unsigned)((total + 255) / 256));
    switch (p->prec) {
    case NFFT2D_NDFT_FP32:
        hipLaunchKernelGGL((ndft::k_ndft_prep<ndft::kNdftFp32, kNdftC>), grid, dim3(256), 0, s, F, p->scale,
                           (ndft::Slice<ndft::kNdftFp32> *)p->G, p->N1, p->N2, p->nch, p->nks);
        break;
    case NFFT2D_NDFT_BF16X3:
        hipLaunchKernelGGL((ndft::k_ndft_prep<ndft::kNdftBf16x3, kNdftC>), grid, dim3(256), 0, s, F, p->scale,
                           (ndft::Slice<ndft::kNdftBf16x3> *)p->G, p->N1, p->N2, p->nch, p->nks);
        break;
    default:
        hipLaunchKernelGGL((ndft::k_ndft_prep<ndft::kNdftFp16, kNdftC>), grid, dim3(256), 0, s, F, p->scale,
                           (ndft::Slice<ndft::kNdftFp16> *)p->G, p->N1, p->N2, p->nch, p->nks);
        break;
    }
    NFFT2D_LAUNCH_CHECK();
    return NFFT2D_OK;
}

extern "C" int nfft2d_ndft_eval(nfft2d_ndft_plan *p, nfft2d_c64 *result, const float *x, const float *y, int M,
                                void *stream)
{
    if (!p) return nfft2d_fail(NFFT2D_ERR_ARG, "nfft2d_ndft_eval: null plan");
    if (M < 0) return nfft2d_fail(NFFT2D_ERR_ARG, "nfft2d_ndft_eval: negative M");
    if (M == 0) return NFFT2D_OK;
    if (!result || !x || !y) return nfft2d_fail(NFFT2D_ERR_ARG, "nfft2d_ndft_eval: null pointer");
    int rc = nfft2d_check_device(p->device);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((unsigned)((M + ndft::kPtsPerGroup - 1) / ndft::kPtsPerGroup));
    float2 *out = reinterpret_cast<float2 *>(result);
#ifndef NDFT_SPLIT
#define NDFT_SPLIT 2
#endif
    const dim3 block(64 * ndft::kWaves * NDFT_SPLIT);
    switch (p->prec) {
    case NFFT2D_NDFT_FP32:
        hipLaunchKernelGGL((ndft::k_ndft_t2<ndft::kNdftFp32, 4, NDFT_SPLIT>), grid, block, 0, s,
                           (const ndft::Slice<ndft::kNdftFp32> *)p->G, p->inv_scale, x, y, out, p->N1, p->N2, M,
                           p->nch, p->nks);
        break;
    case NFFT2D_NDFT_BF16X3:
        hipLaunchKernelGGL((ndft::k_ndft_t2<ndft::kNdftBf16x3, 8, NDFT_SPLIT>), grid, block, 0, s,
                           (const ndft::Slice<ndft::kNdftBf16x3> *)p->G, p->inv_scale, x, y, out, p->N1, p->N2, M,
                           p->nch, p->nks);
        break;
    default:
        hipLaunchKernelGGL((ndft::k_ndft_t2<ndft::kNdftFp16, 16, NDFT_SPLIT>), grid, block, 0, s,
                           (const ndft::Slice<ndft::kNdftFp16> *)p->G, p->inv_scale, x, y, out, p->N1, p->N2, M,
                           p->nch, p->nks);
        break;
    }
    NFFT2D_LAUNCH_CHECK();
    return NFFT2D_OK;
}

extern "C" int nfft2d_ndft_type2(nfft2d_ndft_plan *p, nfft2d_c64 *result, const nfft2d_c64 *data, const float *x,
                                 const float *y, int M, void *stream)
{
    int rc = nfft2d_ndft_set_modes(p, data, stream);
    if (rc != NFFT2D_OK) return rc;
    return nfft2d_ndft_eval(p, result, x, y, M, stream);
}

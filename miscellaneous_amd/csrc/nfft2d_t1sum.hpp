// nfft2d_t1sum.hpp -- small type-1 transforms as direct sums on the matrix cores.
//
//     F[k1][k2] = sum_p d_p e^{-2 pi i (k1 x_p / N1 + k2 y_p / N2)},  k in [-N/2, N/2)
//
// With h = k + 1/2 = s (j + 1/2), s = +-1, j = 0..N/2-1, and the half step
// e^{+pi i (x/N1 + y/N2)} moved into the sample (d' below), the modes of one
// dimension are conjugate pairs: with c, s the cosine and sine of
// 2 pi (2j + 1) x / (2N),
//     F(s1 j1, s2 j2) = sum d' (c1 - i s1 sin1)(c2 - i s2 sin2),
// so four complex sums d' {c1, sin1} {c2, sin2} give four modes: the real
// matrix product A B of A[(j1; d'r c, d'i c, d'r sin, d'i sin)][p] and
// B[p][(j2; c, sin)], 2 N1 N2 real multiply-adds per point, half of the plain
// complex product's.
//
// v_mfma_f32_32x32x16_f16 takes the product with each operand split in two
// FP16 values (x = hi + lo, round to nearest), lo*hi + hi*lo + hi*hi in FP32,
// as the tile spread does; d' is scaled by a power of two from the block's
// largest sample, the phasors by 2^14.  Phases are 32-bit fractions of a turn
// (from FP64, wrapping products exact), so the sum has no window error:
// rel-L2 against FP64 sums is below the NFFT's.
//
// A block of 8 waves takes KC points at a time (a stage).  Its threads write
// the operands of stage i + 1 into one of two LDS panels while the products of
// stage i run from the other: waves 0-3 issue the products first and waves 4-7
// the operands, so on each SIMD one wave's VALU work runs under the other's
// products.  A thread evaluates the phasor of one j at 4 points (sine and
// cosine polynomials) and steps to j + JS, j + 2 JS ... by complex products
// with e^{2 JS i pi x/N}, computed once per point and stage.
//
// Measured (gfx950): 250 transforms of 88 x 88 modes from 1,936 points, a call of
// 105 us with the two launches of its sort (about 14 us) in it, where spread,
// column pass and row pass alone took 144 + 195 + 51; 45 GFLOP executed, about
// 0.5 PFLOP/s: a stage's 27 products per wave (0.8 us of matrix time on each
// SIMD) and its ~400 VALU instructions per wave make 2.9 us, held by the latency
// of the operand chain at 2 waves per SIMD.  One transform of that size: 13.1 us
// a call in two launches, where sort, spread and passes took 30.
#pragma once

#include "nfft2d_batch.hpp"
#include "nfft2d_kernels.hpp"

#include <algorithm>

namespace nfft2d {

struct T1SumArgs {
    const BatchDesc* bd;          // a batch: transform t = block / (S m1 m2); null: the arrays below
    const float *x, *y;
    const float2* d;
    float2* F;                    // S = 1 of a batch writes the modes, else the partial sums go to part
    float2* part;                 // [S][N1][N2]
    const float* scale;           // null, or N1 x N2 factors of the modes
    int M, N1, N2;
    int S, m1, m2;                // point ranges, mode chunks per dimension
    int k1c, k2c;                 // pairs j per chunk
    int jm, js1, js2;             // phasors per thread; its steps in j
    int kp1, kp2;                 // LDS rows per operand kind
    double inv1, inv2;            // 1 / (2 N)
};

typedef __attribute__((address_space(1))) float gfloat;
typedef __attribute__((address_space(1))) f2v gfloat2;
constexpr int kSumThreads = 512;
constexpr int kSumMaxLds = 160 * 1024;
// A phase is off by at most (2j + 1) 2^-33 turns, 1.9e-7 rad per dimension at the
// last mode of N = 256 (about 6e-8 rms over its modes and points), beside 1e-7 of
// the phasors' FP32 evaluation and 1.5e-7 and more of the sums.
constexpr int kT1SumMaxN = 256;
constexpr int kT1SumMaxS = 12;           // every batch plan's spread scratch holds 12 partial results
// A lone transform: up to 12 ranges of 8 stages of 64 points, and the work where
// the sort, spread and FFT passes (30-38 us, launches mostly) are as fast.
// NFFT2_2D_GPU, direct sum against those, us: 88 x 88 modes from 1,936 points
// 13.6 / 30.2; 96 x 98 from 5,000 16.7 / 34.8; 256 x 256 from 10,000 35.9 / 35.3;
// 64 x 64 from 30,000 54 / 33.
constexpr double kT1SumOneWork = 4e8;
constexpr int kT1SumOnePoints = 6144;
struct SumPoint {                 // a stage's point
    unsigned u1, u2;              // x / (2 N1), y / (2 N2), fractions of a turn
    float2 d, w1, w2;             // scaled d', steps of js1 and js2 pairs
};
__host__ __device__ constexpr int sum_panel_bytes(int KC, int kp1, int kp2) { return (KC / 8) * 16 * 2 * (4 * kp1 + 2 * kp2); }
__host__ __device__ constexpr int sum_lds_bytes(int KC, int kp1, int kp2)
{
    return 2 * sum_panel_bytes(KC, kp1, kp2) + 2 * KC * (int)sizeof(SumPoint);
}

// cos and sin of 2 pi t / 2^32.  r in [-1/8, 1/8] turn, minimax polynomials
// (2.4e-9 and 5e-11; 7e-8 .. 1e-7 with their FP32 evaluation).
__device__ __forceinline__ float2 turn_cs(unsigned t)
{
    const unsigned q = (t + 0x20000000u) >> 30;
    const float r = (float)(int)(t - (q << 30)) * 2.3283064365386963e-10f;
    const float z = r * r;
    float s = fmaf(z, -75.40206754490094f, 81.59255353216126f);
    s = fmaf(z, s, -41.34166263301897f);
    s = fmaf(z, s, 6.283185287867181f);
    s *= r;
    float c = fmaf(z, 59.22040719541854f, -85.44285211857814f);
    c = fmaf(z, c, 64.93931620842821f);
    c = fmaf(z, c, -19.7392086503579f);
    c = fmaf(z, c, 0.9999999999526008f);
    const bool sw = (q & 1) != 0;
    const unsigned cc = __float_as_uint(sw ? s : c) ^ (((q + 1) & 2) << 30);   // cos < 0 in quadrants 1, 2
    const unsigned ss = __float_as_uint(sw ? c : s) ^ ((q & 2) << 30);         // sin < 0 in quadrants 2, 3
    return make_float2(__uint_as_float(cc), __uint_as_float(ss));
}

// x / (2N) as a 32-bit fraction of a turn: the reduction by 2N is exact, and
// adding 1.5 * 2^20 leaves the fraction's 32 bits in the low word.
__device__ __forceinline__ unsigned turn_of(double x, double inv2n, int N)
{
    const double r = fma(-rint(x * inv2n), (double)(2 * N), x);
    return (unsigned)__double2loint(fma(r, inv2n, 1572864.0));
}

// 4 values (one operand row at 4 points) split into FP16 planes, 8 bytes each
__device__ __forceinline__ void put_split(char* hi, char* lo, float a, float b, float c, float d)
{
    uint2 h, l;
    split_h2(a, b, h.x, l.x);
    split_h2(c, d, h.y, l.y);
    *reinterpret_cast<uint2*>(hi) = h;
    *reinterpret_cast<uint2*>(lo) = l;
}

// Waves: RG row groups of TR tiles (32 rows = 8 pairs j1 x 4 kinds) by KG
// groups of 16 points; every wave has all CT column tiles (16 pairs j2 x 2).
// LDS panel: [plane hi, lo][8-point group][kind][row j] of 16 bytes, A then B.
// A lane reads its row of an operand as 16 bytes; rows per kind kp1 = 4 or 12
// mod 16 and kp2 = 8 mod 16 put the kinds of a 16-lane group on different
// banks.  Padding rows of a last tile read the bytes that follow (inside the
// allocation); they only reach outputs that are not stored.
template <int RG, int TR, int CT>
__global__ __launch_bounds__(kSumThreads) void k_t1_sum(T1SumArgs a)
{
    constexpr int KG = 8 / RG, KC = 16 * KG;
    extern __shared__ __attribute__((aligned(16))) char sum_lds[];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    int b = blockIdx.x;
    const int c2 = b % a.m2;
    b /= a.m2;
    const int c1 = b % a.m1;
    b /= a.m1;
    const int s = b % a.S, t = b / a.S;
    if (a.bd) {
        const BatchDesc& d = a.bd[t];
        a.x = d.x;
        a.y = d.y;
        a.d = d.d1;
        a.F = d.F1;
        a.part = d.scratch;
        a.M = d.M;
    }
    // global, not flat: a flat load in flight counts as an LDS operation, and the
    // next wait for an operand would wait for memory too
    const gfloat* gx = (const gfloat*)a.x;
    const gfloat* gy = (const gfloat*)a.y;
    const gfloat2* gd = (const gfloat2*)a.d;
    const int j1o = c1 * a.k1c, n1 = min(a.k1c, a.N1 / 2 - j1o);
    const int j2o = c2 * a.k2c, n2 = min(a.k2c, a.N2 / 2 - j2o);
    const int nst_all = (a.M + KC - 1) / KC, per = (nst_all + a.S - 1) / a.S;
    const int p_lo = min(a.M, s * per * KC), p_hi = min(a.M, p_lo + per * KC);
    const int nst = (p_hi - p_lo + KC - 1) / KC;
    const int panel = sum_panel_bytes(KC, a.kp1, a.kp2);
    const int plA = (KC / 8) * 4 * a.kp1 * 16, plB = (KC / 8) * 2 * a.kp2 * 16;   // bytes per plane
    SumPoint* pd = reinterpret_cast<SumPoint*>(sum_lds + 2 * panel);

    // point data: thread roles (u1 w1), (u2 w2), (d') of a stage's points, on
    // the waves whose operand tasks are the cheaper B rows
    const int role = (tid ^ 256) / KC, rp = tid % KC;
    struct Pt { float x, y; f2v v; };
    auto load_point = [&](int st) {
        const int p = p_lo + st * KC + rp;
        const bool ok = role < 3 && p < p_hi;
        Pt r;
        r.x = ok && role != 1 ? gx[p] : 0.f;
        r.y = ok && role != 0 ? gy[p] : 0.f;
        r.v = ok && role == 2 ? gd[p] : f2v{0.f, 0.f};
        return r;
    };
    const Pt first = load_point(0), second = load_point(1);

    // the scale 2^se brings the range's largest sample component to [2^13, 2^14).  For
    // samples below 2^-98 it and its inverse take two factors each, the second one 1 for
    // all others (ldexp on every mode instead, or a branch that scales the sums: 105.2 ->
    // 107.5 us for 250 transforms of 88 x 88 modes)
    float mx = 0.f;
    for (int p0 = p_lo; p0 < p_hi; p0 += 4 * kSumThreads) {   // 4 loads in flight
        f2v v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = gd[min(p0 + k * kSumThreads + tid, p_hi - 1)];
#pragma unroll
        for (int k = 0; k < 4; ++k) mx = fmaxf(mx, fmaxf(fabsf(v[k].x), fabsf(v[k].y)));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    float* red = reinterpret_cast<float*>(sum_lds);
    if (lane == 0) red[w] = mx;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; ++k) mx = fmaxf(mx, red[k]);
    __syncthreads();
    const int se = __builtin_amdgcn_readfirstlane(14 - __builtin_amdgcn_frexp_expf(mx));
    const int sa = min(se, 112), sb = se - sa;
    auto pow2 = [](int e) { return __uint_as_float((unsigned)(127 + e) << 23); };
    const float sc = pow2(sa), sc2 = pow2(sb), inv_sc = pow2(-sa - 14), inv_sc2 = pow2(-sb);   // and the phasors' 2^14

    auto put_point = [&](int st, const Pt& r) {
        SumPoint& q = pd[(st & 1) * KC + rp];
        if (role == 0) {
            const unsigned u = turn_of((double)r.x, a.inv1, a.N1);
            q.u1 = u;
            q.w1 = turn_cs(2u * (unsigned)a.js1 * u);
        } else if (role == 1) {
            const unsigned u = turn_of((double)r.y, a.inv2, a.N2);
            q.u2 = u;
            q.w2 = turn_cs(2u * (unsigned)a.js2 * u);
        } else if (role == 2) {
            const float2 e = turn_cs(turn_of((double)r.x, a.inv1, a.N1) + turn_of((double)r.y, a.inv2, a.N2));
            const float vx = r.v.x * sc * sc2, vy = r.v.y * sc * sc2;
            float2 v = make_float2(vx * e.x - vy * e.y, vx * e.y + vy * e.x);
            // coordinates beyond the transform's range give NaN, as locate() does
            if (!(fabsf((float)kC * r.x) < 1073741824.f) || !(fabsf((float)kC * r.y) < 1073741824.f))
                v = make_float2(NAN, NAN);
            q.d = v;
        }
    };
    // operand task of this thread: dimension, 4-point group, first pair.  The
    // two groups of an 8-point unit are on adjacent lanes (8-byte stores, contiguous)
    const int nt1 = a.js1 * (KC / 4), nt2 = a.js2 * (KC / 4);
    const bool dim1 = tid < nt1;
    const int tt = dim1 ? tid : tid - nt1;
    const int js = dim1 ? a.js1 : a.js2, gp = tt / (2 * js), rem = tt - gp * 2 * js;
    const int g4 = 2 * gp + (rem & 1), j0 = rem >> 1;
    const bool task = tid < nt1 + nt2;
    const unsigned hf = 2u * (unsigned)((dim1 ? j1o : j2o) + j0) + 1u;
    const int nj = dim1 ? n1 : n2;
    const int ks = (dim1 ? a.kp1 : a.kp2) * 16, pl = dim1 ? plA : plB;
    const int at = (dim1 ? (gp * 4 * a.kp1 + j0) * 16 : 2 * plA + (gp * 2 * a.kp2 + j0) * 16) + (rem & 1) * 8;
    auto operands = [&](int st) {
        if (!task) return;
        char* hi = sum_lds + (st & 1) * panel + at;
        const SumPoint* q = pd + (st & 1) * KC + 4 * g4;
        float2 z[4], w[4];
        if (dim1) {
            float2 d[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                z[k] = turn_cs(hf * q[k].u1);
                w[k] = q[k].w1;
                d[k] = q[k].d;
            }
            for (int m = 0, j = j0; m < a.jm && j < nj; ++m, j += js, hi += js * 16) {
                if (m) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) z[k] = cmul(z[k], w[k]);
                }
                char* lo = hi + pl;
                put_split(hi, lo, d[0].x * z[0].x, d[1].x * z[1].x, d[2].x * z[2].x, d[3].x * z[3].x);
                put_split(hi + ks, lo + ks, d[0].y * z[0].x, d[1].y * z[1].x, d[2].y * z[2].x, d[3].y * z[3].x);
                put_split(hi + 2 * ks, lo + 2 * ks, d[0].x * z[0].y, d[1].x * z[1].y, d[2].x * z[2].y, d[3].x * z[3].y);
                put_split(hi + 3 * ks, lo + 3 * ks, d[0].y * z[0].y, d[1].y * z[1].y, d[2].y * z[2].y, d[3].y * z[3].y);
            }
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                z[k] = cscale(turn_cs(hf * q[k].u2), 16384.f);
                w[k] = q[k].w2;
            }
            for (int m = 0, j = j0; m < a.jm && j < nj; ++m, j += js, hi += js * 16) {
                if (m) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) z[k] = cmul(z[k], w[k]);
                }
                char* lo = hi + pl;
                put_split(hi, lo, z[0].x, z[1].x, z[2].x, z[3].x);
                put_split(hi + ks, lo + ks, z[0].y, z[1].y, z[2].y, z[3].y);
            }
        }
    };

    f16v acc[TR][CT];
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = f16v{};
    const int kgi = w % KG, rgi = w / KG;
    const int g8 = 2 * kgi + (lane >> 5), i32 = lane & 31;
    const int rtl = (n1 + 7) / 8 - 1;               // last row tile that holds pairs
    int offA[TR];
#pragma unroll
    for (int i = 0; i < TR; ++i)
        offA[i] = ((g8 * 4 + (i32 & 3)) * a.kp1 + 8 * min(rgi * TR + i, rtl) + (i32 >> 2)) * 16;
    const int offB = ((g8 * 2 + (i32 & 1)) * a.kp2 + (i32 >> 1)) * 16;
    auto products = [&](int st) {
        const char* buf = sum_lds + (st & 1) * panel;
        h8v ah[TR], al[TR];
#pragma unroll
        for (int i = 0; i < TR; ++i) {
            ah[i] = *reinterpret_cast<const h8v*>(buf + offA[i]);
            al[i] = *reinterpret_cast<const h8v*>(buf + plA + offA[i]);
        }
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            const h8v bh = *reinterpret_cast<const h8v*>(buf + 2 * plA + offB + 256 * j);
            const h8v bl = *reinterpret_cast<const h8v*>(buf + 2 * plA + plB + offB + 256 * j);
#pragma unroll
            for (int i = 0; i < TR; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[i], bh, acc[i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < TR; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i], bl, acc[i][j], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < TR; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i], bh, acc[i][j], 0, 0, 0);
        }
    };

    put_point(0, first);
    put_point(1, second);
    __syncthreads();
    gfloat2* out = (gfloat2*)(a.S == 1 && a.bd ? a.F : a.part + (size_t)s * a.N1 * a.N2);
    const float sg = (lane & 1) ? 1.f : -1.f;       // even lanes write s2 = +, odd lanes s2 = -
    if (nst > 0) {
        operands(0);
        __syncthreads();
        for (int st = 0; st < nst; ++st) {
            const Pt next = load_point(st + 2);
#pragma unroll 1
            for (int ph = 0; ph < 2; ++ph) {
                if ((ph == 0) == (w < 4)) products(st);
                else if (st + 1 < nst) operands(st + 1);
            }
            put_point(st + 2, next);                // over stage st's points, last read before the previous barrier
            __syncthreads();
        }
    }

    // the point groups' sums in a fixed order, one row of tiles at a time, then
    // the four modes of every pair of pairs: an even lane holds the c2 sums of
    // its j2, the odd lane next to it the sin2 sums
    const gfloat* gs = a.S == 1 && a.bd ? (const gfloat*)a.scale : nullptr;   // else k_t1_sum_add scales
#pragma unroll
    for (int i = 0; i < TR; ++i) {
        // this row's factors, in flight together during the exchange
        float fs[CT][4][2];
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int j1 = 8 * (rgi * TR + i) + 2 * q + (lane >> 5), j2 = 16 * j + (i32 >> 1);
                fs[j][q][0] = fs[j][q][1] = 1.f;
                if (gs && kgi == 0 && j1 < n1 && j2 < n2) {
                    const int col = (lane & 1) ? a.N2 / 2 - 1 - j2o - j2 : a.N2 / 2 + j2o + j2;
                    fs[j][q][0] = gs[(a.N1 / 2 + j1o + j1) * a.N2 + col];
                    fs[j][q][1] = gs[(a.N1 / 2 - 1 - j1o - j1) * a.N2 + col];
                }
            }
        __syncthreads();
        if (kgi > 0) {
#pragma unroll
            for (int j = 0; j < CT; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    red[(((kgi - 1) * RG + rgi) * CT * 16 + j * 16 + r) * 64 + lane] = acc[i][j][r];
        }
        __syncthreads();
        if (kgi > 0) continue;
#pragma unroll
        for (int j = 0; j < CT; ++j) {
#pragma unroll
            for (int g = 0; g < KG - 1; ++g)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] += red[((g * RG + rgi) * CT * 16 + j * 16 + r) * 64 + lane];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float cr = acc[i][j][4 * q], ci = acc[i][j][4 * q + 1];
                const float sr = acc[i][j][4 * q + 2], si = acc[i][j][4 * q + 3];
                // c -+ i sin: the s1 = + and s1 = - sums
                const float2 ep = make_float2(cr + si, ci - sr), em = make_float2(cr - si, ci + sr);
                const float2 op = make_float2(__shfl_xor(ep.x, 1, 64), __shfl_xor(ep.y, 1, 64));
                const float2 om = make_float2(__shfl_xor(em.x, 1, 64), __shfl_xor(em.y, 1, 64));
                const bool odd = (lane & 1) != 0;
                const float2 Ep = odd ? op : ep, Op = odd ? ep : op, Em = odd ? om : em, Om = odd ? em : om;
                // E -+ i O
                const float2 fp = make_float2((Ep.x - sg * Op.y) * inv_sc, (Ep.y + sg * Op.x) * inv_sc);
                const float2 fm = make_float2((Em.x - sg * Om.y) * inv_sc, (Em.y + sg * Om.x) * inv_sc);
                const int j1 = 8 * (rgi * TR + i) + 2 * q + (lane >> 5), j2 = 16 * j + (i32 >> 1);
                if (j1 < n1 && j2 < n2) {
                    const int col = odd ? a.N2 / 2 - 1 - j2o - j2 : a.N2 / 2 + j2o + j2;
                    out[(size_t)(a.N1 / 2 + j1o + j1) * a.N2 + col] = f2v{fp.x * (fs[j][q][0] * inv_sc2), fp.y * (fs[j][q][0] * inv_sc2)};
                    out[(size_t)(a.N1 / 2 - 1 - j1o - j1) * a.N2 + col] = f2v{fm.x * (fs[j][q][1] * inv_sc2), fm.y * (fs[j][q][1] * inv_sc2)};
                }
            }
        }
    }
}

// F[e] = the S partial sums of e, in order.
__global__ __launch_bounds__(256) void k_t1_sum_add(T1SumArgs a)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    const float2* part = a.part;
    float2* F = a.F;
    if (a.bd) {
        part = a.bd[blockIdx.y].scratch;
        F = a.bd[blockIdx.y].F1;
    }
    const int n = a.N1 * a.N2;
    if (e >= n) return;
    float2 v = make_float2(0.f, 0.f);
#pragma unroll 4
    for (int s = 0; s < a.S; ++s) v = cadd(v, part[(size_t)s * n + e]);
    F[e] = a.scale ? cscale(v, a.scale[e]) : v;
}

// ---------------------------------------------------------------- host side
// How a transform (or a batch of count equal sizes) is split: mode chunks of
// 16 to 64 pairs per dimension and S point ranges, the split of least
// estimated time.  Every product of 16 points rounds the FP32 sums three times,
// so their error grows with the square root of a range's products per point
// group; chain bounds it (t1_sum_chain).
struct T1SumPlan {
    T1SumArgs a;
    int rg, tr, ct, lds;
    long long blocks;
    double t;                     // estimated time, us
};
inline int sum_rows(int n, int r0, int r1)   // smallest row count >= n that is r0 or r1 mod 16
{
    while (n % 16 != r0 && n % 16 != r1) ++n;
    return n;
}
inline T1SumPlan t1_sum_plan(int N1, int N2, int M, int count, int chain)
{
    T1SumPlan best = {};
    const int K1 = N1 / 2, K2 = N2 / 2;
    auto chunk = [](int K, int c) { const int n = (K + c - 1) / c; return (K + n - 1) / n; };
    for (int c = 64; c >= 16; c -= 16) {
        T1SumPlan p = {};
        T1SumArgs& a = p.a;
        a.M = M; a.N1 = N1; a.N2 = N2;
        a.inv1 = 0.5 / N1; a.inv2 = 0.5 / N2;
        a.k1c = chunk(K1, c);
        a.k2c = chunk(K2, c);
        a.m1 = (K1 + a.k1c - 1) / a.k1c;
        a.m2 = (K2 + a.k2c - 1) / a.k2c;
        a.kp1 = sum_rows(a.k1c, 4, 12);
        a.kp2 = sum_rows(a.k2c, 8, 8);
        p.rg = a.k1c <= 48 && a.k2c <= 48 && sum_lds_bytes(64, a.kp1, a.kp2) <= kSumMaxLds ? 2 : 4;
        const int KG = 8 / p.rg, KC = 16 * KG, st = std::max(1, (M + KC - 1) / KC);
        p.tr = p.rg == 2 ? (a.k1c + 15) / 16 : 2;
        p.ct = (a.k2c + 15) / 16;
        const long long tiles = (long long)count * a.m1 * a.m2;
        const int s_min = (st + chain - 1) / chain;
        if (s_min > kT1SumMaxS) continue;
        a.S = (int)std::max<long long>(s_min, std::min<long long>(std::min(kT1SumMaxS, st), 256 / tiles));
        p.blocks = tiles * a.S;
        // us, one block per CU at a time, fitted: per point 9 ns, 0.35 ns per pair of the
        // chunk and 0.6 ns per tile slot; per block 8 us and 1 us per tile of a wave
        // (88 x 88 modes: 105 us for 1,936 points, 126 x 126: 180 for 2,500); then
        // the partial sums, written and read
        p.t = (double)((p.blocks + 255) / 256) *
              (((st + a.S - 1) / a.S) * KC * (0.009 + 0.00035 * (a.k1c + a.k2c) + 0.0006 * p.rg * p.tr * p.ct) + 8.0 + p.tr * p.ct);
        if (a.S > 1) p.t += 4.0 + 16.0 * count * a.S * N1 * N2 / 3e6;
        if (best.blocks && p.t >= best.t) continue;
        a.jm = 1;
        do {
            a.js1 = (a.k1c + a.jm - 1) / a.jm;
            a.js2 = (a.k2c + a.jm - 1) / a.jm;
        } while ((a.js1 + a.js2) * (KC / 4) > kSumThreads && ++a.jm);
        p.lds = std::max(sum_lds_bytes(KC, a.kp1, a.kp2), (KG - 1) * p.rg * p.ct * 16 * 64 * 4);
        best = p;
    }
    return best;                                    // blocks = 0: no split keeps the chains short enough
}

inline void t1_sum_launch(const T1SumPlan& p, int count, hipStream_t s)
{
    auto go = [&](auto k) { hipLaunchKernelGGL(k, dim3((unsigned)p.blocks), dim3(kSumThreads), p.lds, s, p.a); };
    if (p.rg == 2) {
        switch (3 * (p.tr - 1) + p.ct - 1) {
        case 0: go(k_t1_sum<2, 1, 1>); break;
        case 1: go(k_t1_sum<2, 1, 2>); break;
        case 2: go(k_t1_sum<2, 1, 3>); break;
        case 3: go(k_t1_sum<2, 2, 1>); break;
        case 4: go(k_t1_sum<2, 2, 2>); break;
        case 5: go(k_t1_sum<2, 2, 3>); break;
        case 6: go(k_t1_sum<2, 3, 1>); break;
        case 7: go(k_t1_sum<2, 3, 2>); break;
        default: go(k_t1_sum<2, 3, 3>); break;
        }
    } else {
        switch (p.ct) {
        case 1: go(k_t1_sum<4, 2, 1>); break;
        case 2: go(k_t1_sum<4, 2, 2>); break;
        case 3: go(k_t1_sum<4, 2, 3>); break;
        default: go(k_t1_sum<4, 2, 4>); break;
        }
    }
    if (p.a.S > 1 || !p.a.bd)
        hipLaunchKernelGGL(k_t1_sum_add, dim3((unsigned)((p.a.N1 * p.a.N2 + 255) / 256), (unsigned)count), dim3(256), 0, s,
                           p.a);
}

}  // namespace nfft2d

// nfft2d_czt.hpp -- the four FFT passes of a plan for line lengths that are
// not powers of two, as chirp-z (Bluestein) transforms.
//
// Every pass maps P inputs of a line to Q outputs
//     Y[q] = sum_{p<P} x[p] w^{(p + p0)(q + q0)},  w = e^{-2 pi i / L},  L = 2N,
// (type-2 rows / columns: P = N, Q = L, p0 = -N/2, q0 = 0, modes centred;
//  type-1 columns / rows: P = L, Q = N, p0 = 0, q0 = -N/2), which with
// ab = (a^2 + b^2 - (b - a)^2) / 2 and c[k] = w^{k^2/2} = e^{-i pi k^2 / L} is
//     Y[q] = c[q + q0] sum_p (x[p] c[p + p0]) conj(c[(q - p) + q0 - p0]),
// a linear convolution, taken circularly at the power of two m >= P + Q - 1
// through two FFTs of m points.  The inverse direction (e^{+}) conjugates the
// input and the output.  The chirps (P and Q entries), the transform of the
// convolution kernel and the FFT's twiddles e^{-2 pi i t / m} (m entries each)
// are computed on the host in FP64 at plan creation.  O(m log m) per line
// instead of the O(N L) of the direct passes.
//
// What bounds these passes is the LDS: a radix-4 form that kept the line there
// moved it through LDS 26 times at m = 2048 (with two twiddle reads per
// product besides) and ran at a twentieth of the copy rate.  So a line lives
// in registers, 8 values j + q m/8 (q < 8) per role j < m/8, the order in
// which every radix-8 stage of the Stockham form reads and the last one
// leaves them: the kernel product and the start of the second FFT need no
// exchange, and each FFT makes stages - 1 (three) trips through LDS.  Measured
// on FP64 lines of 500 and 250 (500 x 250 modes, both passes of a type-2 /
// type-1): 36 / 35 -> 21 / 21 us.  The twiddles come from global memory, so
// they lie in the order in which a stage's roles read them: as one table
// e^{-2 pi i j / m} read at strides of m / (8 NS) they were up to 448 cache lines
// per wave and stage, and long lines ran behind the LDS form (type-2 of N x N
// modes to 20,000 points, LDS form / one table / stage order: complex64 N =
// 1,500 386 / 447 / 307 us, 3,000 2,571 / 4,800 / 1,633, complex128 1,800 1,040
// / 880 / 529).
#pragma once

#include <mutex>

#include "../../include/nfft2d.h"
#include "nfft2d_device.hpp"
#include "nfft2d_internal.hpp"

namespace nfft2d {

template <typename T>
struct CztTables {
    const cplx<T> *cin = nullptr;    // c[p + p0], P
    const cplx<T> *cout = nullptr;   // c[q + q0], Q
    const cplx<T> *hhat = nullptr;   // FFT_m of the kernel conj(c[d + q0 - p0]), d = q - p
    const cplx<T> *tw = nullptr;     // the FFT's twiddles, m (czt_tw_index)
    int P = 0, Q = 0, m = 0;
};

constexpr int kCztMinLog = 9;   // m = 512 (N >= 128) .. 16,384 (N <= 4096), FP64 8,192 (N <= 2048)
template <typename T> constexpr int kCztMaxLog = sizeof(T) == 4 ? 14 : 13;

// Smallest power of two m >= 3N - 1 (P + Q - 1 = N + 2N - 1): the chirp-z FFT length of a line of N.
__host__ __device__ constexpr int czt_m(int N)
{
    int m = 1;
    while (m < 3 * N - 1) m <<= 1;
    return m;
}

// Entry e of the twiddle table is e^{-2 pi i czt_tw_index(m, e) / m}: the stages'
// twiddles w^{r k}, r = 1..7, k < NS, one stage after the other in the order
// [r][k], so that neighbouring roles read neighbouring entries (m - r0 in all).
__host__ __device__ constexpr int czt_tw_index(int m, int e)
{
    int n = 0, t = 0;
    while ((1 << n) < m) ++n;
    const int r0 = n % 3 == 0 ? 3 : n % 3, q = e + (1 << r0);   // stage s: q in [NS, 8 NS)
    while ((1 << (t + 1)) <= q) ++t;
    t = (t - r0) / 3 * 3 + r0;
    return t < n ? (((q - (1 << t)) >> t) + 1) * (q & ((1 << t) - 1)) * (m / 8 >> t) : 0;
}

// The chirp-z tables of a line length N inside one table buffer (layout
// [cin2 N][cout2 L][hhat2 m][cin1 L][cout1 N][hhat1 m][tw m], L = 2N), for
// its type-2 (t2 = true) or type-1 pass.
template <typename T>
__host__ __device__ inline CztTables<T> czt_tables_of(const void* buf, int N, int m, bool t2)
{
    using C = cplx<T>;
    const int L = 2 * N;
    const C* b = (const C*)buf;
    CztTables<T> t;
    t.m = m;
    t.tw = b + 3 * L + 2 * m;          // after both passes' chirps and kernels
    if (t2) {
        t.P = N;
        t.Q = L;
        t.cin = b;
        t.cout = b + N;
        t.hhat = b + N + L;
    } else {
        const C* o = b + N + L + m;
        t.P = L;
        t.Q = N;
        t.cin = o;
        t.cout = o + L;
        t.hhat = o + L + N;
    }
    return t;
}

// a b with the order of the roundings written out: left to contract a.x b.x -
// a.y b.y, the compiler fuses either product, one way in a plan's pass and the
// other in a batch's.
template <typename C> __device__ __forceinline__ C cmul_f(C a, C b)
{
    return mk(fma(-a.y, b.y, a.x * b.x), fma(a.y, b.x, a.x * b.y));
}

// FFT of 2^LOGM points (e^{-2 pi i jk / m}), the Stockham stages of
// nfft2d_device.hpp with the line in registers between the LDS exchanges.
// A role is one of the m/8 workers of a line: role (l, j) holds x[j + q m/8]
// in v[q] on entry and X[j + q m/8] on return.  A thread plays K roles
// (act: the role exists); a role may name another (line, j) for the input
// (la, ja), the middle stages (lm, jm) and the output (lo, jo), the exchanges
// make the remap free.  lds: line l at l * lds_line<m>().  Every barrier is
// reached by all threads; the LDS must be free on entry, and is being read
// when the function returns.
template <typename T, int LOGM, int K>
__device__ __forceinline__ void czt_fft(cplx<T> (&v)[K][8], cplx<T>* lds, const cplx<T>* __restrict__ tw,
                                        const bool (&act)[K], const int (&la)[K], const int (&ja)[K],
                                        const int (&lm)[K], const int (&jm)[K], const int (&lo)[K],
                                        const int (&jo)[K])
{
    using C = cplx<T>;
    constexpr int M = 1 << LOGM, TPL = M / 8, LL = lds_line<M>(), R0 = FftPlan<M>::r0, B0 = 8 / R0;
    constexpr int S = FftPlan<M>::stages;
    static_assert(S >= 3, "m >= 512");
#pragma unroll
    for (int u = 0; u < K; ++u) {
#pragma unroll
        for (int b = 0; b < B0; ++b) {
            C a[R0];
#pragma unroll
            for (int r = 0; r < R0; ++r) a[r] = v[u][b + r * B0];
            dftR<R0, -1>(a);
            if (act[u]) {
#pragma unroll
                for (int r = 0; r < R0; ++r) lds[la[u] * LL + lpad((ja[u] + b * TPL) * R0 + r)] = a[r];
            }
        }
    }
#pragma unroll
    for (int s = 1; s < S; ++s) {
        const int NS = FftPlan<M>::ns(s);
        const bool last = s == S - 1;
        // the stage's twiddles, in flight across the barrier and the LDS reads; with
        // two roles a thread only when each is played (both roles' spill)
        C w[7];
        auto twiddles = [&](int j) {
            const C* __restrict__ t = tw + NS - R0 + (j & (NS - 1));
#pragma unroll
            for (int r = 1; r < 8; ++r) w[r - 1] = t[(r - 1) * NS];
        };
        if constexpr (K == 1) twiddles(last ? jo[0] : jm[0]);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < K; ++u) {
            const int l = last ? lo[u] : lm[u], j = last ? jo[u] : jm[u];
            if (act[u]) {
#pragma unroll
                for (int q = 0; q < 8; ++q) v[u][q] = lds[l * LL + lpad(j + q * TPL)];
            }
        }
        if (!last) __syncthreads();
#pragma unroll
        for (int u = 0; u < K; ++u) {
            const int j = last ? jo[u] : jm[u], k = j & (NS - 1);
            if constexpr (K > 1) twiddles(j);
#pragma unroll
            for (int r = 1; r < 8; ++r) v[u][r] = cmul_f(v[u][r], w[r - 1]);
            dft8<-1>(v[u]);
            if (!last && act[u]) {
                const int o = (j - k) * 8 + k;
#pragma unroll
                for (int r = 0; r < 8; ++r) lds[lm[u] * LL + lpad(o + r * NS)] = v[u][r];
            }
        }
    }
}

// Lines line0 .. line0 + B - 1 (below `lines`) of a chirp-z pass by the whole
// block: B m/8 roles, K per thread (blockDim.x * K >= B m/8).  Line b reads
// x[p] = in[b in_ls + p in_es] and writes out[b out_ls + q out_es]; COL_IN /
// COL_OUT: the lines lie side by side there (ls = 1), neighbouring threads
// take neighbouring lines.  scale_in (type-2 rows): the input is scaled by
// sl[b] se[p] (the pre-compensation D1[k1] D2[k2]); else the output by sl[b]
// se[q] (the deconvolution); sl null: no scaling.  conj: the inverse
// direction.  Every butterfly and product is the same whatever B and K, so
// plans and batches (other block sizes) get the same bits.
template <typename T, int LOGM, int B, int K, bool COL_IN, bool COL_OUT>
__device__ __forceinline__ void czt_lines(int line0, int lines, cplx<T>* lds, const cplx<T>* __restrict__ in,
                                          long long in_ls, long long in_es, cplx<T>* __restrict__ out,
                                          long long out_ls, long long out_es, const T* __restrict__ sl,
                                          const T* __restrict__ se, bool scale_in, bool conj, const CztTables<T>& tb)
{
    using C = cplx<T>;
    constexpr int M = 1 << LOGM, TPL = M / 8;
    // kernel and output factors loaded ahead of the FFT they follow; at 1,024
    // threads (128 registers each) only when they are used
    constexpr bool kAhead = LOGM < 13;
    bool act[K];
    int la[K], ja[K], lm[K], jm[K], lo[K], jo[K];
#pragma unroll
    for (int u = 0; u < K; ++u) {
        const int role = (int)threadIdx.x + u * (int)blockDim.x;
        act[u] = role < B * TPL;
        lm[u] = role / TPL;
        jm[u] = role % TPL;
        la[u] = COL_IN ? role % B : lm[u];
        ja[u] = COL_IN ? role / B : jm[u];
        lo[u] = COL_OUT ? role % B : lm[u];
        jo[u] = COL_OUT ? role / B : jm[u];
    }
    // every load at a clamped index, so that none waits in a branch
    C v[K][8], h[K][8];
#pragma unroll
    for (int u = 0; u < K; ++u) {
        const int b = min(line0 + la[u], lines - 1);
        C c[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int p = min(ja[u] + q * TPL, tb.P - 1);
            v[u][q] = in[b * in_ls + p * in_es];
            c[q] = tb.cin[p];
        }
        if (scale_in && sl) {
            const T lsc = sl[b];
            T e[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) e[q] = se[min(ja[u] + q * TPL, tb.P - 1)];
#pragma unroll
            for (int q = 0; q < 8; ++q) v[u][q] = cscale(v[u][q], lsc * e[q]);
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            C x = v[u][q];
            if (conj) x = cconj(x);
            x = cmul_f(x, c[q]);
            v[u][q] = ja[u] + q * TPL < tb.P ? x : mk((T)0, (T)0);
        }
        if constexpr (kAhead)
#pragma unroll
            for (int q = 0; q < 8; ++q) h[u][q] = tb.hhat[(jm[u] + q * TPL) & (M - 1)];
    }
    czt_fft<T, LOGM, K>(v, lds, tb.tw, act, la, ja, lm, jm, lm, jm);
#pragma unroll
    for (int u = 0; u < K; ++u) {
        if constexpr (!kAhead)
#pragma unroll
            for (int q = 0; q < 8; ++q) h[u][q] = tb.hhat[(jm[u] + q * TPL) & (M - 1)];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[u][q] = cconj(cmul_f(v[u][q], h[u][q]));
    }
    __syncthreads();
    if constexpr (kAhead)
#pragma unroll
        for (int u = 0; u < K; ++u)
#pragma unroll
            for (int q = 0; q < 8; ++q) h[u][q] = tb.cout[min(jo[u] + q * TPL, tb.Q - 1)];
    czt_fft<T, LOGM, K>(v, lds, tb.tw, act, lm, jm, lm, jm, lo, jo);
    const T inv = (T)1 / (T)M;
#pragma unroll
    for (int u = 0; u < K; ++u) {
        const int b = line0 + lo[u];
        if (!act[u] || b >= lines) continue;
        const T lsc = !scale_in && sl ? sl[b] : (T)1;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int o = jo[u] + q * TPL;
            if (o < tb.Q) {
                if constexpr (!kAhead) h[u][q] = tb.cout[o];
                C x = cmul_f(cscale(cconj(v[u][q]), inv), h[u][q]);
                if (conj) x = cconj(x);
                if (!scale_in && sl) x = cscale(x, lsc * se[o]);
                out[b * out_ls + o * out_es] = x;
            }
        }
    }
}

// A plan's pass: one line per block where the lines are contiguous on both
// sides, else 4,096 values (512 roles) of neighbouring lines; one role per
// thread up to m = 8192, two at 16,384.  Neighbouring blocks go to
// one XCD (grid: a multiple of 8), so that the lines that share cache lines in
// the strided direction meet in one L2.
template <int LOGM, bool COL> constexpr int czt_block_lines() { return !COL || LOGM >= 12 ? 1 : 4096 >> LOGM; }
template <int LOGM> constexpr int czt_roles_per_thread() { return LOGM > 13 ? 2 : 1; }
template <int LOGM, bool COL> constexpr int czt_threads()
{
    return czt_block_lines<LOGM, COL>() * ((1 << LOGM) / 8) / czt_roles_per_thread<LOGM>();
}
template <typename T, int LOGM, bool COL> constexpr int czt_lds_bytes()
{
    return (int)sizeof(cplx<T>) * czt_block_lines<LOGM, COL>() * lds_line<1 << LOGM>();
}
template <typename T, int LOGM, bool COL_IN, bool COL_OUT>
__global__ __launch_bounds__((czt_threads<LOGM, COL_IN || COL_OUT>())) void k_czt(const cplx<T> *__restrict__ in, long long in_ls,
                                                            long long in_es, cplx<T> *__restrict__ out,
                                                            long long out_ls, long long out_es,
                                                            const T *__restrict__ sl, const T *__restrict__ se,
                                                            bool scale_in, bool conj, int lines, CztTables<T> tb)
{
    extern __shared__ unsigned char smem_raw[];
    constexpr int B = czt_block_lines<LOGM, COL_IN || COL_OUT>();
    const int line0 = xcd_block((int)blockIdx.x, (int)gridDim.x) * B;
    if (line0 >= lines) return;
    czt_lines<T, LOGM, B, czt_roles_per_thread<LOGM>(), COL_IN, COL_OUT>(
        line0, lines, reinterpret_cast<cplx<T> *>(smem_raw), in, in_ls, in_es, out, out_ls, out_es, sl, se, scale_in,
        conj, tb);
}

// Launches one chirp-z pass over `lines` lines: MODE 0 both sides contiguous
// along a line, 1 the input's lines side by side (in_ls = 1), 2 the output's.
template <typename T, int LOGM, int MODE>
int czt_launch_m(const CztTables<T> &tb, int lines, const cplx<T> *in, long long in_ls, long long in_es,
                        cplx<T> *out, long long out_ls, long long out_es, const T *sl, const T *se, bool scale_in,
                        bool conj, hipStream_t s)
{
    static std::once_flag once;
    static hipError_t attr = hipSuccess;
    auto kern = k_czt<T, LOGM, MODE == 1, MODE == 2>;
    constexpr int bytes = czt_lds_bytes<T, LOGM, MODE != 0>();
    std::call_once(once, [&] {
        attr = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    });
    if (attr != hipSuccess) return nfft2d_fail(NFFT2D_ERR_HIP, "chirp-z pass: %s", hipGetErrorString(attr));
    constexpr int B = czt_block_lines<LOGM, MODE != 0>();
    const unsigned blocks = ((unsigned)(lines + B - 1) / B + 7) & ~7u;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(czt_threads<LOGM, MODE != 0>()), bytes, s, in, in_ls, in_es, out, out_ls, out_es,
                       sl, se, scale_in, conj, lines, tb);
    NFFT2D_LAUNCH_CHECK();
    return NFFT2D_OK;
}
template <typename T, int MODE, int LOGM = kCztMinLog, typename... A>
int czt_launch(const CztTables<T> &tb, A... a)
{
    if (tb.m == 1 << LOGM) return czt_launch_m<T, LOGM, MODE>(tb, a...);
    if constexpr (LOGM < kCztMaxLog<T>)
        return czt_launch<T, MODE, LOGM + 1>(tb, a...);
    else
        return nfft2d_fail(NFFT2D_ERR_SIZE, "chirp-z pass: no transform of %d points", tb.m);
}

}  // namespace nfft2d

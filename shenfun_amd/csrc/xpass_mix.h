// Fused x-pass (DCT-II -> stencil -> Helmholtz solve -> to_ortho -> DCT-III) on
// the plan's restart states for lengths with prime factors up to 13: the
// mixed-radix passes of fft_mixed.h around helm_chain_solve_bs.
//
// A workgroup takes 8 neighbouring lines (one 128-byte segment per x row) with
// 32 threads each: 16 segments of the even chain and 16 of the odd one.  The
// FFT passes map lanes over lines; everything between the two FFTs belongs to
// the line's own 32 lanes, half a wave, so it needs no workgroup barrier.  Each
// step reads its line's values, holds them in registers and writes the next
// form into the same LDS area: FFT outputs (digit order) -> solution (natural
// order) -> DCT-III inputs.
//
// It replaces a form without a plan (a scan of normalised 3 x 3 products with
// IEEE divides per row, one LDS step per phase on two buffers): that was bound
// by its arithmetic, 260 us at 180 x 150 x 101 lines Neumann against 17 us for
// the array at copy speed.
#pragma once
#include "fft_mixed.h"
#include "fft_pow2.h"
#include "helm_scan.h"

namespace sfa {

constexpr int XM_T = 8;
constexpr int XM_THREADS = 256;

struct XMixArgs {
    double2* W;       // element (x, L) of array b at W[b bstride + x sa + L], L = ky Kp + kz
    int64_t sa, bstride, nl;
    int Kp, Nzh;
    int N, LS;        // length, LDS elements between lines
    int neumann;
    double alpha;
    const double* K2;
    XPlan pl;
    const double2* tw;  // exp(-2 pi i m / N)
    const double2* tq;  // exp(-i pi k / (2N))
    MixPlan plan;
};

// E rows per lane (as in the plan).
template <int E>
__global__ void __launch_bounds__(XM_THREADS, E <= 6 ? 3 : 1) xpass_mix_kernel(XMixArgs a)
{
    extern __shared__ double2 smem[];
    constexpr int T = XM_T, PADW = 2 * E;
    auto pd = [](int k) { return k + k / PADW; };
    const MixPlan& pl = a.plan;
    const int tid = threadIdx.x, nth = XM_THREADS;
    const int N = a.N, M = N - 2, LS = a.LS;
    const int64_t L0 = (int64_t)blockIdx.x * T;
    double2* W = a.W + (int64_t)blockIdx.y * a.bstride + L0;
    const int64_t sa = a.sa;
    MixTile m;
    m.T = T;
    m.Tv = (int)((a.nl - L0) < T ? (a.nl - L0) : T);
    m.shift = 3;
    m.ps = 1;
    m.ts = LS;
    m.t_fast = true;
    const int twT = T * LS, tqs = twT + N, t0s = tqs + N;
    // this thread's chain: line t, parity p, segment lane
    const int t = tid >> 5, p = (tid >> 4) & 1, lane = tid & 15, l32 = tid & 31;
    int u;
    {
        const uint32_t L = (uint32_t)(L0 + t), ky = L / (uint32_t)a.Kp, kz = L - ky * (uint32_t)a.Kp;
        const bool ok = t < m.Tv && kz < (uint32_t)a.Nzh;  // else absent, or a pitch-padding line
        const int v = a.pl.linemap[ok ? ky * a.Nzh + kz : 0];
        u = ok ? v : 0;
    }
    mix_twiddles(pl, twT, a.tw, tid, nth);
    for (int i = tid; i < N; i += nth) lds_put(tqs + i, a.tq[i]);

    // 1. DCT-II: the FFT of the even/odd permuted line
    mix_first<false>(
        pl, m, 0, twT, tid, nth, [&](int tt, int) -> int64_t { return tt; }, 0,
        [&](int64_t o, int, int i) { return W[o + (2 * i < N ? 2 * i : 2 * (N - 1 - i) + 1) * sa]; },
        [](int, int) -> int64_t { return 0; }, 0,
        [&](int64_t, int tt, int, int pos, double2 v) { lds_put(pos + tt * LS, v); });
    const double be = a.alpha + a.pl.svals[u];
    const double4 b4 = a.pl.bs[((int64_t)2 * u + p) * 16 + lane];
    mix_rest<false>(
        pl, m, 0, a.tw, tid, nth, [](int, int) -> int64_t { return 0; }, 0,
        [&](int64_t, int tt, int, int pos, double2 v) { lds_put(pos + tt * LS, v); });
    __syncthreads();

    // 2. X_k = sc (Re(w (V_k + conj V_{N-k})) + i Im(w (V_k - conj V_{N-k}))), stencil
    const int ln = t * LS;
    const double sc = 3.14159265358979323846 / (2.0 * N);
    auto coef = [&](int k) {
        const double2 P = lds_get(ln + mix_pos(pl, k)), Q = cconj(lds_get(ln + mix_pos(pl, k == 0 ? 0 : N - k)));
        const double2 w = lds_get(tqs + k);
        return make_double2(cmul(w, cadd(P, Q)).x * sc, cmul(w, csub(P, Q)).y * sc);
    };
    double2 f[E];
    {
        const int i0 = 2 * lane * E + p;
        double2 x0 = coef(i0 < N ? i0 : 0);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = i0 + 2 * e;
            const double2 x2 = coef(i + 2 < N ? i + 2 : 0);
            const double kk = a.K2[i < M ? i : 0];
            f[e] = i < M ? make_double2(x0.x + kk * x2.x, x0.y + kk * x2.y) : make_double2(0.0, 0.0);
            x0 = x2;
        }
    }
    wave_sync();
    // 3. Helmholtz solve of both chains into natural order, boundary slots zero
    double2* X = smem + ln;
    helm_chain_solve_bs<E, 16, double2, PADW>(f, X, p, M, be, a.neumann != 0, b4, lane);
    if (lane == 0) X[pd(M + p)] = make_double2(0.0, 0.0);
    wave_sync();
    // 4. to_ortho t_k = u_k + K2_{k-2} u_{k-2} (u = 0 in the slots), and the
    // DCT-III inputs V_k = conj(w_k) (t_k - i t_{N-k}), k = l32 + 32 r
    constexpr int NV = E + 1;  // N <= 32 E + 2
    double2 v[NV];
    auto ortho = [&](int k) {
        const double2 x = lds_get(ln + pd(k)), y = lds_get(ln + pd(k >= 2 ? k - 2 : 0));
        const double kk = k >= 2 ? a.K2[k - 2] : 0.0;
        return make_double2(x.x + kk * y.x, x.y + kk * y.y);
    };
#pragma unroll
    for (int r = 0; r < NV; ++r) {
        const int k = l32 + 32 * r;
        const int kc = k < N ? k : 0;
        const double2 ck = ortho(kc);
        double2 cn = ortho(kc == 0 ? 0 : N - kc);
        if (kc == 0) cn = make_double2(0.0, 0.0);
        v[r] = cmul(cconj(lds_get(tqs + kc)), make_double2(ck.x + cn.y, ck.y - cn.x));
        if (k == 0) lds_put(t0s + t, ck);
    }
    wave_sync();
    const float inv_nb = 1.0f / (float)pl.sub[0];
#pragma unroll
    for (int r = 0; r < NV; ++r) {
        const int k = l32 + 32 * r;
        if (k < N) lds_put(ln + mix_in_pos(pl, k, inv_nb), v[r]);
    }
    __syncthreads();
    // 5. DCT-III: inverse FFT, 0.5 y + t_0 / 2 with the inverse permutation
    auto st = [&](int64_t, int tt, int k, int, double2 y) {
        const double2 c0 = lds_get(t0s + tt);
        W[tt + (2 * k < N ? 2 * k : 2 * (N - 1 - k) + 1) * sa] =
            make_double2(0.5 * y.x + 0.5 * c0.x, 0.5 * y.y + 0.5 * c0.y);
    };
    mix_first<true>(
        pl, m, 0, twT, tid, nth, [&](int tt, int j) -> int64_t { return j + tt * LS; }, pl.P,
        [&](int64_t o, int, int) { return lds_get((int)o); }, [](int, int) -> int64_t { return 0; }, 0, st);
    mix_rest<true>(pl, m, 0, a.tw, tid, nth, [](int, int) -> int64_t { return 0; }, 0, st);
}

// The solve alone, in place on the stencilled coefficients: for the lengths with
// larger prime factors, between a DCT-II and a DCT-III of their own (three passes
// over the array; 218 x 38 x 144 lines 1042 us in the form without a plan, 160
// in this one).  The same workgroup and plan as above.
template <int E>
__global__ void __launch_bounds__(XM_THREADS) xsolve_kernel(XMixArgs a)
{
    extern __shared__ double2 smem[];
    constexpr int T = XM_T, PADW = 2 * E;
    auto pd = [](int k) { return k + k / PADW; };
    const int tid = threadIdx.x;
    const int N = a.N, M = N - 2, LS = a.LS;
    const int64_t L0 = (int64_t)blockIdx.x * T, sa = a.sa;
    double2* W = a.W + (int64_t)blockIdx.y * a.bstride + L0;
    const int Tv = (int)((a.nl - L0) < T ? (a.nl - L0) : T);
    const int t = tid >> 5, p = (tid >> 4) & 1, lane = tid & 15;
    int u;
    {
        const uint32_t L = (uint32_t)(L0 + t), ky = L / (uint32_t)a.Kp, kz = L - ky * (uint32_t)a.Kp;
        const bool ok = t < Tv && kz < (uint32_t)a.Nzh;
        const int v = a.pl.linemap[ok ? ky * a.Nzh + kz : 0];
        u = ok ? v : 0;
    }
    // lanes over lines for the array, over segments for the solve
    const int tl = tid & (T - 1), r0 = tid >> 3, tc = tl < Tv ? tl : 0;
#pragma unroll 4
    for (int i = r0; i < M; i += XM_THREADS / T) lds_put(tl * LS + pd(i), W[tc + i * sa]);
    const double be = a.alpha + a.pl.svals[u];
    const double4 b4 = a.pl.bs[((int64_t)2 * u + p) * 16 + lane];
    __syncthreads();
    double2 f[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = 2 * (lane * E + e) + p;
        const double2 v = lds_get(t * LS + pd(i < M ? i : 0));
        f[e] = i < M ? v : make_double2(0.0, 0.0);
    }
    wave_sync();
    helm_chain_solve_bs<E, 16, double2, PADW>(f, smem + t * LS, p, M, be, a.neumann != 0, b4, lane);
    __syncthreads();
    if (tl < Tv) {
#pragma unroll 4
        for (int i = r0; i < M; i += XM_THREADS / T) W[tl + i * sa] = lds_get(tl * LS + pd(i));
        if (r0 < 2) W[tl + (M + r0) * sa] = make_double2(0.0, 0.0);  // boundary slots
    }
}

inline size_t xpass_mix_lds(const XMixArgs& a)
{
    return sizeof(double2) * ((size_t)XM_T * a.LS + 2 * (size_t)a.N + XM_T);
}

// The x-pass, or the solve alone where the plan has no passes (a.plan.np == 0).
template <int E>
int xpass_mix_run(const XMixArgs& a, int64_t nb, hipStream_t s)
{
    auto k = a.plan.np ? xpass_mix_kernel<E> : xsolve_kernel<E>;
    const size_t lds = xpass_mix_lds(a);
    if (lds > 64 * 1024)
        SFA_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k, dim3((unsigned)((a.nl + XM_T - 1) / XM_T), (unsigned)nb), dim3(XM_THREADS), lds, s, a);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

// one translation unit each
int xpass_mix_1(const XMixArgs& a, int64_t nb, hipStream_t s);
int xpass_mix_2(const XMixArgs& a, int64_t nb, hipStream_t s);
int xpass_mix_3(const XMixArgs& a, int64_t nb, hipStream_t s);
int xpass_mix_4(const XMixArgs& a, int64_t nb, hipStream_t s);
int xpass_mix_6(const XMixArgs& a, int64_t nb, hipStream_t s);
int xpass_mix_8(const XMixArgs& a, int64_t nb, hipStream_t s);
int xpass_mix_12(const XMixArgs& a, int64_t nb, hipStream_t s);
int xpass_mix_16(const XMixArgs& a, int64_t nb, hipStream_t s);

}  // namespace sfa

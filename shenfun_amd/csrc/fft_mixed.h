// Mixed-radix line FFT (FP64) for the lengths the power-of-two kernels do not
// take: N = R_1 R_2 .. R_np with every R_l <= 16, as few passes as the factors
// allow (two up to 256, three up to 4096).
//
// Decimation in frequency, in place: pass l takes the R_l values of a butterfly
// into registers, transforms them, multiplies by the twiddles and puts them
// back where they came from, so one LDS buffer serves every pass with one
// barrier between two of them.  The first pass takes its values from wherever
// the caller reads them (global memory, with the transform's own
// pre-processing) and the last one hands them to the caller, so a plain
// complex transform touches LDS np - 1 times.
//
// Value (q_1, .., q_{l}, j) of a line, after pass l, lies at
// pos = q_1 P + q_2 n_2 + .. + q_l n_l + j with n_l = N / (R_1 .. R_l); P is n_1,
// made odd where lanes run along the line, so that lanes P apart meet
// different banks.  Output k = q_1 + R_1 (q_2 + R_2 (q_3 + ..)).
#pragma once
#include "fft_device.h"

namespace sfa {

constexpr int kMixMaxRadix = 16;
constexpr int kMixMaxPasses = 4;

struct MixPlan {
    int n;                      // length
    int np;                     // passes
    int r[kMixMaxPasses];       // radices
    int sub[kMixMaxPasses];     // n_l, l = 1 .. np (sub[np - 1] = 1)
    int P;                      // distance of two q_1 rows in LDS
    unsigned magic[kMixMaxPasses];  // 2^20 / r[l] rounded up: k / r[l] for k < 2^12
    __host__ __device__ int size() const { return r[0] * P; }  // LDS elements of a line
};

// Host: the plan of length n with row distance n_1 (odd = 0) or n_1 | 1; false
// if a prime factor exceeds 13 or the passes are too many.
inline bool make_mix_plan(int n, bool odd, MixPlan* p)
{
    if (n < 1 || n > 4096) return false;
    int best[kMixMaxPasses], cur[kMixMaxPasses];
    int bn = 0, bsum = 1 << 30;
    // all factorisations into non-increasing radices <= 16, the fewest passes
    // first, then the smallest sum (arithmetic and registers)
    struct Rec {
        static void go(int m, int top, int depth, int* cur, int* best, int& bn, int& bsum)
        {
            if (m == 1) {
                int s = 0;
                for (int i = 0; i < depth; ++i) s += cur[i];
                if (bn == 0 || depth < bn || (depth == bn && s < bsum)) {
                    bn = depth;
                    bsum = s;
                    for (int i = 0; i < depth; ++i) best[i] = cur[i];
                }
                return;
            }
            if (depth == kMixMaxPasses) return;
            for (int r = top < m ? top : m; r >= 2; --r)
                if (m % r == 0) {
                    cur[depth] = r;
                    go(m / r, r, depth + 1, cur, best, bn, bsum);
                }
        }
    };
    if (n == 1) {
        bn = 1;
        best[0] = 1;
    } else {
        Rec::go(n, kMixMaxRadix, 0, cur, best, bn, bsum);
    }
    if (bn == 0) return false;
    p->n = n;
    p->np = bn;
    int m = n;
    for (int l = 0; l < kMixMaxPasses; ++l) {
        p->r[l] = l < bn ? best[l] : 1;
        m /= p->r[l];
        p->sub[l] = m;
        p->magic[l] = ((1u << 20) + p->r[l] - 1) / p->r[l];
    }
    p->P = odd ? (p->sub[0] | 1) : p->sub[0];
    return true;
}

// cos and sin of 2 pi m / R, folded at compile time
template <int R>
struct Root {
    static constexpr double PI2 = 6.283185307179586476925286766559;
    template <int M>
    __device__ static inline double c()
    {
        constexpr int m = M % R;
        return __builtin_cos(PI2 * m / R);
    }
    template <int M>
    __device__ static inline double s()
    {
        constexpr int m = M % R;
        return __builtin_sin(PI2 * m / R);
    }
};

template <int I>
struct IC {
    static constexpr int v = I;
};

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F f)
{
    if constexpr (I < N) {
        f(IC<I>{});
        static_for<I + 1, N>(f);
    }
}

// a * exp(-+ 2 pi i M / R)
template <int R, int M, bool INV>
__device__ inline double2 root_mul(double2 a)
{
    constexpr int m = M % R;
    if constexpr (m == 0) return a;
    else if constexpr (16 % R == 0) return tw16<m * (16 / R), INV>(a);
    else if constexpr (2 * m == R) return make_double2(-a.x, -a.y);
    else if constexpr (4 * m == R) return tw16<4, INV>(a);
    else if constexpr (4 * m == 3 * R) return tw16<12, INV>(a);
    else {
        const double c = Root<R>::template c<m>();
        const double s = INV ? Root<R>::template s<m>() : -Root<R>::template s<m>();
        return make_double2(a.x * c - a.y * s, a.x * s + a.y * c);
    }
}

// odd prime R: the sums and differences of a_r and a_{R-r} halve the products
template <int R, bool INV>
__device__ inline void dft_prime(double2* a)
{
    constexpr int H = (R - 1) / 2;
    double2 sp[H], sm[H];
#pragma unroll
    for (int r = 0; r < H; ++r) {
        sp[r] = cadd(a[r + 1], a[R - 1 - r]);
        sm[r] = csub(a[r + 1], a[R - 1 - r]);
    }
    const double2 a0 = a[0];
    static_for<1, H + 1>([&](auto Q) {
        constexpr int q = decltype(Q)::v;
        double2 e = a0, o = make_double2(0.0, 0.0);
        static_for<1, H + 1>([&](auto RR) {
            constexpr int r = decltype(RR)::v;
            const double c = Root<R>::template c<q * r>(), s = Root<R>::template s<q * r>();
            e.x += sp[r - 1].x * c;
            e.y += sp[r - 1].y * c;
            o.x += sm[r - 1].x * s;
            o.y += sm[r - 1].y * s;
        });
        // forward: e - i o, inverse: e + i o
        const double2 u = make_double2(e.x + o.y, e.y - o.x), v = make_double2(e.x - o.y, e.y + o.x);
        a[q] = INV ? v : u;
        a[R - q] = INV ? u : v;
    });
    double2 s0 = a0;
#pragma unroll
    for (int r = 0; r < H; ++r) s0 = cadd(s0, sp[r]);
    a[0] = s0;
}

template <int R, bool INV>
__device__ inline void mix_dft(double2* a);

// R = A B, input r = B r1 + r2, output q = q1 + A q2
template <int A, int B, bool INV>
__device__ inline void dft_comp(double2* a)
{
    double2 c[A * B];
    static_for<0, B>([&](auto R2) {
        constexpr int r2 = decltype(R2)::v;
        double2 x[A];
#pragma unroll
        for (int r1 = 0; r1 < A; ++r1) x[r1] = a[B * r1 + r2];
        mix_dft<A, INV>(x);
        static_for<0, A>([&](auto Q1) {
            constexpr int q1 = decltype(Q1)::v;
            c[q1 * B + r2] = root_mul<A * B, r2 * q1, INV>(x[q1]);
        });
    });
#pragma unroll
    for (int q1 = 0; q1 < A; ++q1) {
        double2 x[B];
#pragma unroll
        for (int r2 = 0; r2 < B; ++r2) x[r2] = c[q1 * B + r2];
        mix_dft<B, INV>(x);
#pragma unroll
        for (int q2 = 0; q2 < B; ++q2) a[q1 + A * q2] = x[q2];
    }
}

template <int R, bool INV>
__device__ inline void mix_dft(double2* a)
{
    if constexpr (R == 1) return;
    else if constexpr (R == 2 || R == 4 || R == 8 || R == 16) dft<R, INV>(a);
    else if constexpr (R == 6) dft_comp<2, 3, INV>(a);
    else if constexpr (R == 9) dft_comp<3, 3, INV>(a);
    else if constexpr (R == 10) dft_comp<2, 5, INV>(a);
    else if constexpr (R == 12) dft_comp<4, 3, INV>(a);
    else if constexpr (R == 14) dft_comp<2, 7, INV>(a);
    else if constexpr (R == 15) dft_comp<3, 5, INV>(a);
    else dft_prime<R, INV>(a);
}

// f(IC<R>) for the run-time radix r
template <class F>
__device__ __forceinline__ void radix_switch(int r, F f)
{
    switch (r) {
        case 2: f(IC<2>{}); break;
        case 3: f(IC<3>{}); break;
        case 4: f(IC<4>{}); break;
        case 5: f(IC<5>{}); break;
        case 6: f(IC<6>{}); break;
        case 7: f(IC<7>{}); break;
        case 8: f(IC<8>{}); break;
        case 9: f(IC<9>{}); break;
        case 10: f(IC<10>{}); break;
        case 11: f(IC<11>{}); break;
        case 12: f(IC<12>{}); break;
        case 13: f(IC<13>{}); break;
        case 14: f(IC<14>{}); break;
        case 15: f(IC<15>{}); break;
        case 16: f(IC<16>{}); break;
        default: f(IC<1>{}); break;
    }
}

// Element i of the workgroup's dynamic LDS: addressed from the array itself, so
// that the compiler sees LDS accesses wherever an offset has been.
__device__ __forceinline__ double2 lds_get(int i)
{
    extern __shared__ double2 smem[];
    return smem[i];
}
__device__ __forceinline__ void lds_put(int i, double2 v)
{
    extern __shared__ double2 smem[];
    smem[i] = v;
}

// How a block's lines lie in LDS and how its threads take butterflies: value
// pos of line t at pos * ps + t * ts.  t_fast: T (a power of two) lines
// interleaved, a wave's lanes over lines; else lanes along the line.
struct MixTile {
    int T, Tv, shift;  // lines, valid lines, log2 T (t_fast)
    int ps, ts;
    bool t_fast;
};

__device__ __forceinline__ int mix_div(int k, unsigned magic) { return (int)(((unsigned)k * magic) >> 20); }

// x unchanged, but unknown to the optimiser: a running offset stays an add per
// element instead of a scalar product per (radix, element), which the switch
// over radices had hoisted into more scalar registers than there are.
template <class I>
__device__ __forceinline__ I running(I x)
{
    asm volatile("" : "+v"(x));
    return x;
}

// This thread's (line t, index k < len) pairs: the elements tid, tid + nth, ..
// of the tile, lines fastest (t_fast) or k fastest, without a division per step.
struct MixIter {
    int t, k, dt, dk, len, Tv;
    bool t_fast;
    __device__ __forceinline__ MixIter(const MixTile& m, int n, int tid, int nth) : len(n), Tv(m.Tv), t_fast(m.t_fast)
    {
        if (t_fast) {
            t = tid & (m.T - 1);
            k = tid >> m.shift;
            dt = 0;
            dk = nth >> m.shift;
        } else {
            const float inv = 1.0f / (float)n;
            t = div(tid, inv);
            k = tid - t * n;
            dt = div(nth, inv);
            dk = nth - dt * n;
        }
    }
    __device__ __forceinline__ int div(int x, float inv) const  // x < 2^16
    {
        int q = (int)((float)x * inv);
        const int r = x - q * len;
        if (r < 0) --q;
        if (r >= len) ++q;
        return q;
    }
    __device__ __forceinline__ bool done() const { return t_fast ? k >= len : t >= Tv; }
    __device__ __forceinline__ bool here() const { return t < Tv && k < len; }
    __device__ __forceinline__ void next()
    {
        t += dt;
        k += dk;
        if (!t_fast && k >= len) {
            k -= len;
            ++t;
        }
    }
};

// LDS position of output k
__device__ __forceinline__ int mix_pos(const MixPlan& pl, int k)
{
    if (pl.np == 1) return k * pl.P;
    int d = mix_div(k, pl.magic[0]);
    int pos = (k - d * pl.r[0]) * pl.P;
#pragma unroll
    for (int l = 1; l < kMixMaxPasses - 1; ++l) {
        if (l >= pl.np - 1) break;
        const int q = d;
        d = mix_div(q, pl.magic[l]);
        pos += (q - d * pl.r[l]) * pl.sub[l];
    }
    return pos + d;
}

// twT, buf: offsets in LDS.  twT (n entries): the first pass' twiddles,
// exp(-2 pi i q j / n) at q n_1 + j, from tw = exp(-2 pi i m / n) (global):
// lanes along the line read neighbours (tw[j q] strides by q, a bank conflict
// for every even q).
__device__ __forceinline__ void mix_twiddles(const MixPlan& pl, int twT, const double2* __restrict__ tw, int tid,
                                             int nth)
{
    const int nb = pl.sub[0];
    const float inv_nb = 1.0f / (float)nb;
    for (int i = tid; i < pl.n; i += nth) {
        int q = (int)((float)i * inv_nb);
        int j = i - q * nb;
        if (j < 0) { --q; j += nb; }
        if (j >= nb) { ++q; j -= nb; }
        lds_put(twT + i, tw[q * j]);
    }
}

// LDS position of input i before a first pass that reads LDS (mix_staged):
// rows of n_1 inputs P apart, so that a butterfly's inputs and outputs share
// their places.
__device__ __forceinline__ int mix_in_pos(const MixPlan& pl, int i, float inv_nb)
{
    int r = (int)((float)i * inv_nb);
    int j = i - r * pl.sub[0];
    if (j < 0) { --r; j += pl.sub[0]; }
    if (j >= pl.sub[0]) { ++r; j -= pl.sub[0]; }
    return r * pl.P + j;
}

// First pass.  at = lb(t, j) is where the caller's input j of line t lies, ls
// how far apart the inputs j + r n_1 are, and ld(at, t, j + r n_1) reads one;
// the outputs go to buf, or with np == 1 straight to the caller as in mix_rest.
// A barrier lies between the loads of a thread's first butterfly and its
// twiddles, for what the caller has put in LDS (twT among it); with inputs in
// LDS the caller puts one before the call too.
template <bool INV, class LB, class LD, class SB, class ST>
__device__ __forceinline__ void mix_first(const MixPlan& pl, const MixTile& m, int buf, int twT, int tid, int nth,
                                          LB lb, int64_t ls, LD ld, SB sb, int64_t ss, ST st)
{
    const int nb = pl.sub[0], step = pl.P * m.ps;
    radix_switch(pl.r[0], [&](auto RC) {
        constexpr int R = decltype(RC)::v;
        MixIter it(m, nb, tid, nth);
        double2 a[R];
        auto take = [&]() {
            int64_t o = lb(it.t, it.k);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                a[r] = ld(o, it.t, it.k + r * nb);
                o = running(o + ls);
            }
        };
        if (it.here()) take();
        __syncthreads();
        while (!it.done()) {
            if (it.here()) {
                const int j = it.k, t = it.t;
                mix_dft<R, INV>(a);
                if (pl.np == 1) {
                    int64_t o = sb(t, 0);
#pragma unroll
                    for (int q = 0; q < R; ++q) {
                        st(o, t, q, q * pl.P, a[q]);
                        o = running(o + ss);
                    }
                } else {
                    // the twiddles in groups of 5: all 15 of a radix 16 at once
                    // held 60 registers more
                    int w0 = twT + nb + j, o = buf + j * m.ps + t * m.ts;
                    lds_put(o, a[0]);
#pragma unroll
                    for (int q0 = 1; q0 < R; q0 += 5) {
                        double2 w[5];
#pragma unroll
                        for (int i = 0; i < 5; ++i)
                            if (q0 + i < R) {
                                w[i] = lds_get(w0);
                                w0 = running(w0 + nb);
                            }
#pragma unroll
                        for (int i = 0; i < 5; ++i)
                            if (q0 + i < R) {
                                if (INV) w[i].y = -w[i].y;
                                o = running(o + step);
                                lds_put(o, cmul(a[q0 + i], w[i]));
                            }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            it.next();
            if (it.here()) take();
        }
    });
}

// Passes 2 .. np, each after a barrier; output k of line t goes to
// st(at, t, k, pos, value) with at = sb(t, k) (k a butterfly's first output,
// then ss further for each k after it).  st may put it at pos of buf (=
// mix_pos(k)): that is in place.  tw: exp(-2 pi i m / n), global.
template <bool INV, class SB, class ST>
__device__ __forceinline__ void mix_rest(const MixPlan& pl, const MixTile& m, int buf, const double2* __restrict__ tw,
                                         int tid, int nth, SB sb, int64_t ss, ST st)
{
    for (int l = 1; l < pl.np; ++l) {
        __syncthreads();
        const int nb = pl.n / pl.r[l];
        const int nl = pl.sub[l], step = nl * m.ps;
        const int tws = pl.n / pl.sub[l - 1];
        const bool last = l == pl.np - 1;
        const int kr = pl.n / pl.r[l];  // last pass: R_1 .. R_{np-1}
        const int64_t sstep = ss * kr;
        radix_switch(pl.r[l], [&](auto RC) {
            constexpr int R = decltype(RC)::v;
            for (MixIter it(m, nb, tid, nth); !it.done(); it.next()) {
                if (!it.here()) continue;
                const int t = it.t;
                // g = q_1 + R_1 (rest); rest: q_2 .. q_{l-1} and the j of this pass
                int rest = mix_div(it.k, pl.magic[0]);
                const int q1 = it.k - rest * pl.r[0];
                int pos = q1 * pl.P;
#pragma unroll
                for (int i = 1; i < kMixMaxPasses - 1; ++i) {
                    if (i >= l) break;
                    const int d = mix_div(rest, pl.magic[i]);
                    pos += (rest - d * pl.r[i]) * pl.sub[i];
                    rest = d;
                }
                const int j = rest;
                pos += j;
                double2 a[R];
                const int o0 = buf + pos * m.ps + t * m.ts;
                int o = o0;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    a[r] = lds_get(o);
                    o = running(o + step);
                }
                mix_dft<R, INV>(a);
                if (last) {  // rest = 0: g is the butterfly's first output
                    int64_t so = sb(t, it.k);
                    int k = it.k;
#pragma unroll
                    for (int q = 0; q < R; ++q) {
                        st(so, t, k, pos + q, a[q]);
                        so = running(so + sstep);
                        k = running(k + kr);
                    }
                } else {
                    int w0 = 0;
#pragma unroll
                    for (int q = 1; q < R; ++q) {
                        w0 = running(w0 + j * tws);
                        double2 w = tw[w0];
                        if (INV) w.y = -w.y;
                        a[q] = cmul(a[q], w);
                    }
                    o = o0;
#pragma unroll
                    for (int q = 0; q < R; ++q) {
                        lds_put(o, a[q]);
                        o = running(o + step);
                    }
                }
            }
        });
    }
}

}  // namespace sfa

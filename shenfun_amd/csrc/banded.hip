// Banded solves along one axis of strided 1-3D arrays (FP64 factors,
// float64 or complex128 right-hand sides).  All band offsets are even, so the
// even and odd unknowns form two independent chains.  The TDMA and Helmholtz
// solves cut a chain into segments, a thread each (chain_solve_kernel); the
// diagonal solve takes a thread per element; the others a thread per (line,
// parity) chain, consecutive threads on consecutive lines so every step of the
// recurrence is a coalesced access across the wave.
#include "common.h"

namespace sfa {

__device__ inline double sub_mul(double a, double s, double b) { return a - s * b; }
__device__ inline double2 sub_mul(double2 a, double s, double2 b)
{
    return make_double2(a.x - s * b.x, a.y - s * b.y);
}
__device__ inline double mul(double a, double s) { return a * s; }
__device__ inline double2 mul(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
__device__ inline double divd(double a, double s) { return a / s; }
__device__ inline double2 divd(double2 a, double s) { return make_double2(a.x / s, a.y / s); }
__device__ inline double add(double a, double b) { return a + b; }
__device__ inline double2 add(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
template <typename T>
__device__ inline T zero();
template <>
__device__ inline double zero<double>() { return 0.0; }
template <>
__device__ inline double2 zero<double2>() { return make_double2(0.0, 0.0); }

struct LineMap {
    int64_t sa, s1, s2, d2, nlines;
    __device__ inline int64_t off(int64_t L) const
    {
        const int64_t i1 = L / d2;
        return i1 * s1 + (L - i1 * d2) * s2;
    }
};

__device__ inline int last_of_parity(int n, int p) { return (n - 1) - (((n - 1) - p) & 1); }

// ----------------------------------------------------------------- TDMA
__global__ void tdma_lu_kernel(double* __restrict__ data, int n, int64_t nbatch)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= 2 * nbatch) return;
    const int p = (int)(gid / nbatch);
    const int64_t b = gid - (int64_t)p * nbatch;
    double* ld = data + b * 3 * n;
    double* d = ld + n;
    double* ud = ld + 2 * n + 2;
    for (int i = p + 2; i < n; i += 2) {
        ld[i - 2] = ld[i - 2] / d[i - 2];
        d[i] = d[i] - ld[i - 2] * ud[i - 2];
    }
}

// ----------------------------------------------------------------- PDMA
template <typename T>
__global__ void pdma_solve_kernel(T* __restrict__ u, LineMap g, const double* __restrict__ data,
                                  int n, int64_t dls, int64_t skip)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nl = g.nlines;
    if (gid >= 2 * nl) return;
    const int p = (int)(gid / nl);
    const int64_t L = gid - (int64_t)p * nl;
    if (L < skip || p >= n) return;
    T* v = u + g.off(L);
    const int64_t sa = g.sa;
    const double* a = data + L * dls;
    const double* b = a + n;
    const double* d = a + 2 * n;
    const double* e = a + 3 * n + 2;
    const double* f = a + 4 * n + 4;
    // forward
    T pm2 = v[p * sa];  // u[i-2]
    T pm4 = zero<T>();  // u[i-4]
    if (p + 2 < n) {
        T cur = sub_mul(v[(p + 2) * sa], b[p], pm2);
        v[(p + 2) * sa] = cur;
        pm4 = pm2;
        pm2 = cur;
    }
    for (int k = p + 4; k < n; k += 2) {
        T s = add(mul(pm2, b[k - 2]), mul(pm4, a[k - 4]));
        T cur = add(v[k * sa], mul(s, -1.0));
        v[k * sa] = cur;
        pm4 = pm2;
        pm2 = cur;
    }
    // backward
    const int il = last_of_parity(n, p);
    T n2 = divd(v[il * sa], d[il]);  // u[k+2]
    v[il * sa] = n2;
    T n4 = zero<T>();                // u[k+4]
    if (il - 2 >= 0) {
        T cur = divd(sub_mul(v[(il - 2) * sa], e[il - 2], n2), d[il - 2]);
        v[(il - 2) * sa] = cur;
        n4 = n2;
        n2 = cur;
    }
    for (int k = il - 4; k >= 0; k -= 2) {
        T cur = divd(sub_mul(sub_mul(v[k * sa], e[k], n2), f[k], n4), d[k]);
        v[k * sa] = cur;
        n4 = n2;
        n2 = cur;
    }
}

__global__ void pdma_lu_kernel(double* __restrict__ data, int n, int64_t nbatch)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= 2 * nbatch) return;
    const int p = (int)(gid / nbatch);
    const int64_t bb = gid - (int64_t)p * nbatch;
    double* a = data + bb * 5 * n;
    double* b = a + n;
    double* d = a + 2 * n;
    double* e = a + 3 * n + 2;
    double* f = a + 4 * n + 4;
    for (int i = p; i < n - 4; i += 2) {
        double lam = b[i] / d[i];
        d[i + 2] -= lam * e[i];
        e[i + 2] -= lam * f[i];
        b[i] = lam;
        lam = a[i] / d[i];
        b[i + 2] -= lam * e[i];
        d[i + 4] -= lam * f[i];
        a[i] = lam;
    }
    for (int i = n - 4; i <= n - 3; ++i) {
        if (i < 0 || ((i & 1) != p)) continue;
        const double lam = b[i] / d[i];
        d[i + 2] -= lam * e[i];
        b[i] = lam;
    }
}

// ----------------------------------------------------------------- DiagMA
// One thread per element, lanes along the line where the axis is the
// contiguous one and over lines otherwise.
template <typename T>
__global__ void diag_solve_kernel(T* __restrict__ u, LineMap g, const double* __restrict__ dd,
                                  int n, int64_t dls, int64_t skip, int along)
{
    const int64_t gid = wide_block() * blockDim.x + threadIdx.x;
    if (gid >= g.nlines * n) return;
    const int64_t L = along ? gid / n : gid % g.nlines;
    const int i = (int)(along ? gid - L * n : gid / g.nlines);
    if (L < skip) return;
    T* v = u + g.off(L) + (int64_t)i * g.sa;
    *v = divd(*v, dd[L * dls + i]);
}

// ----------------------------------------------------------------- other band patterns
// TwoDMA (offsets 0, 2), ThreeDMA (0, 2, 4), FDMA (-2, 0, 2, 4) and HeptaDMA
// (-4, -2, 0, 2, 4, 6, 8) with S = 2 (two parity chains per line), and the
// odd-offset TDMA_O (-1, 0, 1) with S = 1 (one chain).  DIA rows in offset
// order: NL lower bands (row NL - l holds offset -S l by column, after the LU
// the unit-L multipliers), the diagonal (row NL), NU upper bands (row NL + k
// holds offset S k by column).  Forward elimination subtracts the summed lower
// terms, back substitution subtracts the upper terms one by one, as la.pyx's
// *_inner_solve_ptr loops do; terms beyond either end of the line are absent.
template <typename T, int NL, int NU, int S>
__global__ void band_solve_kernel(T* __restrict__ u, LineMap g, const double* __restrict__ data,
                                  int n, int64_t dls, int64_t skip)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nl = g.nlines;
    if (gid >= S * nl) return;
    const int p = (int)(gid / nl);
    const int64_t L = gid - (int64_t)p * nl;
    if (L < skip || p >= n) return;
    T* v = u + g.off(L);
    const int64_t sa = g.sa;
    const double* rows = data + L * dls;
    const double* d = rows + (int64_t)NL * n;
    if constexpr (NL > 0) {
        T w[NL];  // w[l] = u[i - S (l + 1)]
#pragma unroll
        for (int l = 0; l < NL; ++l) w[l] = zero<T>();
        w[0] = v[p * sa];
        for (int i = p + S; i < n; i += S) {
            T s = mul(w[0], rows[(int64_t)(NL - 1) * n + i - S]);
#pragma unroll
            for (int l = 1; l < NL; ++l) {
                const int c = i - S * (l + 1);
                if (c >= 0) s = add(s, mul(w[l], rows[(int64_t)(NL - 1 - l) * n + c]));
            }
            const T cur = add(v[i * sa], mul(s, -1.0));
            v[i * sa] = cur;
#pragma unroll
            for (int l = NL - 1; l > 0; --l) w[l] = w[l - 1];
            w[0] = cur;
        }
    }
    const int il = (S == 2) ? last_of_parity(n, p) : n - 1;
    T nx[NU];  // nx[k] = u[i + S (k + 1)]
#pragma unroll
    for (int k = 0; k < NU; ++k) nx[k] = zero<T>();
    for (int i = il; i >= 0; i -= S) {
        T acc = v[i * sa];
#pragma unroll
        for (int k = 1; k <= NU; ++k) {
            const int c = i + S * k;
            if (c < n) acc = sub_mul(acc, rows[(int64_t)(NL + k) * n + c], nx[k - 1]);
        }
        const T cur = divd(acc, d[i]);
        v[i * sa] = cur;
#pragma unroll
        for (int k = NU - 1; k > 0; --k) nx[k] = nx[k - 1];
        nx[0] = cur;
    }
}

// Doolittle LU without pivoting of a general band matrix with offsets
// -NL..NU (unit stride), in place on its DIA rows (A(i, j) at row NL + j - i,
// column j): the multipliers replace the lower bands, U the diagonal and the
// upper bands, the layout band_solve_kernel<T, NL, NU, 1> reads.  One thread
// per system.  Stands in for the reference's general sparse fallback
// (la.py:823-844, SuperLU) on the banded systems the Galerkin spaces give;
// without pivoting it needs nonzero pivots (SPD or diagonally dominant
// matrices, as the mass and Helmholtz matrices are).
template <int NL, int NU>
__global__ void band_lu_kernel(double* __restrict__ data, int n, int64_t nbatch)
{
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbatch) return;
    double* r = data + b * (int64_t)(NL + 1 + NU) * n;
    for (int k = 0; k + 1 < n; ++k) {
        const double piv = r[(int64_t)NL * n + k];
#pragma unroll
        for (int l = 1; l <= NL; ++l) {
            if (k + l >= n) break;
            double* lik = r + (int64_t)(NL - l) * n + k;  // A(k + l, k)
            const double m = *lik / piv;
            *lik = m;
#pragma unroll
            for (int q = 1; q <= NU; ++q) {
                if (k + q >= n) break;
                // A(k + l, k + q) -= m A(k, k + q); offset q - l in [1 - NL, NU - 1]
                r[(int64_t)(NL + q - l) * n + k + q] -= m * r[(int64_t)(NL + q) * n + k + q];
            }
        }
    }
}

// la.pyx:254-263 TDMA_O_LU, one thread per system
__global__ void tdma_o_lu_kernel(double* __restrict__ data, int n, int64_t nbatch)
{
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbatch) return;
    double* ld = data + b * 3 * n;
    double* d = ld + n;
    double* ud = ld + 2 * n + 1;
    for (int i = 1; i < n; ++i) {
        ld[i - 1] = ld[i - 1] / d[i - 1];
        d[i] = d[i] - ld[i - 1] * ud[i - 1];
    }
}

// la.pyx:199-211 FDMA_LU, one thread per (system, parity)
__global__ void fdma_lu_kernel(double* __restrict__ data, int n, int64_t nbatch)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= 2 * nbatch) return;
    const int p = (int)(gid / nbatch);
    const int64_t b = gid - (int64_t)p * nbatch;
    double* ld = data + b * 4 * n;
    double* d = ld + n;
    double* u1 = ld + 2 * n + 2;
    double* u2 = ld + 3 * n + 4;
    for (int i = p + 2; i < n; i += 2) {
        ld[i - 2] = ld[i - 2] / d[i - 2];
        d[i] = d[i] - ld[i - 2] * u1[i - 2];
        if (i < n - 2) u1[i] = u1[i] - ld[i - 2] * u2[i - 2];
    }
}

// la.pyx:265-303 HeptaDMA_LU (band spacing 2), one thread per (system, parity)
__global__ void heptadma_lu_kernel(double* __restrict__ data, int n, int64_t nbatch)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= 2 * nbatch) return;
    const int p = (int)(gid / nbatch);
    const int64_t bb = gid - (int64_t)p * nbatch;
    double* a = data + bb * 7 * n;
    double* b = a + n;
    double* d = a + 2 * n;
    double* e = a + 3 * n + 2;
    double* f = a + 4 * n + 4;
    double* g = a + 5 * n + 6;
    double* h = a + 6 * n + 8;
    for (int i = p; i < n - 4; i += 2) {
        double lam = b[i] / d[i];
        d[i + 2] -= lam * e[i];
        e[i + 2] -= lam * f[i];
        if (i < n - 6) f[i + 2] -= lam * g[i];
        if (i < n - 8) g[i + 2] -= lam * h[i];
        b[i] = lam;
        lam = a[i] / d[i];
        b[i + 2] -= lam * e[i];
        d[i + 4] -= lam * f[i];
        if (i < n - 6) e[i + 4] -= lam * g[i];
        if (i < n - 8) f[i + 4] -= lam * h[i];
        a[i] = lam;
    }
    for (int i = n - 4; i <= n - 3; ++i) {
        if ((i & 1) != p) continue;
        const double lam = b[i] / d[i];
        d[i + 2] -= lam * e[i];
        b[i] = lam;
    }
}

// ----------------------------------------------------------------- Helmholtz
struct HelmDiags {
    const double *A0, *A2, *A4, *Bm2, *B0, *B2;
    int M;
    int neumann;
};

__global__ void helmholtz_lu_kernel(HelmDiags h, const double* __restrict__ alfa,
                                    const double* __restrict__ beta, int64_t abs_, LineMap g,
                                    double* __restrict__ d0, double* __restrict__ d1,
                                    double* __restrict__ d2, double* __restrict__ Lf)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nl = g.nlines;
    if (gid >= 2 * nl) return;
    const int p = (int)(gid / nl);
    const int64_t L = gid - (int64_t)p * nl;
    const int M = h.M;
    if (p >= M) return;
    const int64_t o = g.off(L), sa = g.sa;
    const double al = alfa[L * abs_], be = beta[L * abs_];
    const bool nm = h.neumann != 0;
    const bool zb = nm && fabs(be) < 1e-8;
    auto a0 = [&](int i) {
        double v = h.A0[i];
        if (nm) {
            if (i == 0) { if (zb) v = 1.0 / al; }
            else v /= (double)i * i;
        }
        return v;
    };
    auto b0 = [&](int i) {
        double v = h.B0[i];
        if (nm) {
            if (i == 0) { if (zb) v = 0.0; }
            else v /= (double)i * i;
        }
        return v;
    };
    auto a2 = [&](int i) {
        if (i >= M - 2) return 0.0;
        double v = h.A2[i];
        if (nm) v /= (double)(i + 2) * (i + 2);
        return v;
    };
    auto b2 = [&](int i) {
        if (i >= M - 2) return 0.0;
        double v = h.B2[i];
        if (nm) v /= (double)(i + 2) * (i + 2);
        return v;
    };
    auto a4 = [&](int i) {
        if (i >= M - 4) return 0.0;
        double v = h.A4[i];
        if (nm) v /= (double)(i + 4) * (i + 4);
        return v;
    };
    auto bm2 = [&](int i) {
        double v = h.Bm2[i];
        if (nm && i >= 1) v /= (double)i * i;
        return v;
    };
    double d0p = al * a0(p) + be * b0(p);
    double d1p = al * a2(p) + be * b2(p);
    double d2p = al * a4(p);
    d0[o + p * sa] = d0p;
    if (p < M - 2) d1[o + p * sa] = d1p;
    if (p < M - 4) d2[o + p * sa] = d2p;
    for (int i = p + 2; i < M; i += 2) {
        const double l = be * bm2(i - 2) / d0p;
        Lf[o + (i - 2) * sa] = l;
        const double d0v = al * a0(i) + be * b0(i) - l * d1p;
        double d1v = 0.0, d2v = 0.0;
        if (i < M - 2) d1v = al * a2(i) + be * b2(i) - l * d2p;
        if (i < M - 4) d2v = al * a4(i) - l * d2p;
        d0[o + i * sa] = d0v;
        if (i < M - 2) d1[o + i * sa] = d1v;
        if (i < M - 4) d2[o + i * sa] = d2v;
        d0p = d0v;
        d1p = d1v;
        d2p = d2v;
    }
}

template <typename T>
__global__ void helmholtz_matvec_kernel(const T* __restrict__ v, T* __restrict__ c, LineMap gv,
                                        LineMap gc, int M, int neumann,
                                        const double* __restrict__ A0, const double* __restrict__ At,
                                        const double* __restrict__ Bm2, const double* __restrict__ B0,
                                        const double* __restrict__ B2, const double* __restrict__ alfa,
                                        const double* __restrict__ beta, int64_t abs_)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nl = gv.nlines;
    if (gid >= 2 * nl) return;
    const int p = (int)(gid / nl);
    const int64_t L = gid - (int64_t)p * nl;
    const T* vl = v + gv.off(L);
    T* cl = c + gc.off(L);
    const int64_t sv = gv.sa, sc = gc.sa;
    const double al = alfa[L * abs_], be = beta[L * abs_];
    cl[(M + p) * sc] = zero<T>();  // BC slots N-2, N-1
    if (p >= M) return;
    const int il = last_of_parity(M, p);
    T S = zero<T>();  // sum_{j>=1} w_{k+2j} v_{k+2j}
    for (int k = il; k >= 0; k -= 2) {
        if (k + 2 < M) {
            const double w = neumann ? (double)(k + 2) * (k + 2) : 1.0;
            S = add(S, mul(vl[(k + 2) * sv], w));
        }
        T r = mul(vl[k * sv], al * A0[k] + be * B0[k]);
        if (k >= 2) r = add(r, mul(vl[(k - 2) * sv], be * Bm2[k - 2]));
        if (k + 2 < M) {
            r = add(r, mul(vl[(k + 2) * sv], be * B2[k]));
            r = add(r, mul(S, al * At[k]));
        }
        cl[k * sc] = r;
    }
}

template <typename T>
__global__ void poisson_add_kernel(const T* __restrict__ b, T* __restrict__ u, LineMap gb,
                                   LineMap gu, int M, const double* __restrict__ d,
                                   const double* __restrict__ d1, double scale)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nl = gu.nlines;
    if (gid >= 2 * nl) return;
    const int p = (int)(gid / nl);
    const int64_t L = gid - (int64_t)p * nl;
    if (p >= M) return;
    const T* bl = b + gb.off(L);
    T* ul = u + gu.off(L);
    const int64_t sb = gb.sa, su = gu.sa;
    const int il = last_of_parity(M, p);
    T n2 = divd(bl[il * sb], d[il]);
    ul[il * su] = n2;
    T S = zero<T>();
    for (int k = il - 2; k >= 0; k -= 2) {
        S = add(S, n2);
        T cur = divd(sub_mul(bl[k * sb], d1[k], S), d[k]);
        ul[k * su] = cur;
        n2 = cur;
    }
    if (!(fabs(scale - 1.0) < 1e-8))
        for (int k = p; k < M; k += 2) ul[k * su] = divd(ul[k * su], scale);
}

// ----------------------------------------------------------------- chain scans
// TDMA and Helmholtz solves with every chain cut into segments of E rows, one
// thread each.  A solve is two sweeps of a linear recurrence along the chain
//   y_m = f_m + a_m y_{m-1}                          (forward elimination)
//   x_m = f_m + q_m x_{m+1} [+ w_m s_{m+1}],  s_m = s_{m+1} + x_{m+1}
// (the running sum s is the constant tail of the Chebyshev stiffness rows), so
// a segment is an affine map of the state that enters it: each thread composes
// its own, a scan over the segments gives every thread its entering state, and
// it runs its rows once more.  Bound: a thread per chain waits for memory once
// per row with too few waves to hide it (8,320 lines of 63 rows at 128^3 are
// 260 waves on 1,024 SIMDs); here all of a thread's rows are loaded before the
// first of them is used and a chain is spread over 4 to 256 threads.
//
// A workgroup has TL lines x 256 / TL segments, a line's segments TL lanes
// apart, so that lanes run over lines (coalesced where the lines are
// neighbours in memory).  Chains longer than 256 / TL * E rows go in chunks,
// the state carried from one to the next and y kept in u.
//
// Measured against a thread per chain (and, for the Helmholtz solve of one long
// line, a workgroup whose first thread ran both sweeps from LDS): Helmholtz
// 128 x 128 x 65 complex 47.3 -> 18.0 us (its arrays are 68 MB: 14 us at copy
// speed), one line of 1024 reals 44.8 -> 5.5 us; TDMA 192 x 96 x 81 complex with
// shared factors 40.1 -> 11.1 us, 510 x 129 with factors per line 133 -> 7.4 us
// (and mode 0 in the same launch: 123 us in one of its own before).
//
// The maps' factors are kept as a number times a power of two: a product of
// multipliers may pass the largest double, or fall below the smallest, where the
// values themselves, row by row, stay in range (and a line of zeros stays zero).
// A segment's factor is split once, after its rows (at most 8 multipliers); the
// numbers of products over the at most 256 segments then stay far inside the
// range.  Against plain doubles a solve takes 0.3 us (TDMA) and 0.9 to 1.3 us
// (Helmholtz: 128 x 128 x 65 16.7 -> 18.0) more.
struct ChainFac {
    double a;
    int e;  // times 2^e
};
__device__ inline ChainFac chain_fac(double a, int e = 0)  // a in [1/2, 1) or 0
{
    return ChainFac{__builtin_amdgcn_frexp_mant(a), e + __builtin_amdgcn_frexp_exp(a)};
}
__device__ inline ChainFac chain_mul(ChainFac f, ChainFac g) { return ChainFac{f.a * g.a, f.e + g.e}; }
__device__ inline ChainFac chain_add(ChainFac f, ChainFac g)
{
    const int e = f.a == 0.0 ? g.e : g.a == 0.0 ? f.e : f.e > g.e ? f.e : g.e;
    return chain_fac(ldexp(f.a, f.e - e) + ldexp(g.a, g.e - e), e);
}

template <typename T>
struct ChainArgs {
    const T* b;
    T* u;
    LineMap gb, gu;
    int n;            // rows of the system
    int zero;         // rows after them set to zero (boundary slots)
    int64_t skip;     // lines below it are left alone
    // TDMA: DIA rows of la.pyx:243-252's LU, line L at data + L dls
    const double* data;
    int64_t dls;
    // Helmholtz: factor arrays of LU_Helmholtz (la.pyx:708-843)
    const double *d0, *d1, *d2, *Lf;
    LineMap gf;
    int neumann;
};

__device__ inline double shflu(double v, int d) { return __shfl_up(v, d); }
__device__ inline double2 shflu(double2 v, int d) { return make_double2(__shfl_up(v.x, d), __shfl_up(v.y, d)); }
__device__ inline double shfld(double v, int d) { return __shfl_down(v, d); }
__device__ inline double2 shfld(double2 v, int d) { return make_double2(__shfl_down(v.x, d), __shfl_down(v.y, d)); }
__device__ inline double ldx(double a, int e) { return ldexp(a, e); }
__device__ inline double2 ldx(double2 a, int e) { return make_double2(ldexp(a.x, e), ldexp(a.y, e)); }
__device__ inline double axpb(double a, double x, double b) { return a * x + b; }
__device__ inline double2 axpb(double a, double2 x, double2 b) { return make_double2(a * x.x + b.x, a * x.y + b.y); }
template <typename T>
__device__ inline T axpb(ChainFac f, T x, T b)
{
    return add(ldx(mul(x, f.a), f.e), b);
}

template <typename T, int TL, int E, bool HELM, bool ONE>
__global__ void __launch_bounds__(256) chain_solve_kernel(ChainArgs<T> g)
{
    constexpr int SG = 256 / TL, WS = 64 / TL, NW = 4;
    __shared__ ChainFac sA[NW][TL], sF[NW][TL];  // forward, backward (no barrier lies between them)
    __shared__ T sB[NW][TL];
    __shared__ double sM[NW][TL][HELM ? 3 : 1];
    __shared__ int sE[NW][TL];
    __shared__ T sC[NW][TL][2];
    const int tid = threadIdx.x, t = tid % TL, seg = tid / TL, wave = tid >> 6, ws = seg % WS;
    const int p = blockIdx.y, n = g.n;
    const int64_t L = wide_block() * TL + t;
    const bool valid = L < g.gu.nlines && L >= g.skip;
    const int64_t Lc = valid ? L : 0;
    const T* bl = g.b + g.gb.off(Lc);
    T* ul = g.u + g.gu.off(Lc);
    const int64_t sb = g.gb.sa, su = g.gu.sa;
    // lower multiplier of row i at lo[(i - 2) sf], pivot at dg[i sf], upper
    // bands at up[i sf] and (Helmholtz tail) tl[i sf]
    const double *lo, *dg, *up, *tl = nullptr;
    int64_t sf = 1;
    if constexpr (HELM) {
        const int64_t of = g.gf.off(Lc);
        lo = g.Lf + of;
        dg = g.d0 + of;
        up = g.d1 + of;
        tl = g.d2 + of;
        sf = g.gf.sa;
    } else {
        lo = g.data + Lc * g.dls;
        dg = lo + n;
        up = lo + 2 * (int64_t)n + 2;
    }
    const int K = (n - p + 1) / 2;  // rows i = p + 2 m, m < K
    const int nch = ONE ? 1 : (K + SG * E - 1) / (SG * E);

    if (valid && seg == 0)
        for (int i = n + p; i < n + g.zero; i += 2) ul[(int64_t)i * su] = zero<T>();

    T y[E];
    double iv[E], q[E], w[HELM ? E : 1];
    auto load_back = [&](int m0) {  // pivots and upper bands, clamped to row p where outside
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int m = m0 + e;
            const bool in = valid && m < K, in1 = valid && m + 1 < K;
            iv[e] = dg[in ? (int64_t)(p + 2 * m) * sf : 0];
            q[e] = in1 ? up[(int64_t)(p + 2 * m) * sf] : 0.0;
            if constexpr (HELM) w[e] = valid && m + 2 < K ? tl[(int64_t)(p + 2 * m) * sf] : 0.0;
        }
    };
    // ---------------------------------------------------------- forward
    T carry = zero<T>();
    for (int c = 0; c < nch; ++c) {
        const int m0 = (c * SG + seg) * E;
        double am[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int m = m0 + e;
            const bool in = valid && m < K;
            y[e] = in ? bl[(int64_t)(p + 2 * m) * sb] : zero<T>();
            am[e] = in && m > 0 ? -lo[(int64_t)(p + 2 * m - 2) * sf] : 0.0;
        }
        if (ONE) load_back(m0);
        double A0 = 1.0;
        T B = zero<T>();
#pragma unroll
        for (int e = 0; e < E; ++e) {
            B = axpb(am[e], B, y[e]);
            A0 *= am[e];
        }
        ChainFac A = chain_fac(A0);
#pragma unroll
        for (int k = 1; k < WS; k <<= 1) {
            const ChainFac oA{shflu(A.a, TL * k), __shfl_up(A.e, TL * k)};
            const T oB = shflu(B, TL * k);
            if (ws >= k) {
                B = axpb(A, oB, B);
                A = chain_mul(A, oA);
            }
        }
        ChainFac eA{shflu(A.a, TL), __shfl_up(A.e, TL)};
        T eB = shflu(B, TL);
        if (ws == 0) {
            eA = ChainFac{1.0, 0};
            eB = zero<T>();
        }
        if (ws == WS - 1) {
            sA[wave][t] = A;
            sB[wave][t] = B;
        }
        __syncthreads();
        T in = carry;
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            carry = axpb(sA[k][t], carry, sB[k][t]);
            if (k < wave) in = carry;
        }
        T yv = axpb(eA, in, eB);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            yv = axpb(am[e], yv, y[e]);
            y[e] = yv;
        }
        if (!ONE) {
#pragma unroll
            for (int e = 0; e < E; ++e)
                if (valid && m0 + e < K) ul[(int64_t)(p + 2 * (m0 + e)) * su] = y[e];
            __syncthreads();  // sA, sB are written again by the next chunk
        }
    }
    // ---------------------------------------------------------- backward
    T cx = zero<T>(), cs = zero<T>();  // state after the last row
    for (int c = nch - 1; c >= 0; --c) {
        const int m0 = (c * SG + seg) * E;
        if (!ONE) {
            load_back(m0);
#pragma unroll
            for (int e = 0; e < E; ++e)
                y[e] = valid && m0 + e < K ? ul[(int64_t)(p + 2 * (m0 + e)) * su] : zero<T>();
        }
        const double d00 = iv[0];
        T Bx = zero<T>(), Bs = zero<T>();
        // the segment's map: x from x by F, the other three of the 2 x 2 matrix
        // (Helmholtz) times 2^Me.  F keeps its own exponent: beside M10 >= 1
        // (the sum takes x as it is) it may be below the smallest double.
        double M00 = 1.0, M01 = 0.0, M10 = 0.0, M11 = 1.0;
        int Me = 0;
        auto scaled = [&]() {  // the largest of the three in [1/2, 1)
            const int ex = __builtin_amdgcn_frexp_exp(fmax(fabs(M01), fmax(fabs(M10), fabs(M11))));
            M01 = ldexp(M01, -ex);
            M10 = ldexp(M10, -ex);
            M11 = ldexp(M11, -ex);
            Me += ex;
        };
#pragma unroll
        for (int e = E - 1; e >= 0; --e) {
            const bool in = valid && m0 + e < K;
            const double r = 1.0 / iv[e];
            y[e] = in ? mul(y[e], r) : zero<T>();
            q[e] = in ? -q[e] * r : 0.0;
            if constexpr (HELM) {
                w[e] = in ? -w[e] * r : 0.0;
                const T nx = add(axpb(q[e], Bx, y[e]), mul(Bs, w[e]));
                Bs = add(Bs, Bx);
                Bx = nx;
                const double n00 = q[e] * M00 + w[e] * M10, n01 = q[e] * M01 + w[e] * M11;
                M10 += M00;
                M11 += M01;
                M00 = n00;
                M01 = n01;
            } else {
                Bx = axpb(q[e], Bx, y[e]);
                M00 *= q[e];
            }
        }
        ChainFac F = chain_fac(M00);
        if constexpr (HELM) scaled();
#pragma unroll
        for (int k = 1; k < WS; k <<= 1) {
            const ChainFac oF{shfld(F.a, TL * k), __shfl_down(F.e, TL * k)};
            const T ox = shfld(Bx, TL * k);
            if constexpr (HELM) {
                const double o01 = shfld(M01, TL * k), o10 = shfld(M10, TL * k), o11 = shfld(M11, TL * k);
                const int oe = __shfl_down(Me, TL * k);
                const T os = shfld(Bs, TL * k);
                if (ws + k < WS) {
                    Bx = add(axpb(F, ox, Bx), ldx(mul(os, M01), Me));
                    Bs = add(ldx(axpb(M10, ox, mul(os, M11)), Me), Bs);
                    const double o00 = ldexp(oF.a, oF.e - oe), f00 = ldexp(F.a, F.e - Me);
                    const double n01 = f00 * o01 + M01 * o11;
                    const double n10 = M10 * o00 + M11 * o10, n11 = M10 * o01 + M11 * o11;
                    F = chain_add(chain_mul(F, oF), chain_mul(ChainFac{M01, Me}, ChainFac{o10, oe}));
                    M01 = n01;
                    M10 = n10;
                    M11 = n11;
                    Me += oe;
                    scaled();
                }
            } else if (ws + k < WS) {
                Bx = axpb(F, ox, Bx);
                F = chain_mul(F, oF);
            }
        }
        // the maps of the segments after this one in the wave
        ChainFac eF{shfld(F.a, TL), __shfl_down(F.e, TL)};
        double e01 = 0.0, e10 = 0.0, e11 = 1.0;
        int ee = 0;
        T ex = shfld(Bx, TL), es = zero<T>();
        if constexpr (HELM) {
            e01 = shfld(M01, TL);
            e10 = shfld(M10, TL);
            e11 = shfld(M11, TL);
            ee = __shfl_down(Me, TL);
            es = shfld(Bs, TL);
        }
        if (ws == WS - 1) {
            eF = ChainFac{1.0, 0};
            e11 = 1.0;
            e01 = e10 = 0.0;
            ee = 0;
            ex = es = zero<T>();
        }
        if (ws == 0) {
            sF[wave][t] = F;
            sC[wave][t][0] = Bx;
            if constexpr (HELM) {
                sE[wave][t] = Me;
                sM[wave][t][0] = M01;
                sM[wave][t][1] = M10;
                sM[wave][t][2] = M11;
                sC[wave][t][1] = Bs;
            }
        }
        __syncthreads();
        T ix = cx, is = cs;
#pragma unroll
        for (int k = NW - 1; k >= 0; --k) {
            if constexpr (HELM) {
                const T nx = add(axpb(sF[k][t], cx, sC[k][t][0]), ldx(mul(cs, sM[k][t][0]), sE[k][t]));
                cs = add(ldx(axpb(sM[k][t][1], cx, mul(cs, sM[k][t][2])), sE[k][t]), sC[k][t][1]);
                cx = nx;
            } else {
                cx = axpb(sF[k][t], cx, sC[k][t][0]);
            }
            if (k > wave) {
                ix = cx;
                is = cs;
            }
        }
        T x = axpb(eF, ix, ex), s = zero<T>();
        if constexpr (HELM) {
            x = add(x, ldx(mul(is, e01), ee));
            s = add(ldx(axpb(e10, ix, mul(is, e11)), ee), es);
        }
#pragma unroll
        for (int e = E - 1; e >= 0; --e) {
            const int m = m0 + e, i = p + 2 * m;
            if constexpr (HELM) {
                const T nx = add(axpb(q[e], x, y[e]), mul(s, w[e]));
                s = add(s, x);
                x = nx;
            } else {
                x = axpb(q[e], x, y[e]);
            }
            if (valid && m < K) {
                T out = x;
                if constexpr (HELM) {
                    if (g.neumann) {  // column scaling and k = 0 gauge (la.pyx:907-912)
                        if (i > 0) out = divd(out, (double)i * i);
                        else if ((d00 - 1.0) * (d00 - 1.0) < 1e-16) out = zero<T>();
                    }
                }
                ul[(int64_t)i * su] = out;
            }
        }
        if (!ONE) __syncthreads();
    }
}

template <int TL, int E, bool ONE, bool HELM, typename T>
static void chain_run(const ChainArgs<T>& a, hipStream_t s)
{
    hipLaunchKernelGGL((chain_solve_kernel<T, TL, E, HELM, ONE>), wide_grid((a.gu.nlines + TL - 1) / TL, 2),
                       dim3(256), 0, s, a);
}

// The fewest rows per thread that hold the chain in one chunk, of those that
// chain_tl's choice of TL can meet.
template <int TL, bool HELM, typename T>
static void chain_launch_tl(const ChainArgs<T>& a, hipStream_t s)
{
    constexpr int SG = 256 / TL;
    const int K = (a.n + 1) / 2;
    if constexpr (TL == 1 || TL == 16)
        if (K <= SG) return chain_run<TL, 1, true, HELM>(a, s);
    if (K <= 2 * SG) return chain_run<TL, 2, true, HELM>(a, s);
    if (K <= 4 * SG) return chain_run<TL, 4, true, HELM>(a, s);
    if constexpr (TL == 8 || TL == 16)
        if (K <= 6 * SG) return chain_run<TL, 6, true, HELM>(a, s);
    if (K <= 8 * SG) return chain_run<TL, 8, true, HELM>(a, s);
    chain_run<TL, 8, false, HELM>(a, s);
}

// Lines per workgroup for chains of K rows.  At least as many as leave a thread
// one or two of its 256 / TL share of the rows (a chain of 7 rows over 256 threads
// takes as long as one of 511), at most as many as hold the chain in one chunk of
// 8 rows a thread, and between the two by the number of lines, so that at least
// 128 workgroups of each parity are in flight.
//   Lines side by side in memory (complex, TDMA / Helmholtz, microseconds; TL by
//   this rule | 16, 4 or 1 by the number of lines alone | a thread per chain):
//   14 rows x 131072 lines 13.6/24.1 | 42.9/70.2 | 10.5/24.2, 62 x 32768 12.0/25.4 |
//   17.4/28.4 | 17.8/32.3, 254 x 8192 15.3/24.7 in both | 53/94, 510 x 32768 98/288 |
//   145/289 | 177/370.  From 65536 lines on chains beyond one chunk of 16 lines go
//   64 lines wide (1022 x 131072: 1542/2458, 16 wide 1656/2735, thread per chain
//   1569/2488); reals, half as wide in bytes, take 16 lines where 8 hold a chunk
//   (510 x 8192 47, 8 lines 59).
//   Lines along memory: a thread's two rows share its cache line with its
//   neighbours', so the smallest count is the best one (62 x 32768 22.5/48.3, 1
//   line per workgroup 300/518, a thread per chain 33/73; 254 x 32768 103/247,
//   306/520, 146/403; 510 x 131072 938/2193, 1228/2232, 2731/7762); up to 128 of
//   them are spread over the chip instead (254 x 16: 4.2/5.9 against 4.8/6.3).
//   TDMA factors of each line's own lie along memory whatever the lines do, so
//   those stay at 16 lines where 64 would do (64 x 32768 side by side 27, 64 lines
//   36) and take a line along memory alone from 193 rows of a chain on (512 x 32768
//   373, 4 lines 559; up to there 256 x 32768 182, alone 302).
static int chain_tl(int K, int64_t nlines, bool across, bool cplx, bool own)
{
    const int least = K <= 8 ? 64 : K <= 32 ? 16 : K <= 64 ? 8 : K <= (own ? 192 : 256) ? 4 : 1;
    if (!across) return K > 32 && nlines <= 128 ? 1 : least;
    if (K > 128 && nlines >= 65536) return 64;
    if (K > 256) return nlines < 128 ? 1 : nlines < 2048 ? 4 : 16;
    const int most = K <= 32 && !own ? 64 : K <= 128 || !cplx ? 16 : 8;
    const int fill = nlines >= 8192 ? 64 : nlines >= 2048 ? 16 : nlines >= 1024 ? 8 : 4;
    const int tl = fill < most ? fill : most;
    return tl > least ? tl : least;
}

template <typename T, bool HELM>
static void chain_launch(const ChainArgs<T>& a, hipStream_t s)
{
    auto absl = [](int64_t v) { return v < 0 ? -v : v; };
    const bool across = absl(a.gu.s2) < absl(a.gu.sa) && a.gu.d2 > 1;
    switch (chain_tl((a.n + 1) / 2, a.gu.nlines, across, sizeof(T) == 16, !HELM && a.dls > 0)) {
        case 64: return chain_launch_tl<64, HELM>(a, s);
        case 16: return chain_launch_tl<16, HELM>(a, s);
        case 8: return chain_launch_tl<8, HELM>(a, s);
        case 4: return chain_launch_tl<4, HELM>(a, s);
        default: return chain_launch_tl<1, HELM>(a, s);
    }
}

// ----------------------------------------------------------------- host
static int line_map(int ndim, const int64_t* shape, const int64_t* strides, int axis, LineMap* m,
                    int64_t* n)
{
    Geom g;
    int rc = make_geom(ndim, shape, strides, axis, &g);
    if (rc) return rc;
    m->sa = g.sa;
    m->s1 = g.s1;
    m->s2 = g.s2;
    m->d2 = g.d2;
    m->nlines = g.d1 * g.d2;
    if (n) *n = g.n;
    return SFA_OK;
}

static inline dim3 grid_for(int64_t nthreads, int bs)
{
    return dim3((unsigned)((nthreads + bs - 1) / bs));
}

}  // namespace sfa

using namespace sfa;

template <typename T>
static ChainArgs<T> tdma_args(T* u, const LineMap& g, const double* data, int64_t n, int64_t dls,
                              int64_t skip, int nzero)
{
    ChainArgs<T> a{};
    a.zero = nzero;
    a.b = u;
    a.u = u;
    a.gb = a.gu = g;
    a.n = (int)n;
    a.skip = skip;
    a.data = data;
    a.dls = dls;
    return a;
}

template <int KIND>
static int banded_solve(void* u, int dtype, int ndim, const int64_t* shape, const int64_t* strides,
                        int axis, const double* data, int64_t n, int64_t dls, int64_t skip,
                        void* stream, int64_t nzero = 0)
{
    LineMap g;
    int64_t len;
    int rc = line_map(ndim, shape, strides, axis, &g, &len);
    if (rc) return rc;
    SFA_CHECK(dtype == SFA_F64 || dtype == SFA_C128, SFA_ERR_ARG, "bad dtype %d", dtype);
    SFA_CHECK(n >= 1 && n <= len, SFA_ERR_ARG, "system size %lld must be in [1, %lld]",
              (long long)n, (long long)len);
    SFA_CHECK(KIND == 0 || n >= (KIND == 1 ? 2 : 4), SFA_ERR_ARG, "system too small (n=%lld)",
              (long long)n);
    SFA_CHECK(dls >= 0 && skip >= 0, SFA_ERR_ARG, "negative stride/skip");
    SFA_CHECK(nzero >= 0 && n + nzero <= len, SFA_ERR_ARG, "%lld rows and %lld zeroed ones on a line of %lld",
              (long long)n, (long long)nzero, (long long)len);
    const int bs = 256;
    auto absl = [](int64_t v) { return v < 0 ? -v : v; };
    const int along = absl(g.sa) <= absl(g.s2) ? 1 : 0;
    dim3 grid = wide_grid((g.nlines * n + bs - 1) / bs, 1);  // DiagMA
    if (KIND == 2) {
        SFA_CHECK(2 * g.nlines < (1ll << 32), SFA_ERR_UNSUPPORTED, "too many lines");
        grid = grid_for(2 * g.nlines, bs);
    }
    hipStream_t s = (hipStream_t)stream;
    if (dtype == SFA_C128) {
        double2* uu = (double2*)u;
        if (KIND == 0) hipLaunchKernelGGL(diag_solve_kernel<double2>, grid, dim3(bs), 0, s, uu, g, data, (int)n, dls, skip, along);
        if (KIND == 1) chain_launch<double2, false>(tdma_args(uu, g, data, n, dls, skip, (int)nzero), s);
        if (KIND == 2) hipLaunchKernelGGL(pdma_solve_kernel<double2>, grid, dim3(bs), 0, s, uu, g, data, (int)n, dls, skip);
    } else {
        double* uu = (double*)u;
        if (KIND == 0) hipLaunchKernelGGL(diag_solve_kernel<double>, grid, dim3(bs), 0, s, uu, g, data, (int)n, dls, skip, along);
        if (KIND == 1) chain_launch<double, false>(tdma_args(uu, g, data, n, dls, skip, (int)nzero), s);
        if (KIND == 2) hipLaunchKernelGGL(pdma_solve_kernel<double>, grid, dim3(bs), 0, s, uu, g, data, (int)n, dls, skip);
    }
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

extern "C" int sfa_tdma_solve(void* u, int dtype, int ndim, const int64_t* shape,
                              const int64_t* strides, int axis, const double* data, int64_t n,
                              int64_t data_line_stride, int64_t skip_lines, void* stream)
{
    return banded_solve<1>(u, dtype, ndim, shape, strides, axis, data, n, data_line_stride,
                           skip_lines, stream);
}

extern "C" int sfa_tdma_mass_solve(void* u, int dtype, int ndim, const int64_t* shape, const int64_t* strides,
                                   int axis, const double* data, int64_t n, int64_t nzero, void* stream)
{
    return banded_solve<1>(u, dtype, ndim, shape, strides, axis, data, n, 0, 0, stream, nzero);
}

extern "C" int sfa_pdma_solve(void* u, int dtype, int ndim, const int64_t* shape,
                              const int64_t* strides, int axis, const double* data, int64_t n,
                              int64_t data_line_stride, int64_t skip_lines, void* stream)
{
    return banded_solve<2>(u, dtype, ndim, shape, strides, axis, data, n, data_line_stride,
                           skip_lines, stream);
}

extern "C" int sfa_diagma_solve(void* u, int dtype, int ndim, const int64_t* shape,
                                const int64_t* strides, int axis, const double* d, int64_t n,
                                int64_t data_line_stride, int64_t skip_lines, void* stream)
{
    return banded_solve<0>(u, dtype, ndim, shape, strides, axis, d, n, data_line_stride,
                           skip_lines, stream);
}

extern "C" int sfa_tdma_lu(double* data, int64_t n, int64_t nbatch, void* stream)
{
    SFA_CHECK(n >= 2 && nbatch >= 1, SFA_ERR_ARG, "bad TDMA size n=%lld nbatch=%lld", (long long)n,
              (long long)nbatch);
    hipLaunchKernelGGL(tdma_lu_kernel, grid_for(2 * nbatch, 256), dim3(256), 0, (hipStream_t)stream,
                       data, (int)n, nbatch);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

template <int NL, int NU, int S>
static int band_solve(const char* name, int64_t nmin, void* u, int dtype, int ndim,
                      const int64_t* shape, const int64_t* strides, int axis, const double* data,
                      int64_t n, int64_t dls, int64_t skip, void* stream)
{
    LineMap g;
    int64_t len;
    int rc = line_map(ndim, shape, strides, axis, &g, &len);
    if (rc) return rc;
    SFA_CHECK(dtype == SFA_F64 || dtype == SFA_C128, SFA_ERR_ARG, "%s: bad dtype %d", name, dtype);
    SFA_CHECK(n >= nmin && n <= len, SFA_ERR_ARG, "%s: system size %lld must be in [%lld, %lld]",
              name, (long long)n, (long long)nmin, (long long)len);
    SFA_CHECK(n <= (1 << 26), SFA_ERR_ARG, "%s: system size %lld too large", name, (long long)n);
    SFA_CHECK(data != nullptr && dls >= 0 && skip >= 0, SFA_ERR_ARG,
              "%s: null factors or negative stride/skip", name);
    if (g.nlines == 0) return SFA_OK;
    const int bs = 256;
    const dim3 grid = grid_for(S * g.nlines, bs);
    hipStream_t s = (hipStream_t)stream;
    if (dtype == SFA_C128)
        hipLaunchKernelGGL((band_solve_kernel<double2, NL, NU, S>), grid, dim3(bs), 0, s,
                           (double2*)u, g, data, (int)n, dls, skip);
    else
        hipLaunchKernelGGL((band_solve_kernel<double, NL, NU, S>), grid, dim3(bs), 0, s,
                           (double*)u, g, data, (int)n, dls, skip);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

#define SFA_BAND_SOLVE(fn, NL, NU, S, NMIN)                                                      \
    extern "C" int fn(void* u, int dtype, int ndim, const int64_t* shape,                        \
                      const int64_t* strides, int axis, const double* data, int64_t n,           \
                      int64_t data_line_stride, int64_t skip_lines, void* stream)                \
    {                                                                                            \
        return band_solve<NL, NU, S>(#fn, NMIN, u, dtype, ndim, shape, strides, axis, data, n,   \
                                     data_line_stride, skip_lines, stream);                      \
    }
SFA_BAND_SOLVE(sfa_tdma_o_solve, 1, 1, 1, 1)
SFA_BAND_SOLVE(sfa_twodma_solve, 0, 1, 2, 2)
SFA_BAND_SOLVE(sfa_threedma_solve, 0, 2, 2, 4)
SFA_BAND_SOLVE(sfa_fdma_solve, 1, 2, 2, 4)
SFA_BAND_SOLVE(sfa_heptadma_solve, 2, 4, 2, 8)
#undef SFA_BAND_SOLVE

static int band_lu(const char* name, void (*kern)(double*, int, int64_t), int chains, int64_t nmin,
                   double* data, int64_t n, int64_t nbatch, void* stream)
{
    SFA_CHECK(data != nullptr && n >= nmin && n <= (1 << 26) && nbatch >= 1, SFA_ERR_ARG,
              "bad %s size n=%lld nbatch=%lld (n >= %lld)", name, (long long)n,
              (long long)nbatch, (long long)nmin);
    hipLaunchKernelGGL(kern, grid_for(chains * nbatch, 256), dim3(256), 0, (hipStream_t)stream,
                       data, (int)n, nbatch);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

// general banded systems, offsets -nl..nu (0 <= nl <= 4, 1 <= nu <= 4), unit stride
using BandSolveFn = int (*)(const char*, int64_t, void*, int, int, const int64_t*,
                            const int64_t*, int, const double*, int64_t, int64_t, int64_t, void*);
#define SFA_ROW(NL) {band_solve<NL, 1, 1>, band_solve<NL, 2, 1>, band_solve<NL, 3, 1>,           \
                     band_solve<NL, 4, 1>}
static const BandSolveFn kBandSolve[5][4] = {SFA_ROW(0), SFA_ROW(1), SFA_ROW(2), SFA_ROW(3),
                                             SFA_ROW(4)};
#undef SFA_ROW
#define SFA_ROW(NL) {band_lu_kernel<NL, 1>, band_lu_kernel<NL, 2>, band_lu_kernel<NL, 3>,        \
                     band_lu_kernel<NL, 4>}
static void (*const kBandLU[5][4])(double*, int, int64_t) = {SFA_ROW(0), SFA_ROW(1), SFA_ROW(2),
                                                               SFA_ROW(3), SFA_ROW(4)};
#undef SFA_ROW

extern "C" int sfa_band_lu(double* data, int64_t n, int nl, int nu, int64_t nbatch, void* stream)
{
    SFA_CHECK(nl >= 0 && nl <= 4 && nu >= 1 && nu <= 4, SFA_ERR_ARG,
              "band_lu: bands -%d..%d outside -4..4 (nu >= 1)", nl, nu);
    return band_lu("band", kBandLU[nl][nu - 1], 1, 1, data, n, nbatch, stream);
}

extern "C" int sfa_band_solve(void* u, int dtype, int ndim, const int64_t* shape,
                              const int64_t* strides, int axis, const double* data, int64_t n,
                              int64_t data_line_stride, int64_t skip_lines, int nl, int nu,
                              void* stream)
{
    SFA_CHECK(nl >= 0 && nl <= 4 && nu >= 1 && nu <= 4, SFA_ERR_ARG,
              "band_solve: bands -%d..%d outside -4..4 (nu >= 1)", nl, nu);
    return kBandSolve[nl][nu - 1]("sfa_band_solve", 1, u, dtype, ndim, shape, strides, axis, data,
                                  n, data_line_stride, skip_lines, stream);
}

extern "C" int sfa_tdma_o_lu(double* data, int64_t n, int64_t nbatch, void* stream)
{
    return band_lu("TDMA_O", tdma_o_lu_kernel, 1, 1, data, n, nbatch, stream);
}

extern "C" int sfa_fdma_lu(double* data, int64_t n, int64_t nbatch, void* stream)
{
    return band_lu("FDMA", fdma_lu_kernel, 2, 4, data, n, nbatch, stream);
}

extern "C" int sfa_heptadma_lu(double* data, int64_t n, int64_t nbatch, void* stream)
{
    return band_lu("HeptaDMA", heptadma_lu_kernel, 2, 8, data, n, nbatch, stream);
}

extern "C" int sfa_pdma_lu(double* data, int64_t n, int64_t nbatch, void* stream)
{
    SFA_CHECK(n >= 5 && nbatch >= 1, SFA_ERR_ARG, "bad PDMA size n=%lld nbatch=%lld", (long long)n,
              (long long)nbatch);
    hipLaunchKernelGGL(pdma_lu_kernel, grid_for(2 * nbatch, 256), dim3(256), 0, (hipStream_t)stream,
                       data, (int)n, nbatch);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

extern "C" int sfa_helmholtz_lu(int neumann, int64_t N, const double* A0, const double* A2,
                                const double* A4, const double* Bm2, const double* B0,
                                const double* B2, const double* alfa, const double* beta,
                                int64_t ab_stride, double* d0, double* d1, double* d2, double* L,
                                int ndim, const int64_t* shape, const int64_t* f_strides, int axis,
                                void* stream)
{
    LineMap g;
    int64_t len;
    int rc = line_map(ndim, shape, f_strides, axis, &g, &len);
    if (rc) return rc;
    SFA_CHECK(len == N, SFA_ERR_ARG, "factor axis length %lld != N %lld", (long long)len, (long long)N);
    SFA_CHECK(N >= 8, SFA_ERR_ARG, "Helmholtz solver needs N >= 8 (got %lld)", (long long)N);
    SFA_CHECK(ab_stride == 0 || ab_stride == 1, SFA_ERR_ARG, "ab_stride must be 0 or 1");
    HelmDiags h{A0, A2, A4, Bm2, B0, B2, (int)(N - 2), neumann};
    hipLaunchKernelGGL(helmholtz_lu_kernel, grid_for(2 * g.nlines, 256), dim3(256), 0,
                       (hipStream_t)stream, h, alfa, beta, ab_stride, g, d0, d1, d2, L);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

template <typename T>
static void helm_launch(const void* b, void* u, const LineMap& gb, const LineMap& gu, const LineMap& gf,
                        int M, int neumann, const double* d0, const double* d1, const double* d2,
                        const double* L, hipStream_t s)
{
    ChainArgs<T> a{};
    a.b = (const T*)b;
    a.u = (T*)u;
    a.gb = gb;
    a.gu = gu;
    a.gf = gf;
    a.n = M;
    a.neumann = neumann;
    a.d0 = d0;
    a.d1 = d1;
    a.d2 = d2;
    a.Lf = L;
    chain_launch<T, true>(a, s);
}

extern "C" int sfa_helmholtz_solve(const void* b, void* u, int dtype, int ndim, const int64_t* shape,
                                   const int64_t* b_strides, const int64_t* u_strides, int axis,
                                   int neumann, const double* d0, const double* d1,
                                   const double* d2, const double* L, const int64_t* f_strides,
                                   void* stream)
{
    LineMap gb, gu, gf;
    int64_t N;
    int rc;
    if ((rc = line_map(ndim, shape, b_strides, axis, &gb, &N))) return rc;
    if ((rc = line_map(ndim, shape, u_strides, axis, &gu, nullptr))) return rc;
    if ((rc = line_map(ndim, shape, f_strides, axis, &gf, nullptr))) return rc;
    SFA_CHECK(dtype == SFA_F64 || dtype == SFA_C128, SFA_ERR_ARG, "bad dtype %d", dtype);
    SFA_CHECK(N >= 8, SFA_ERR_ARG, "Helmholtz solver needs N >= 8 (got %lld)", (long long)N);
    const int M = (int)N - 2;
    if (dtype == SFA_C128)
        helm_launch<double2>(b, u, gb, gu, gf, M, neumann, d0, d1, d2, L, (hipStream_t)stream);
    else
        helm_launch<double>(b, u, gb, gu, gf, M, neumann, d0, d1, d2, L, (hipStream_t)stream);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

extern "C" int sfa_helmholtz_matvec(const void* v, void* c, int dtype, int ndim,
                                    const int64_t* shape, const int64_t* v_strides,
                                    const int64_t* c_strides, int axis, int neumann,
                                    const double* A0, const double* At, const double* Bm2,
                                    const double* B0, const double* B2, const double* alfa,
                                    const double* beta, int64_t ab_stride, void* stream)
{
    LineMap gv, gc;
    int64_t N;
    int rc;
    if ((rc = line_map(ndim, shape, v_strides, axis, &gv, &N))) return rc;
    if ((rc = line_map(ndim, shape, c_strides, axis, &gc, nullptr))) return rc;
    SFA_CHECK(dtype == SFA_F64 || dtype == SFA_C128, SFA_ERR_ARG, "bad dtype %d", dtype);
    SFA_CHECK(N >= 4, SFA_ERR_ARG, "matvec needs N >= 4");
    SFA_CHECK(v != c, SFA_ERR_ARG, "matvec cannot run in place");
    SFA_CHECK(ab_stride == 0 || ab_stride == 1, SFA_ERR_ARG, "ab_stride must be 0 or 1");
    const int M = (int)N - 2;
    dim3 grid = grid_for(2 * gv.nlines, 256);
    if (dtype == SFA_C128)
        hipLaunchKernelGGL(helmholtz_matvec_kernel<double2>, grid, dim3(256), 0, (hipStream_t)stream,
                           (const double2*)v, (double2*)c, gv, gc, M, neumann, A0, At, Bm2, B0, B2,
                           alfa, beta, ab_stride);
    else
        hipLaunchKernelGGL(helmholtz_matvec_kernel<double>, grid, dim3(256), 0, (hipStream_t)stream,
                           (const double*)v, (double*)c, gv, gc, M, neumann, A0, At, Bm2, B0, B2,
                           alfa, beta, ab_stride);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

extern "C" int sfa_poisson_add_solve(const void* b, void* u, int dtype, int ndim,
                                     const int64_t* shape, const int64_t* b_strides,
                                     const int64_t* u_strides, int axis, const double* A0,
                                     const double* A2, double scale, void* stream)
{
    LineMap gb, gu;
    int64_t N;
    int rc;
    if ((rc = line_map(ndim, shape, b_strides, axis, &gb, &N))) return rc;
    if ((rc = line_map(ndim, shape, u_strides, axis, &gu, nullptr))) return rc;
    SFA_CHECK(dtype == SFA_F64 || dtype == SFA_C128, SFA_ERR_ARG, "bad dtype %d", dtype);
    SFA_CHECK(N >= 4, SFA_ERR_ARG, "Poisson solver needs N >= 4");
    const int M = (int)N - 2;
    dim3 grid = grid_for(2 * gu.nlines, 256);
    if (dtype == SFA_C128)
        hipLaunchKernelGGL(poisson_add_kernel<double2>, grid, dim3(256), 0, (hipStream_t)stream,
                           (const double2*)b, (double2*)u, gb, gu, M, A0, A2, scale);
    else
        hipLaunchKernelGGL(poisson_add_kernel<double>, grid, dim3(256), 0, (hipStream_t)stream,
                           (const double*)b, (double*)u, gb, gu, M, A0, A2, scale);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

// ----------------------------------------------------------------- banded matvec
// c(.., i, ..) (+)= s(line) sum_r D[r][i] v(.., i + off_r, ..) for i < nrows,
// 0 <= i + off_r < ncols (SparseMatrix.matvec, matrixbase.py:87-144, with the
// per-mode scale of TPMatrix.matvec :1437-1449).  D holds the diagonals by row
// (D[r][i] = A[i][i + off_r]); without accumulate, rows >= nrows of c are zeroed.
namespace sfa {
template <typename T>
__global__ void band_matvec_kernel(const T* __restrict__ v, T* __restrict__ c, LineMap gv,
                                   LineMap gc, int nout, int nrows, int ncols, int noffs,
                                   const int64_t* __restrict__ offs, const double* __restrict__ D,
                                   const double* __restrict__ scales, int accumulate)
{
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= gc.nlines * nout) return;
    const int i = (int)(gid % nout);
    const int64_t L = gid / nout;
    const T* vl = v + gv.off(L);
    T* cl = c + gc.off(L) + (int64_t)i * gc.sa;
    T acc = zero<T>();
    if (i < nrows) {
        for (int r = 0; r < noffs; ++r) {
            const int64_t j = i + offs[r];
            if (j >= 0 && j < ncols) acc = add(acc, mul(vl[(int64_t)j * gv.sa], D[(int64_t)r * nrows + i]));
        }
        if (scales) acc = mul(acc, scales[L]);
    } else if (accumulate) {
        return;
    }
    *cl = accumulate ? add(*cl, acc) : acc;
}
}  // namespace sfa

extern "C" int sfa_band_matvec(const void* v, void* c, int dtype, int ndim, const int64_t* v_shape,
                               const int64_t* v_strides, const int64_t* c_shape,
                               const int64_t* c_strides, int axis, int64_t nrows, int64_t ncols,
                               int noffs, const int64_t* offsets, const double* D,
                               const double* scales, int accumulate, void* stream)
{
    LineMap gv, gc;
    int64_t nv, nc;
    int rc = line_map(ndim, v_shape, v_strides, axis, &gv, &nv);
    if (rc) return rc;
    rc = line_map(ndim, c_shape, c_strides, axis, &gc, &nc);
    if (rc) return rc;
    SFA_CHECK(v != nullptr && c != nullptr && D != nullptr && offsets != nullptr && v != c,
              SFA_ERR_ARG, "band_matvec: null or aliased arrays");
    SFA_CHECK(dtype == SFA_F64 || dtype == SFA_C128, SFA_ERR_ARG, "band_matvec: bad dtype %d", dtype);
    for (int d = 0; d < ndim; ++d)
        SFA_CHECK(d == axis || v_shape[d] == c_shape[d], SFA_ERR_ARG,
                  "band_matvec: shapes differ off the axis (dim %d)", d);
    SFA_CHECK(noffs >= 1, SFA_ERR_ARG, "band_matvec: no diagonals");
    SFA_CHECK(nrows >= 1 && nrows <= nc && ncols >= 1 && ncols <= nv && nc <= (1 << 28), SFA_ERR_ARG,
              "band_matvec: matrix %lld x %lld does not fit the arrays (%lld, %lld)", (long long)nrows,
              (long long)ncols, (long long)nc, (long long)nv);
    const int64_t total = gc.nlines * nc;
    if (total == 0) return SFA_OK;
    const dim3 grid((unsigned)((total + 255) / 256));
    if (dtype == SFA_C128)
        hipLaunchKernelGGL(band_matvec_kernel<double2>, grid, dim3(256), 0, (hipStream_t)stream,
                           (const double2*)v, (double2*)c, gv, gc, (int)nc, (int)nrows, (int)ncols, noffs,
                           offsets, D, scales, accumulate);
    else
        hipLaunchKernelGGL(band_matvec_kernel<double>, grid, dim3(256), 0, (hipStream_t)stream,
                           (const double*)v, (double*)c, gv, gc, (int)nc, (int)nrows, (int)ncols, noffs,
                           offsets, D, scales, accumulate);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

// Batched 2D Helmholtz solves (alpha - lap) u = f on Legendre(SD or SN) x
// Fourier(R2C) in one persistent launch.
//
// Per problem (Nx x Ny physical, M = Nx - 2 composite dofs, Nyh = Ny/2 + 1):
//   T1 = P f                P = Phi^T diag(w): composite Legendre scalar product
//                           (spectralbase.py:550-558 with the stencil of
//                           legendre/bases.py:374 / :502, spectralbase.py:1462-1474)
//   T2 = T1 Df              R2C along y with 1/Ny (fourier/bases.py:157-162),
//                           stored as complex (re, im) pairs
//   per ky: (A + (alpha + ky^2) B) u_hat = T2[:, ky]   (la.py:1346-1364: the
//                           per-mode TDMA of SolverGeneric1ND; A, B closed forms of
//                           legendre/matrices.py:110-162, 271-315)
//   U1 = Phi u_hat          composite synthesis (to_ortho + recursive backward,
//                           spectralbase.py:1616-1634, :484-491)
//   u = U1 Di               C2R along y (imag of k = 0 and Nyquist ignored)
// Phi[j, m] = L_m(x_j) + K2_m L_{m+2}(x_j) on the Legendre-Gauss nodes; Df, Di
// are the real DFT matrices.  All four contractions are FP64 GEMMs on MFMA
// (v_mfma_f64_16x16x4f64), each over half of its inner length: the points are
// symmetric, so even and odd functions act on the sums and differences of
// mirrored values (fold_tile).  The per-ky solves are segmented scans
// (leg_solve_group).  One workgroup owns a problem from start to end; the
// host assigns problems to workgroups largest first (static LPT schedule), so
// the launch needs no atomics and every workgroup exits after its list.
#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <numeric>
#include <queue>
#include <vector>

#include "common.h"
#include "helm_scan.h"
#include "mfma_gemm.h"

namespace sfa {

// ----------------------------------------------------------------- problem table
struct B2Prob {
    int64_t f_off, u_off;     // element offsets of f and u (row-major Nx x Ny float64)
    int64_t phi_off, p_off;   // Phi (Nx x M) and P (M x Nx) in the matrix arena (doubles)
    int64_t df_off, di_off;   // Df (Ny x (Ny+2)) and Di ((Ny+2) x Ny)
    int32_t Nx, Ny, bc, pad;  // bc: 0 Dirichlet (SD), 1 Neumann (SN)
    double alpha;
};

// ----------------------------------------------------------------- MFMA GEMM
constexpr int B2_THREADS = GEMM_THREADS;

// The stage's product (fold_tile: all four matrices are even and odd functions
// on symmetric grids) by the whole workgroup, in tiles of BM x BN outputs, K
// folded and in steps of BK.  An output's MFMA chain does not depend on BM, BN,
// BK, on which workgroup computes the tile, or on the order of the tiles.
template <int MODE>
constexpr int b2_bmu(int BM) { return MODE == FOLD_ROWS_IN || MODE == FOLD_ROWS_OUT ? BM / 2 : BM; }
template <int MODE>
constexpr int b2_bnu(int BN) { return MODE == FOLD_ROWS_IN || MODE == FOLD_ROWS_OUT ? BN : BN / 2; }

template <int MODE, int BM, int BN, int BK>
__device__ __forceinline__ void block_gemm(const double* __restrict__ A, int64_t lda, const double* __restrict__ B,
                                           int64_t ldb, double* __restrict__ C, int64_t ldc, int m, int n, int k,
                                           double* sm)
{
    constexpr bool rows = MODE == FOLD_ROWS_IN || MODE == FOLD_ROWS_OUT;
    const int mu = rows ? (m + 1) / 2 : m;
    const int nu = rows ? n : (MODE == FOLD_COLS_IN ? n / 2 : n / 2 + 1);
    for (int m0 = 0; m0 < mu; m0 += b2_bmu<MODE>(BM))
        for (int n0 = 0; n0 < nu; n0 += b2_bnu<MODE>(BN))
            fold_tile<MODE, b2_bmu<MODE>(BM), b2_bnu<MODE>(BN), BK>(A, lda, B, ldb, C, ldc, m, n, k, m0, n0, sm,
                                                                     sm + FoldShape<b2_bmu<MODE>(BM), b2_bnu<MODE>(BN)>::template lds_a<BK>());
    __syncthreads();  // C complete and LDS free before the caller's next stage
}

constexpr int kB2SolveLds = 6 * 2 * 2 * 8;  // doubles of LDS of the per-ky solves

// LDS doubles of a tile over the modes, and of the solves
template <int BM, int BN, int BK>
constexpr int b2_lds()
{
    using R = FoldShape<BM / 2, BN>;
    using C = FoldShape<BM, BN / 2>;
    constexpr int rows = R::template lds_a<BK>() + R::template lds_b<BK>();
    constexpr int cols = C::template lds_a<BK>() + C::template lds_b<BK>();
    constexpr int tile = rows > cols ? rows : cols;
    return tile > kB2SolveLds ? tile : kB2SolveLds;
}

// ----------------------------------------------------------------- per-ky solve
// Legendre composite Galerkin matrices (legendre/matrices.py:110-162, 271-315),
// h_k = 2/(2k+1):  SD  A_kk = 4k+6, B_kk = h_k + h_{k+2}, B_{k,k+2} = -h_{k+2};
// SN  a_k = k(k+1)/((k+2)(k+3)), A_kk = h_k a_k (k+1/2)((k+2)(k+3) - k(k+1)),
//     B_kk = h_k + a_k^2 h_{k+2}, B_{k,k+2} = -a_k h_{k+2}.  B is symmetric.
// Reciprocals by helm_rcp (5 instructions, within an ulp).
__device__ inline void leg_rows(int i, int bc, double& Akk, double& Bkk, double& Bup)
{
    const double k = (double)i;
    const double h0 = 2.0 * helm_rcp(2.0 * k + 1.0), h2 = 2.0 * helm_rcp(2.0 * k + 5.0);
    if (bc == 0) {
        Akk = 4.0 * k + 6.0;
        Bkk = h0 + h2;
        Bup = -h2;
    } else {
        const double a = k * (k + 1.0) * helm_rcp((k + 2.0) * (k + 3.0));
        Akk = h0 * a * (k + 0.5) * ((k + 2.0) * (k + 3.0) - k * (k + 1.0));
        Bkk = h0 + a * a * h2;
        Bup = -a * h2;
    }
}

// Rows i, i + 2, .. of A + beta B (M rows): diagonal d, upper up, lower lo (=
// the upper one of row i - 2).  Neumann with beta = 0 (ky = 0, alpha = 0): the
// singular row 0 is replaced by u_0 = 0 (the constraint (0, 0) of the
// reference's mode-0 solver), told by gauge.
struct LegRows {
    double d, up, lo, bup;
    bool gauge;
    __device__ __forceinline__ LegRows(int i, int bc)
    {
        double x0, x1;
        bup = 0.0;
        if (i >= 2) leg_rows(i - 2, bc, x0, x1, bup);
    }
    __device__ __forceinline__ void row(int i, int M, int bc, double beta)
    {
        lo = beta * bup;
        double Akk, Bkk;
        leg_rows(i, bc, Akk, Bkk, bup);
        d = Akk + beta * Bkk;
        up = i + 2 < M ? beta * bup : 0.0;
        gauge = bc == 1 && i == 0 && fabs(beta) < 1e-12;
    }
};

// The per-ky solves of TL neighbouring columns (c0 ..) of W0 (M rows, row pitch
// ldw doubles, column ky at 2 ky complex), in place, by the whole workgroup:
// every (ky, parity) chain is cut into 128 / TL segments of E rows, one thread
// each, which reads its rows once and holds them through the three recurrences
// of the Thomas algorithm,
//   c_i = up_i / (d_i - lo_i c_{i-2})            a Moebius map of c
//   r_i = (x_i - lo_i r_{i-2}) / (d_i - ..)      affine in r
//   u_i = r_i - c_i u_{i+2}                      affine in u
// For each, a thread composes its segment's map, a scan over the segments (lanes
// TL apart of one wave, then the parity's two waves through LDS) gives it the
// state that enters, and it runs its rows again.  Bound by the array's one read and one
// write; a thread per chain made four passes over it and two over a pivot
// scratch: 1,024 problems up to 512 x 256, 221 us -> 117 us.
template <int E, int TL>
__device__ __forceinline__ void leg_solve_group(double* __restrict__ W0, int64_t ldw, int M, int Nyh, int c0, int bc,
                                                double alpha, double* sm)
{
    constexpr int WS = 64 / TL;  // segments of a wave
    const int tid = threadIdx.x;
    const int t = tid % TL, seg = (tid & 127) / TL, p = tid >> 7, ws = seg % WS, w1 = (tid >> 6) & 1;
    const int ky = c0 + t;
    const bool valid = ky < Nyh;
    const double beta = alpha + (double)ky * (double)ky;
    // the first row, opaque to the optimiser for each of the two passes that form
    // the rows: it kept the first pass' rows for the second one (and, in the
    // persistent kernel, for the next columns), three numbers a row in registers
    int m0 = seg * E;
    asm volatile("" : "+v"(m0));
    const int K = (M - p + 1) / 2;
    double2* xc = reinterpret_cast<double2*>(W0 + 2 * (valid ? ky : 0)) + (int64_t)p * (ldw / 2);
    // number c of wave w of this parity, line t
    auto slot = [&](int c, int w) -> double& { return sm[((c * 2 + w) * 2 + p) * TL + t]; };
    double2 x[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int m = m0 + e < K ? m0 + e : K - 1;  // (beyond the chain: read again, replaced below)
        x[e] = xc[(int64_t)m * ldw];
    }
    // 1. the segment's map of c as a 2 x 2 matrix on (numerator, denominator)
    double n0 = 1.0, n1 = 0.0, e0 = 0.0, e1 = 1.0;
    auto scaled = [&]() {  // by a power of two, the largest entry in [1/2, 1)
        const double mx = fmax(fmax(fabs(n0), fabs(n1)), fmax(fabs(e0), fabs(e1)));
        const int ex = -__builtin_amdgcn_frexp_exp(mx);
        n0 = ldexp(n0, ex);
        n1 = ldexp(n1, ex);
        e0 = ldexp(e0, ex);
        e1 = ldexp(e1, ex);
    };
    {
        LegRows r(p + 2 * m0, bc);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            if (m0 + e < K) {
                r.row(p + 2 * (m0 + e), M, bc, beta);
                const double u = r.gauge ? 0.0 : r.up, d = r.gauge ? 1.0 : r.d, l = r.gauge ? 0.0 : r.lo;
                const double a0 = u * e0, a1 = u * e1;
                e0 = d * e0 - l * n0;
                e1 = d * e1 - l * n1;
                n0 = a0;
                n1 = a1;
            }
            if (e % 4 == 3 || e == E - 1) scaled();
        }
    }
#pragma unroll
    for (int k = 1; k < WS; k <<= 1) {  // (this segment's map) o (the earlier ones')
        const double on0 = __shfl_up(n0, TL * k), on1 = __shfl_up(n1, TL * k);
        const double oe0 = __shfl_up(e0, TL * k), oe1 = __shfl_up(e1, TL * k);
        if (ws >= k) {
            const double a0 = n0 * on0 + n1 * oe0, a1 = n0 * on1 + n1 * oe1;
            const double b0 = e0 * on0 + e1 * oe0, b1 = e0 * on1 + e1 * oe1;
            n0 = a0;
            n1 = a1;
            e0 = b0;
            e1 = b1;
            scaled();
        }
    }
    if (ws == WS - 1) {  // c = 0 before the chain: the image of (0, 1)
        slot(0, w1) = n1;
        slot(1, w1) = e1;
    }
    double pn0 = __shfl_up(n0, TL), pn1 = __shfl_up(n1, TL), pe0 = __shfl_up(e0, TL), pe1 = __shfl_up(e1, TL);
    if (ws == 0) {
        pn0 = pe1 = 1.0;
        pn1 = pe0 = 0.0;
    }
    __syncthreads();
    const double num0 = w1 ? slot(0, 0) : 0.0, den0 = w1 ? slot(1, 0) : 1.0;
    const double num = pn0 * num0 + pn1 * den0, den = pe0 * num0 + pe1 * den0;
    // 2. the rows' pivots from there, and the segment's map of r
    asm volatile("" : "+v"(m0));
    double cc = num * helm_rcp(den);
    double cu[E], al[E];
    double A = 1.0;
    double2 B = make_double2(0.0, 0.0);
    {
        LegRows r(p + 2 * m0, bc);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            cu[e] = al[e] = 0.0;
            if (m0 + e < K) {
                r.row(p + 2 * (m0 + e), M, bc, beta);
                const double dd = r.gauge ? 0.0 : helm_rcp(r.d - r.lo * cc);
                cc = r.up * dd;
                cu[e] = cc;
                al[e] = -r.lo * dd;
                x[e] = make_double2(x[e].x * dd, x[e].y * dd);
            } else {
                x[e] = make_double2(0.0, 0.0);
            }
            B = make_double2(al[e] * B.x + x[e].x, al[e] * B.y + x[e].y);
            A *= al[e];
        }
    }
#pragma unroll
    for (int k = 1; k < WS; k <<= 1) {
        const double oA = __shfl_up(A, TL * k), ox = __shfl_up(B.x, TL * k), oy = __shfl_up(B.y, TL * k);
        if (ws >= k) {
            B = make_double2(A * ox + B.x, A * oy + B.y);
            A *= oA;
        }
    }
    if (ws == WS - 1) {
        slot(2, w1) = B.x;
        slot(3, w1) = B.y;
    }
    double pA = __shfl_up(A, TL);
    double2 pB = make_double2(__shfl_up(B.x, TL), __shfl_up(B.y, TL));
    if (ws == 0) {
        pA = 1.0;
        pB = make_double2(0.0, 0.0);
    }
    __syncthreads();
    double2 v = w1 ? make_double2(slot(2, 0), slot(3, 0)) : make_double2(0.0, 0.0);
    v = make_double2(pA * v.x + pB.x, pA * v.y + pB.y);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        v = make_double2(al[e] * v.x + x[e].x, al[e] * v.y + x[e].y);
        if (m0 + e < K) x[e] = v;  // (beyond the chain r and c stay 0: the state there)
    }
    // 3. back substitution
    A = 1.0;
    B = make_double2(0.0, 0.0);
#pragma unroll
    for (int e = E - 1; e >= 0; --e) {
        B = make_double2(x[e].x - cu[e] * B.x, x[e].y - cu[e] * B.y);
        A *= -cu[e];
    }
#pragma unroll
    for (int k = 1; k < WS; k <<= 1) {
        const double oA = __shfl_down(A, TL * k), ox = __shfl_down(B.x, TL * k), oy = __shfl_down(B.y, TL * k);
        if (ws + k < WS) {
            B = make_double2(A * ox + B.x, A * oy + B.y);
            A *= oA;
        }
    }
    if (ws == 0) {
        slot(4, w1) = B.x;
        slot(5, w1) = B.y;
    }
    pA = __shfl_down(A, TL);
    pB = make_double2(__shfl_down(B.x, TL), __shfl_down(B.y, TL));
    if (ws == WS - 1) {
        pA = 1.0;
        pB = make_double2(0.0, 0.0);
    }
    __syncthreads();
    v = w1 ? make_double2(0.0, 0.0) : make_double2(slot(4, 1), slot(5, 1));
    v = make_double2(pA * v.x + pB.x, pA * v.y + pB.y);
#pragma unroll
    for (int e = E - 1; e >= 0; --e) {
        v = make_double2(x[e].x - cu[e] * v.x, x[e].y - cu[e] * v.y);
        if (valid && m0 + e < K) xc[(int64_t)(m0 + e) * ldw] = v;
    }
}

// Columns per group of the solves of chains of K rows: with 128 / TL segments
// of at most 8 rows.
__host__ __device__ inline int leg_solve_tl(int K) { return K <= 128 ? 8 : K <= 256 ? 4 : 2; }

// The solves of the column groups first, first + step, .. of a problem.  Rows
// per segment by the chain's length alone, so that a column's arithmetic does
// not depend on how the problem is launched.
__device__ __forceinline__ void batch_solve(double* __restrict__ W0, int64_t ldw, int M, int Nyh, int bc, double alpha,
                                            int first, int step, double* sm)
{
    const int K = (M + 1) / 2;
    auto run = [&](auto Ec, auto Tc) {
        constexpr int E = decltype(Ec)::value, TL = decltype(Tc)::value;
        for (int c0 = first * TL; c0 < Nyh; c0 += step * TL) {
            leg_solve_group<E, TL>(W0, ldw, M, Nyh, c0, bc, alpha, sm);
            __syncthreads();  // the columns' LDS maps are read
        }
    };
    using T8 = std::integral_constant<int, 8>;
    using T4 = std::integral_constant<int, 4>;
    using T2 = std::integral_constant<int, 2>;
    if (K <= 32) run(T2{}, T8{});
    else if (K <= 64) run(T4{}, T8{});
    else if (K <= 96) run(std::integral_constant<int, 6>{}, T8{});
    else if (K <= 128) run(T8{}, T8{});
    else if (K <= 192) run(std::integral_constant<int, 6>{}, T4{});
    else if (K <= 256) run(T8{}, T4{});
    else run(T8{}, T2{});
    __syncthreads();
}

// ----------------------------------------------------------------- persistent kernel
struct B2Args {
    const double* F;
    double* U;
    const B2Prob* probs;
    const int* blk_ptr;  // nblocks + 1
    const int* order;    // problem ids, grouped by workgroup
    const double* mats;  // matrix arena
    double* work;        // per workgroup: wstride doubles
    int64_t wstride;
};

template <int BM, int BN, int BK>
__global__ void __launch_bounds__(B2_THREADS) batch2d_kernel(B2Args a)
{
    __shared__ double sm[b2_lds<BM, BN, BK>()];
    const int b = blockIdx.x;
    double* W0 = a.work + (int64_t)b * a.wstride;
    for (int q = a.blk_ptr[b]; q < a.blk_ptr[b + 1]; ++q) {
        const B2Prob pr = a.probs[a.order[q]];
        const int Nx = pr.Nx, Ny = pr.Ny, M = Nx - 2, Nyh = Ny / 2 + 1, L = Ny + 2;
        const double* f = a.F + pr.f_off;
        double* u = a.U + pr.u_off;
        double* W1 = W0 + (int64_t)M * L;  // Nx x L
        const double* Phi = a.mats + pr.phi_off;
        const double* P = a.mats + pr.p_off;
        const double* Df = a.mats + pr.df_off;
        const double* Di = a.mats + pr.di_off;
        // T1 = P f (M x Ny), held in u
        block_gemm<FOLD_ROWS_IN, BM, BN, BK>(P, Nx, f, Ny, u, Ny, M, Ny, Nx, sm);
        // T2 = T1 Df (M x L) in W0
        block_gemm<FOLD_COLS_IN, BM, BN, BK>(u, Ny, Df, L, W0, L, M, L, Ny, sm);
        // per-ky solve in place
        batch_solve(W0, L, M, Nyh, pr.bc, pr.alpha, 0, 1, sm);
        // U1 = Phi u_hat (Nx x L) in W1
        block_gemm<FOLD_ROWS_OUT, BM, BN, BK>(Phi, M, W0, L, W1, L, Nx, L, M, sm);
        // u = U1 Di (Nx x Ny)
        block_gemm<FOLD_COLS_OUT, BM, BN, BK>(W1, L, Di, Ny, u, Ny, Nx, Ny, L, sm);
    }
}

// ----------------------------------------------------------------- tile-parallel mode
// Each GEMM stage runs as one launch over all (problem, output tile) tasks, the
// solve as one launch over all (problem, group of ky) tasks, so that one large
// problem, or a batch of uneven ones, spreads over the device (512 x 256 alone:
// 62 us, a workgroup for the problem 2259; 1,024 problems up to 512 x 256: 722
// and 2092).
// Per-problem intermediates live at work + woff[p] (W0: (Nx-2) x (Ny+2),
// then W1: Nx x (Ny+2)); T1 is held in u as in the persistent kernel.
struct B2Task {
    int32_t prob, m0, n0, tile;  // first unit row and column of the tile; tile class
};

struct B2WideArgs {
    const double* F;
    double* U;
    const B2Prob* probs;
    const B2Task* tasks;   // this stage's tasks
    const int64_t* woff;   // per problem, in doubles
    const int2* groups;    // the solve launch's problem and column group per workgroup
    const double* mats;
    double* work;
};

constexpr int B2W_BK = 16;
// output tiles (rows, columns) of the tile classes, by stage parity: the
// contractions over x (stages 0, 2) fold rows, those over y (1, 3) columns
constexpr int kB2WClasses = 2;
constexpr int kB2WTile[kB2WClasses][2][2] = {{{32, 64}, {64, 32}}, {{64, 64}, {64, 64}}};

// One task per workgroup, all of a launch's tasks of tile class CLS; every
// output keeps its one MFMA chain over K, so the results do not depend on the
// class.
template <int STAGE, int CLS>
__global__ void __launch_bounds__(B2_THREADS) batch2d_tile_kernel(B2WideArgs a)
{
    constexpr int MODE = STAGE == 0 ? FOLD_ROWS_IN : STAGE == 1 ? FOLD_COLS_IN : STAGE == 2 ? FOLD_ROWS_OUT : FOLD_COLS_OUT;
    constexpr int BMU = b2_bmu<MODE>(kB2WTile[CLS][STAGE & 1][0]), BNU = b2_bnu<MODE>(kB2WTile[CLS][STAGE & 1][1]);
    __shared__ double sA[FoldShape<BMU, BNU>::template lds_a<B2W_BK>()];
    __shared__ double sB[FoldShape<BMU, BNU>::template lds_b<B2W_BK>()];
    const B2Task tk = a.tasks[blockIdx.x];
    const B2Prob pr = a.probs[tk.prob];
    const int Nx = pr.Nx, Ny = pr.Ny, M = Nx - 2, L = Ny + 2;
    double* u = a.U + pr.u_off;
    double* W0 = a.work + a.woff[tk.prob];
    double* W1 = W0 + (int64_t)M * L;
    if constexpr (STAGE == 0)  // T1 = P f (M x Ny) in u
        fold_tile<MODE, BMU, BNU, B2W_BK>(a.mats + pr.p_off, Nx, a.F + pr.f_off, Ny, u, Ny, M, Ny, Nx, tk.m0, tk.n0,
                                          sA, sB);
    else if constexpr (STAGE == 1)  // T2 = T1 Df (M x L) in W0
        fold_tile<MODE, BMU, BNU, B2W_BK>(u, Ny, a.mats + pr.df_off, L, W0, L, M, L, Ny, tk.m0, tk.n0, sA, sB);
    else if constexpr (STAGE == 2)  // U1 = Phi u_hat (Nx x L) in W1
        fold_tile<MODE, BMU, BNU, B2W_BK>(a.mats + pr.phi_off, M, W0, L, W1, L, Nx, L, M, tk.m0, tk.n0, sA, sB);
    else  // u = U1 Di (Nx x Ny)
        fold_tile<MODE, BMU, BNU, B2W_BK>(W1, L, a.mats + pr.di_off, Ny, u, Ny, Nx, Ny, L, tk.m0, tk.n0, sA, sB);
}

// Unit rows and columns of a stage's product, and of its tiles.
struct B2Units {
    int64_t m, n, bm, bn;
};
static B2Units b2_units(int st, int cls, int64_t Nx, int64_t Ny)
{
    const int64_t M = Nx - 2, L = Ny + 2;
    const int64_t bm = kB2WTile[cls][st & 1][0], bn = kB2WTile[cls][st & 1][1];
    switch (st) {
        case 0: return {(M + 1) / 2, Ny, bm / 2, bn};
        case 1: return {M, L / 2, bm, bn / 2};
        case 2: return {(Nx + 1) / 2, L, bm / 2, bn};
        default: return {Nx, Ny / 2 + 1, bm, bn / 2};
    }
}

template <int STAGE>
static int launch_wide_stage(const B2WideArgs& a, int cls, int64_t ntask, hipStream_t s)
{
    const dim3 blk(B2_THREADS), grid((unsigned)ntask);
    if (cls == 1)
        hipLaunchKernelGGL((batch2d_tile_kernel<STAGE, 1>), grid, blk, 0, s, a);
    else
        hipLaunchKernelGGL((batch2d_tile_kernel<STAGE, 0>), grid, blk, 0, s, a);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

__global__ void __launch_bounds__(B2_THREADS) batch2d_wide_solve_kernel(B2WideArgs a)
{
    const int2 g = a.groups[blockIdx.x];
    const B2Prob pr = a.probs[g.x];
    __shared__ double sm[kB2SolveLds];
    batch_solve(a.work + a.woff[g.x], pr.Ny + 2, pr.Nx - 2, pr.Ny / 2 + 1, pr.bc, pr.alpha, g.y, 1 << 20, sm);
}

// ----------------------------------------------------------------- matrix builders
// Phi (Nx x M) and P (M x Nx) for Legendre-Gauss nodes x, weights w: one thread
// per node, the recurrence L_{k+1} = ((2k+1) x L_k - k L_{k-1})/(k+1) in the
// anm/anp form of transforms.pyx:219-323.
__global__ void b2_phi_kernel(const double* __restrict__ x, const double* __restrict__ w, int Nx,
                              int bc, double* __restrict__ Phi, double* __restrict__ P)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= Nx) return;
    const int M = Nx - 2;
    const double xj = x[j], wj = w[j];
    double Lm = 1.0, L0 = xj;
    double L1 = 1.5 * xj * L0 - 0.5 * Lm;  // L_2
    for (int m = 0; m < M; ++m) {
        // Lm = L_m, L0 = L_{m+1}, L1 = L_{m+2}
        const double km = (double)m;
        const double K2 = (bc == 0) ? -1.0 : -km * (km + 1.0) / ((km + 2.0) * (km + 3.0));
        const double v = Lm + K2 * L1;
        Phi[(int64_t)j * M + m] = v;
        P[(int64_t)m * Nx + j] = wj * v;
        const int n = m + 2;  // L_{n+1} = (1/anm_n) x L_n - (anp_n/anm_n) L_{n-1}
        const double anm = (n + 1.0) / (2.0 * n + 1.0), anp = (double)n / (2.0 * n + 1.0);
        const double Ln = (1.0 / anm) * xj * L1 - (anp / anm) * L0;
        Lm = L0;
        L0 = L1;
        L1 = Ln;
    }
}

// Df (Ny x (Ny+2)): [y][2k] = cos(2 pi k y/Ny)/Ny, [y][2k+1] = -sin(..)/Ny;
// Di ((Ny+2) x Ny): [2k][y] = c_k cos, [2k+1][y] = -c_k sin, c_k = 1 at k = 0 and
// Ny/2, else 2.  Angles reduced exactly ((k y) mod Ny) before sincospi.
__global__ void b2_dft_kernel(int Ny, double* __restrict__ Df, double* __restrict__ Di)
{
    const int Nyh = Ny / 2 + 1;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)Ny * Nyh) return;
    const int y = (int)(t / Nyh), k = (int)(t % Nyh);
    const int r = (int)(((int64_t)k * y) % Ny);
    double s, c;
    sincospi(2.0 * (double)r / (double)Ny, &s, &c);
    const int L = Ny + 2;
    Df[(int64_t)y * L + 2 * k] = c / Ny;
    Df[(int64_t)y * L + 2 * k + 1] = -s / Ny;
    const double ck = (k == 0 || 2 * k == Ny) ? 1.0 : 2.0;
    Di[(int64_t)(2 * k) * Ny + y] = ck * c;
    Di[(int64_t)(2 * k + 1) * Ny + y] = (k == 0 || 2 * k == Ny) ? 0.0 : -ck * s;
}

// MFMA lane-layout probe: A (16 x 4) = i + 100 k, B (4 x 16) = j + 1000 k;
// out[l * 4 + r] = D register r of lane l.
__global__ void mfma_probe_kernel(double* out)
{
    const int l = threadIdx.x;
    const double a = (double)(l % 16) + 100.0 * (l / 16);
    const double b = (double)(l % 16) + 1000.0 * (l / 16);
    v4d d = mfma16(a, b, (v4d){0.0, 0.0, 0.0, 0.0});
    for (int r = 0; r < 4; ++r) out[l * 4 + r] = d[r];
}

// ----------------------------------------------------------------- host side
// Legendre-Gauss nodes (ascending) and weights: Newton on the three-term
// recurrence in long double from the cosine guess, weights 2/((1-x^2) P'^2),
// symmetrised; cached per N for the process.
static std::mutex g_lg_mu;
static std::map<int, std::pair<std::vector<double>, std::vector<double>>> g_lg;

static void lg_nodes(int N, std::vector<double>& xo, std::vector<double>& wo)
{
    {
        std::lock_guard<std::mutex> lk(g_lg_mu);
        auto it = g_lg.find(N);
        if (it != g_lg.end()) {
            xo = it->second.first;
            wo = it->second.second;
            return;
        }
    }
    typedef long double ld;
    const ld pi = 3.141592653589793238462643383279502884L;
    std::vector<ld> x(N), w(N);
    auto pdp = [&](ld xv, ld& p, ld& dp) {
        ld p0 = 1.0L, p1 = xv;
        for (int k = 1; k < N; ++k) {
            const ld p2 = ((2 * k + 1) * xv * p1 - k * p0) / (k + 1);
            p0 = p1;
            p1 = p2;
        }
        p = p1;
        dp = N * (xv * p1 - p0) / (xv * xv - 1.0L);
    };
    for (int i = 0; i < N; ++i) {
        ld xv = std::cos(pi * ((ld)(i + 1) - 0.25L) / ((ld)N + 0.5L));
        for (int it = 0; it < 100; ++it) {
            ld p, dp;
            pdp(xv, p, dp);
            const ld dx = p / dp;
            xv -= dx;
            if (std::fabs(dx) < 1e-19L) break;
        }
        ld p, dp;
        pdp(xv, p, dp);
        x[i] = xv;
        w[i] = 2.0L / ((1.0L - xv * xv) * dp * dp);
    }
    // ascending, rounded, symmetrised
    std::vector<int> o(N);
    std::iota(o.begin(), o.end(), 0);
    std::sort(o.begin(), o.end(), [&](int a, int b) { return x[a] < x[b]; });
    std::vector<double> xs(N), ws(N);
    for (int i = 0; i < N; ++i) {
        xs[i] = (double)x[o[i]];
        ws[i] = (double)w[o[i]];
    }
    xo.assign(N, 0.0);
    wo.assign(N, 0.0);
    for (int i = 0; i < N; ++i) {
        xo[i] = 0.5 * (xs[i] - xs[N - 1 - i]);
        wo[i] = 0.5 * (ws[i] + ws[N - 1 - i]);
    }
    std::lock_guard<std::mutex> lk(g_lg_mu);
    g_lg[N] = std::make_pair(xo, wo);
}

// Device copies of the nodes and weights per N (x then w), for the process.
static std::map<std::pair<int, int>, double*> g_lg_dev;  // (N, device)

static const double* lg_nodes_dev(int N)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    {
        std::lock_guard<std::mutex> lk(g_lg_mu);
        auto it = g_lg_dev.find(std::make_pair(N, dev));
        if (it != g_lg_dev.end()) return it->second;
    }
    std::vector<double> x, w;
    lg_nodes(N, x, w);
    x.insert(x.end(), w.begin(), w.end());
    double* d = nullptr;
    if (hipMalloc(&d, x.size() * sizeof(double)) != hipSuccess) return nullptr;
    if (hipMemcpy(d, x.data(), x.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
        hipFree(d);
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(g_lg_mu);
    g_lg_dev[std::make_pair(N, dev)] = d;
    return d;
}

static int64_t leg_elems(int Nx) { return 2 * (int64_t)Nx * (Nx - 2); }
static int64_t dft_elems(int Ny) { return 2 * (int64_t)Ny * (Ny + 2); }

static int build_leg(int Nx, int bc, double* out, hipStream_t s)
{
    const double* xw = lg_nodes_dev(Nx);
    SFA_CHECK(xw, SFA_ERR_HIP, "node table allocation failed");
    hipLaunchKernelGGL(b2_phi_kernel, dim3((unsigned)((Nx + 127) / 128)), dim3(128), 0, s, xw, xw + Nx, Nx,
                       bc, out, out + (int64_t)Nx * (Nx - 2));
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

static int build_dft(int Ny, double* out, hipStream_t s)
{
    const int64_t nt = (int64_t)Ny * (Ny / 2 + 1);
    hipLaunchKernelGGL(b2_dft_kernel, dim3((unsigned)((nt + 255) / 256)), dim3(256), 0, s, Ny, out,
                       out + (int64_t)Ny * (Ny + 2));
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

static int64_t r256(int64_t b) { return (b + 255) / 256 * 256; }

// plan layout: problem table | blk_ptr | order [| matrix arena (self-contained plans)]
struct B2Layout {
    int64_t off_probs, off_blk, off_order, off_mats, bytes;
};

static void b2_layout(int nprob, int nblocks, int64_t mats_elems, B2Layout* L)
{
    L->off_probs = 0;
    L->off_blk = r256((int64_t)nprob * sizeof(B2Prob));
    L->off_order = L->off_blk + r256((int64_t)(nblocks + 1) * 4);
    L->off_mats = L->off_order + r256((int64_t)nprob * 4);
    L->bytes = L->off_mats + r256(mats_elems * 8);
}

// distinct matrices of a batch: (Nx, bc) -> Phi offset, Ny -> Df offset
static int64_t b2_arena(int nprob, const int* Nx, const int* Ny, const int* bc,
                        std::map<std::pair<int, int>, int64_t>* phi, std::map<int, int64_t>* dft)
{
    int64_t mats = 0;
    for (int i = 0; i < nprob; ++i) {
        const auto key = std::make_pair(Nx[i], bc[i] ? 1 : 0);
        if (!phi->count(key)) {
            (*phi)[key] = mats;
            mats += leg_elems(Nx[i]);
        }
        if (!dft->count(Ny[i])) {
            (*dft)[Ny[i]] = mats;
            mats += dft_elems(Ny[i]);
        }
    }
    return mats;
}

static double b2_cost(int Nx, int Ny)
{
    // flops of the four contractions plus a memory and fixed term (units ~ flops)
    const double x = Nx, y = Ny;
    return 4.0 * x * y * (x + y) + 64.0 * x * y + 2.0e5;
}

struct B2Info {
    int nprob, nblocks;
    int64_t off_probs, off_blk, off_order;
    const double* mats;
    int64_t wstride;  // doubles per workgroup
};
static std::mutex g_b2_mu;
static std::map<const void*, B2Info> g_b2;
// tile-parallel plan: problem table | tasks of the four GEMM stages | woff
struct B2WideInfo {
    int nprob;
    int cls[4];  // tile class of each stage
    int64_t ntask[4], off_task[4];
    int64_t off_probs, off_woff, work_doubles;
    int64_t ngroup;  // column groups of the solve
    const double* mats;
};
static std::map<const void*, B2WideInfo> g_b2w;

static int64_t b2_wstride(int nprob, const int* Nx, const int* Ny)
{
    int64_t mx = 0;
    for (int i = 0; i < nprob; ++i) {
        const int64_t L = Ny[i] + 2;
        mx = std::max(mx, (int64_t)(Nx[i] - 2) * L + (int64_t)Nx[i] * L);
    }
    return (mx + 31) / 32 * 32;
}

// Problem table and static LPT schedule into the plan; registers the plan.
// Validated problem table.
static int b2_table(int nprob, const int* Nx, const int* Ny, const double* alpha, const int* bc,
                    const int64_t* f_off, const int64_t* u_off, int64_t f_elems, int64_t u_elems,
                    const int64_t* phi_off, const int64_t* df_off, int64_t mats_elems,
                    std::vector<B2Prob>& probs)
{
    probs.resize(nprob);
    for (int i = 0; i < nprob; ++i) {
        const int64_t n = (int64_t)Nx[i] * Ny[i];
        SFA_CHECK(f_off[i] >= 0 && f_off[i] + n <= f_elems, SFA_ERR_ARG,
                  "problem %d: f range [%lld, %lld) outside the %lld-element input", i,
                  (long long)f_off[i], (long long)(f_off[i] + n), (long long)f_elems);
        SFA_CHECK(u_off[i] >= 0 && u_off[i] + n <= u_elems, SFA_ERR_ARG,
                  "problem %d: u range outside the %lld-element output", i, (long long)u_elems);
        SFA_CHECK(phi_off[i] >= 0 && phi_off[i] + leg_elems(Nx[i]) <= mats_elems && df_off[i] >= 0 &&
                      df_off[i] + dft_elems(Ny[i]) <= mats_elems,
                  SFA_ERR_ARG, "problem %d: matrix offsets outside the %lld-element arena", i,
                  (long long)mats_elems);
        B2Prob& p = probs[i];
        p.f_off = f_off[i];
        p.u_off = u_off[i];
        p.phi_off = phi_off[i];
        p.p_off = phi_off[i] + (int64_t)Nx[i] * (Nx[i] - 2);
        p.df_off = df_off[i];
        p.di_off = df_off[i] + (int64_t)Ny[i] * (Ny[i] + 2);
        p.Nx = Nx[i];
        p.Ny = Ny[i];
        p.bc = bc[i] ? 1 : 0;
        p.pad = 0;
        p.alpha = alpha[i];
    }
    return SFA_OK;
}

static int b2_plan_core(int nprob, const int* Nx, const int* Ny, const double* alpha, const int* bc,
                        const int64_t* f_off, const int64_t* u_off, int64_t f_elems, int64_t u_elems,
                        const double* mats, const int64_t* phi_off, const int64_t* df_off,
                        int64_t mats_elems, int nblocks, void* plan, int64_t plan_bytes,
                        hipStream_t s)
{
    B2Layout L;
    b2_layout(nprob, nblocks, 0, &L);
    SFA_CHECK(plan_bytes >= L.bytes, SFA_ERR_ARG, "plan buffer too small (%lld < %lld)",
              (long long)plan_bytes, (long long)L.bytes);
    std::vector<B2Prob> probs;
    int rc = b2_table(nprob, Nx, Ny, alpha, bc, f_off, u_off, f_elems, u_elems, phi_off, df_off,
                      mats_elems, probs);
    if (rc) return rc;
    // static LPT schedule: largest first onto the least loaded workgroup
    std::vector<int> ids(nprob);
    std::iota(ids.begin(), ids.end(), 0);
    std::stable_sort(ids.begin(), ids.end(),
                     [&](int a, int b) { return b2_cost(Nx[a], Ny[a]) > b2_cost(Nx[b], Ny[b]); });
    typedef std::pair<double, int> LB;
    std::priority_queue<LB, std::vector<LB>, std::greater<LB>> heap;
    for (int b = 0; b < nblocks; ++b) heap.push(LB(0.0, b));
    std::vector<std::vector<int>> lists(nblocks);
    for (int id : ids) {
        LB t = heap.top();
        heap.pop();
        lists[t.second].push_back(id);
        t.first += b2_cost(Nx[id], Ny[id]);
        heap.push(t);
    }
    std::vector<int> blk(nblocks + 1, 0), order;
    order.reserve(nprob);
    for (int b = 0; b < nblocks; ++b) {
        blk[b] = (int)order.size();
        for (int id : lists[b]) order.push_back(id);
    }
    blk[nblocks] = (int)order.size();
    char* pb = (char*)plan;
    SFA_HIP(hipMemcpyAsync(pb + L.off_probs, probs.data(), probs.size() * sizeof(B2Prob),
                           hipMemcpyHostToDevice, s));
    SFA_HIP(hipMemcpyAsync(pb + L.off_blk, blk.data(), blk.size() * 4, hipMemcpyHostToDevice, s));
    SFA_HIP(hipMemcpyAsync(pb + L.off_order, order.data(), order.size() * 4, hipMemcpyHostToDevice, s));
    SFA_HIP(hipStreamSynchronize(s));  // host vectors are copied before they go out of scope
    std::lock_guard<std::mutex> lk(g_b2_mu);
    g_b2w.erase(plan);  // the address may have held a tile-parallel plan
    g_b2[plan] = B2Info{nprob, nblocks, L.off_probs, L.off_blk, L.off_order, mats,
                        b2_wstride(nprob, Nx, Ny)};
    return SFA_OK;
}


// Tile class of each stage: the largest whose task count still gives every
// one of the kWideCus compute units a few workgroups (more operand reuse per
// tile where the batch is large, more tiles where a few problems must fill the
// device); ntask[st] is that stage's task count.
constexpr int kWideCus = 256;  // compute units of an MI355X

static void b2_wide_shape(int nprob, const int* Nx, const int* Ny, int64_t ntask[4], int64_t* work,
                          int cls[4] = nullptr)
{
    auto cdiv = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
    *work = 0;
    int64_t cnt[4][kB2WClasses] = {};
    for (int i = 0; i < nprob; ++i) {
        const int64_t M = Nx[i] - 2, L = Ny[i] + 2, X = Nx[i], Y = Ny[i];
        for (int st = 0; st < 4; ++st)
            for (int c = 0; c < kB2WClasses; ++c) {
                const B2Units t = b2_units(st, c, X, Y);
                cnt[st][c] += cdiv(t.m, t.bm) * cdiv(t.n, t.bn);
            }
        *work += (M * L + X * L + 31) / 32 * 32;
    }
    for (int st = 0; st < 4; ++st) {
        int c = kB2WClasses - 1;
        while (c > 0 && cnt[st][c] < 4 * kWideCus) --c;
        ntask[st] = cnt[st][c];
        if (cls) cls[st] = c;
    }
}

// A stage's tasks in launch order.  Workgroups go to the 8 XCDs in turn, so the
// tiles of a problem, which share its operands, take every eighth place and read
// them through one L2 (in the order of the problems most of the eight fetched
// them: 1,024 problems up to 512 x 256, the four stages 719 -> 631 us; they were
// 1,011 before the contractions were folded).  The tasks with the longest K come
// first.  A problem with more than a 64th of the tasks is cut into runs of that
// many, so that few problems still use every XCD.
static void b2_wide_order(int st, int cls, int nprob, const int* Nx, const int* Ny, int64_t ntask,
                          std::vector<B2Task>& out)
{
    std::vector<int> ids(nprob);
    std::iota(ids.begin(), ids.end(), 0);
    auto klen = [&](int i) { return st % 2 == 0 ? Nx[i] : Ny[i]; };
    std::stable_sort(ids.begin(), ids.end(), [&](int a, int b) { return klen(a) > klen(b); });
    const int64_t run = std::max<int64_t>(4, ntask / 64);
    std::vector<B2Task> q[8];
    double load[8] = {};
    for (int i : ids) {
        const B2Units t = b2_units(st, cls, Nx[i], Ny[i]);
        const double cost = klen(i) / 32.0 + 4.0;  // K steps of 16 units, and a tile's start and end
        int64_t left = 0;
        int x = 0;
        for (int m0 = 0; m0 < t.m; m0 += (int)t.bm)
            for (int n0 = 0; n0 < t.n; n0 += (int)t.bn) {
                if (left-- == 0) {
                    left = run - 1;
                    x = (int)(std::min_element(load, load + 8) - load);
                }
                q[x].push_back(B2Task{i, m0, n0, cls});
                load[x] += cost;
            }
    }
    size_t at[8] = {};
    out.clear();
    out.reserve((size_t)ntask);
    for (int64_t n = 0; n < ntask; ++n) {
        int x = (int)(n % 8);
        if (at[x] == q[x].size())  // this XCD's list is done: from the longest rest
            for (int y = 0; y < 8; ++y)
                if (q[y].size() - at[y] > q[x].size() - at[x]) x = y;
        out.push_back(q[x][at[x]++]);
    }
}

// plan layout: problem table | tasks of each stage | per-problem workspace
// offsets | column groups of the solve
static int leg_groups(int Nx, int Ny)
{
    const int tl = leg_solve_tl((Nx - 1) / 2);
    return (Ny / 2 + tl) / tl;
}

static int64_t b2_wide_groups(int nprob, const int* Nx, const int* Ny)
{
    int64_t n = 0;
    for (int i = 0; i < nprob; ++i) n += leg_groups(Nx[i], Ny[i]);
    return n;
}

static int64_t b2_wide_bytes(int nprob, const int* Nx, const int* Ny, const int64_t ntask[4], int64_t off_task[4],
                             int64_t* off_woff)
{
    int64_t o = r256((int64_t)nprob * sizeof(B2Prob));
    for (int st = 0; st < 4; ++st) {
        off_task[st] = o;
        o += r256(ntask[st] * (int64_t)sizeof(B2Task));
    }
    *off_woff = o;
    o += r256((int64_t)nprob * 8);
    return o + r256(b2_wide_groups(nprob, Nx, Ny) * (int64_t)sizeof(int2));
}

template <int BM, int BN, int BK>
static int launch_b2(const B2Args& a, int nblocks, hipStream_t s)
{
    hipLaunchKernelGGL((batch2d_kernel<BM, BN, BK>), dim3((unsigned)nblocks), dim3(B2_THREADS), 0, s, a);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

}  // namespace sfa

using namespace sfa;

// block tiles (BM, BN, BK) of the launch variants
// (64, 128, 32) and (128, 64, 32) need more than 256 VGPRs + AGPRs and spill: left out
static const int kB2Variants[][3] = {{64, 64, 16}, {32, 64, 16}, {64, 128, 16}, {128, 64, 16},
                                     {64, 64, 32}};

extern "C" int sfa_batch2d_variants(int* bm, int* bn, int cap)
{
    const int n = (int)(sizeof(kB2Variants) / sizeof(kB2Variants[0]));
    for (int i = 0; i < n && i < cap; ++i) {
        if (bm) bm[i] = kB2Variants[i][0];
        if (bn) bn[i] = kB2Variants[i][1] * 1000 + kB2Variants[i][2];
    }
    return n;
}

static int b2_check(int nprob, const int* Nx, const int* Ny, const int* bc, int nblocks)
{
    SFA_CHECK(nprob >= 1 && Nx && Ny && bc, SFA_ERR_ARG, "need nprob >= 1 and size arrays");
    SFA_CHECK(nblocks >= 1 && nblocks <= 65536, SFA_ERR_ARG, "nblocks must be in [1, 65536]");
    for (int i = 0; i < nprob; ++i) {
        SFA_CHECK(Nx[i] >= 8 && Nx[i] <= 1024 && Nx[i] % 2 == 0, SFA_ERR_ARG,
                  "problem %d: Nx=%d must be even in [8, 1024]", i, Nx[i]);
        SFA_CHECK(Ny[i] >= 4 && Ny[i] <= 1024 && Ny[i] % 2 == 0, SFA_ERR_ARG,
                  "problem %d: Ny=%d must be even in [4, 1024]", i, Ny[i]);
        SFA_CHECK(bc[i] == 0 || bc[i] == 1, SFA_ERR_ARG, "problem %d: bc must be 0 or 1", i);
    }
    return SFA_OK;
}

extern "C" int64_t sfa_batch2d_plan_bytes(int nprob, const int* Nx, const int* Ny, const int* bc,
                                          int nblocks)
{
    if (b2_check(nprob, Nx, Ny, bc, nblocks)) return -1;
    std::map<std::pair<int, int>, int64_t> phi;
    std::map<int, int64_t> dft;
    B2Layout L;
    b2_layout(nprob, nblocks, b2_arena(nprob, Nx, Ny, bc, &phi, &dft), &L);
    return L.bytes;
}

extern "C" int64_t sfa_batch2d_plan_ext_bytes(int nprob, int nblocks)
{
    if (nprob < 1 || nblocks < 1) return -1;
    B2Layout L;
    b2_layout(nprob, nblocks, 0, &L);
    return L.bytes;
}

extern "C" int64_t sfa_batch2d_workspace(int nprob, const int* Nx, const int* Ny, int nblocks)
{
    if (nprob < 1 || nblocks < 1 || !Nx || !Ny) return -1;
    return b2_wstride(nprob, Nx, Ny) * 8 * (int64_t)nblocks;
}

extern "C" int64_t sfa_batch2d_leg_elems(int Nx) { return (Nx >= 8 && Nx % 2 == 0) ? leg_elems(Nx) : -1; }
extern "C" int64_t sfa_batch2d_dft_elems(int Ny) { return (Ny >= 4 && Ny % 2 == 0) ? dft_elems(Ny) : -1; }

extern "C" int sfa_batch2d_leg_matrices(int Nx, int bc, double* out, void* stream)
{
    SFA_CHECK(Nx >= 8 && Nx <= 1024 && Nx % 2 == 0 && (bc == 0 || bc == 1) && out, SFA_ERR_ARG,
              "need even Nx in [8, 1024], bc 0/1, out");
    return build_leg(Nx, bc, out, (hipStream_t)stream);
}

extern "C" int sfa_batch2d_dft_matrices(int Ny, double* out, void* stream)
{
    SFA_CHECK(Ny >= 4 && Ny <= 1024 && Ny % 2 == 0 && out, SFA_ERR_ARG, "need even Ny in [4, 1024], out");
    return build_dft(Ny, out, (hipStream_t)stream);
}

extern "C" int sfa_batch2d_plan(int nprob, const int* Nx, const int* Ny, const double* alpha,
                                const int* bc, const int64_t* f_off, const int64_t* u_off,
                                int64_t f_elems, int64_t u_elems, int nblocks, void* plan,
                                int64_t plan_bytes, void* stream)
{
    int rc;
    if ((rc = b2_check(nprob, Nx, Ny, bc, nblocks))) return rc;
    SFA_CHECK(alpha && f_off && u_off && plan, SFA_ERR_ARG, "NULL argument");
    std::map<std::pair<int, int>, int64_t> phi;
    std::map<int, int64_t> dft;
    const int64_t mats = b2_arena(nprob, Nx, Ny, bc, &phi, &dft);
    B2Layout L;
    b2_layout(nprob, nblocks, mats, &L);
    SFA_CHECK(plan_bytes >= L.bytes, SFA_ERR_ARG, "plan buffer too small (%lld < %lld)",
              (long long)plan_bytes, (long long)L.bytes);
    hipStream_t s = (hipStream_t)stream;
    double* dm = (double*)((char*)plan + L.off_mats);
    for (auto& kv : phi)
        if ((rc = build_leg(kv.first.first, kv.first.second, dm + kv.second, s))) return rc;
    for (auto& kv : dft)
        if ((rc = build_dft(kv.first, dm + kv.second, s))) return rc;
    std::vector<int64_t> po(nprob), dfo(nprob);
    for (int i = 0; i < nprob; ++i) {
        po[i] = phi[std::make_pair(Nx[i], bc[i] ? 1 : 0)];
        dfo[i] = dft[Ny[i]];
    }
    return b2_plan_core(nprob, Nx, Ny, alpha, bc, f_off, u_off, f_elems, u_elems, dm, po.data(),
                        dfo.data(), mats, nblocks, plan, plan_bytes, s);
}

extern "C" int sfa_batch2d_plan_ext(int nprob, const int* Nx, const int* Ny, const double* alpha,
                                    const int* bc, const int64_t* f_off, const int64_t* u_off,
                                    int64_t f_elems, int64_t u_elems, const double* mats,
                                    const int64_t* phi_off, const int64_t* df_off,
                                    int64_t mats_elems, int nblocks, void* plan,
                                    int64_t plan_bytes, void* stream)
{
    int rc;
    if ((rc = b2_check(nprob, Nx, Ny, bc, nblocks))) return rc;
    SFA_CHECK(alpha && f_off && u_off && plan && mats && phi_off && df_off, SFA_ERR_ARG,
              "NULL argument");
    return b2_plan_core(nprob, Nx, Ny, alpha, bc, f_off, u_off, f_elems, u_elems, mats, phi_off,
                        df_off, mats_elems, nblocks, plan, plan_bytes, (hipStream_t)stream);
}

extern "C" int sfa_batch2d_solve(const double* F, double* U, const void* plan, void* work,
                                 int64_t work_bytes, int variant, void* stream)
{
    B2Info pi;
    {
        std::lock_guard<std::mutex> lk(g_b2_mu);
        auto it = g_b2.find(plan);
        SFA_CHECK(it != g_b2.end(), SFA_ERR_ARG, "plan was not built by sfa_batch2d_plan(_ext)");
        pi = it->second;
    }
    SFA_CHECK(F && U && work, SFA_ERR_ARG, "NULL argument");
    SFA_CHECK(work_bytes >= pi.wstride * 8 * (int64_t)pi.nblocks, SFA_ERR_ARG,
              "workspace too small (%lld < %lld)", (long long)work_bytes,
              (long long)(pi.wstride * 8 * (int64_t)pi.nblocks));
    const int nv = sfa_batch2d_variants(nullptr, nullptr, 0);
    SFA_CHECK(variant >= 0 && variant < nv, SFA_ERR_ARG, "variant must be in [0, %d)", nv);
    const char* pb = (const char*)plan;
    B2Args a;
    a.F = F;
    a.U = U;
    a.probs = (const B2Prob*)(pb + pi.off_probs);
    a.blk_ptr = (const int*)(pb + pi.off_blk);
    a.order = (const int*)(pb + pi.off_order);
    a.mats = pi.mats;
    a.work = (double*)work;
    a.wstride = pi.wstride;
    hipStream_t s = (hipStream_t)stream;
    switch (variant) {
        case 0: return launch_b2<64, 64, 16>(a, pi.nblocks, s);
        case 1: return launch_b2<32, 64, 16>(a, pi.nblocks, s);
        case 2: return launch_b2<64, 128, 16>(a, pi.nblocks, s);
        case 3: return launch_b2<128, 64, 16>(a, pi.nblocks, s);
        default: return launch_b2<64, 64, 32>(a, pi.nblocks, s);
    }
}

extern "C" int sfa_batch2d_release(const void* plan)
{
    std::lock_guard<std::mutex> lk(g_b2_mu);
    g_b2.erase(plan);
    g_b2w.erase(plan);
    return SFA_OK;
}

extern "C" int64_t sfa_batch2d_wide_plan_bytes(int nprob, const int* Nx, const int* Ny)
{
    if (nprob < 1 || !Nx || !Ny) return -1;
    int64_t nt[4], ot[4], ow, work;
    b2_wide_shape(nprob, Nx, Ny, nt, &work);
    return b2_wide_bytes(nprob, Nx, Ny, nt, ot, &ow);
}

extern "C" int64_t sfa_batch2d_wide_workspace(int nprob, const int* Nx, const int* Ny)
{
    if (nprob < 1 || !Nx || !Ny) return -1;
    int64_t nt[4], work;
    b2_wide_shape(nprob, Nx, Ny, nt, &work);
    return work * 8;
}

extern "C" int sfa_batch2d_wide_plan(int nprob, const int* Nx, const int* Ny, const double* alpha,
                                     const int* bc, const int64_t* f_off, const int64_t* u_off,
                                     int64_t f_elems, int64_t u_elems, const double* mats,
                                     const int64_t* phi_off, const int64_t* df_off,
                                     int64_t mats_elems, void* plan, int64_t plan_bytes, void* stream)
{
    int rc;
    if ((rc = b2_check(nprob, Nx, Ny, bc, 1))) return rc;
    SFA_CHECK(alpha && f_off && u_off && plan && mats && phi_off && df_off, SFA_ERR_ARG,
              "NULL argument");
    std::vector<B2Prob> probs;
    if ((rc = b2_table(nprob, Nx, Ny, alpha, bc, f_off, u_off, f_elems, u_elems, phi_off, df_off,
                       mats_elems, probs)))
        return rc;
    B2WideInfo wi;
    wi.nprob = nprob;
    int* cls = wi.cls;
    b2_wide_shape(nprob, Nx, Ny, wi.ntask, &wi.work_doubles, cls);
    const int64_t bytes = b2_wide_bytes(nprob, Nx, Ny, wi.ntask, wi.off_task, &wi.off_woff);
    SFA_CHECK(plan_bytes >= bytes, SFA_ERR_ARG, "plan buffer too small (%lld < %lld)",
              (long long)plan_bytes, (long long)bytes);
    wi.off_probs = 0;
    wi.mats = mats;
    wi.ngroup = b2_wide_groups(nprob, Nx, Ny);
    std::vector<B2Task> tasks[4];
    for (int st = 0; st < 4; ++st) b2_wide_order(st, cls[st], nprob, Nx, Ny, wi.ntask[st], tasks[st]);
    std::vector<int64_t> woff(nprob);
    int64_t w = 0;
    for (int i = 0; i < nprob; ++i) {
        const int M = Nx[i] - 2, L = Ny[i] + 2, X = Nx[i];
        woff[i] = w;
        w += ((int64_t)M * L + (int64_t)X * L + 31) / 32 * 32;
    }
    hipStream_t s = (hipStream_t)stream;
    char* pb = (char*)plan;
    SFA_HIP(hipMemcpyAsync(pb, probs.data(), probs.size() * sizeof(B2Prob), hipMemcpyHostToDevice, s));
    for (int st = 0; st < 4; ++st)
        SFA_HIP(hipMemcpyAsync(pb + wi.off_task[st], tasks[st].data(), tasks[st].size() * sizeof(B2Task),
                               hipMemcpyHostToDevice, s));
    SFA_HIP(hipMemcpyAsync(pb + wi.off_woff, woff.data(), woff.size() * 8, hipMemcpyHostToDevice, s));
    // the solve takes the problems with the most rows first, so that they do not
    // finish last
    std::vector<int> order(nprob);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return Nx[x] > Nx[y]; });
    std::vector<int2> groups;
    groups.reserve((size_t)wi.ngroup);
    for (int i : order)
        for (int g = 0; g < leg_groups(Nx[i], Ny[i]); ++g) groups.push_back(make_int2(i, g));
    SFA_HIP(hipMemcpyAsync(pb + wi.off_woff + r256((int64_t)nprob * 8), groups.data(), groups.size() * sizeof(int2),
                           hipMemcpyHostToDevice, s));
    SFA_HIP(hipStreamSynchronize(s));  // host vectors are copied before they go out of scope
    std::lock_guard<std::mutex> lk(g_b2_mu);
    g_b2.erase(plan);  // the address may have held a persistent-mode plan
    g_b2w[plan] = wi;
    return SFA_OK;
}

extern "C" int sfa_batch2d_wide_solve(const double* F, double* U, const void* plan, void* work,
                                      int64_t work_bytes, void* stream)
{
    B2WideInfo wi;
    {
        std::lock_guard<std::mutex> lk(g_b2_mu);
        auto it = g_b2w.find(plan);
        SFA_CHECK(it != g_b2w.end(), SFA_ERR_ARG, "plan was not built by sfa_batch2d_wide_plan");
        wi = it->second;
    }
    SFA_CHECK(F && U && work, SFA_ERR_ARG, "NULL argument");
    SFA_CHECK(work_bytes >= wi.work_doubles * 8, SFA_ERR_ARG, "workspace too small (%lld < %lld)",
              (long long)work_bytes, (long long)(wi.work_doubles * 8));
    const char* pb = (const char*)plan;
    B2WideArgs a;
    a.F = F;
    a.U = U;
    a.probs = (const B2Prob*)pb;
    a.woff = (const int64_t*)(pb + wi.off_woff);
    a.groups = (const int2*)(pb + wi.off_woff + r256((int64_t)wi.nprob * 8));
    a.mats = wi.mats;
    a.work = (double*)work;
    hipStream_t s = (hipStream_t)stream;
    const dim3 blk(B2_THREADS);
    int rc;
    a.tasks = (const B2Task*)(pb + wi.off_task[0]);
    if ((rc = launch_wide_stage<0>(a, wi.cls[0], wi.ntask[0], s))) return rc;
    a.tasks = (const B2Task*)(pb + wi.off_task[1]);
    if ((rc = launch_wide_stage<1>(a, wi.cls[1], wi.ntask[1], s))) return rc;
    hipLaunchKernelGGL(batch2d_wide_solve_kernel, dim3((unsigned)wi.ngroup), blk, 0, s, a);
    SFA_LAUNCH_CHECK();
    a.tasks = (const B2Task*)(pb + wi.off_task[2]);
    if ((rc = launch_wide_stage<2>(a, wi.cls[2], wi.ntask[2], s))) return rc;
    a.tasks = (const B2Task*)(pb + wi.off_task[3]);
    return launch_wide_stage<3>(a, wi.cls[3], wi.ntask[3], s);
}

extern "C" int sfa_mfma_f64_layout_probe(double* out, void* stream)
{
    SFA_CHECK(out != nullptr, SFA_ERR_ARG, "out is NULL");
    hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, out);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

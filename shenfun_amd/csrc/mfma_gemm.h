// FP64 MFMA GEMM tile shared by the batched 2D solver and the dense line
// contraction: C (m x n) = A (m x k) B (k x n), row-major, one workgroup of
// GEMM_THREADS threads per BM x BN output tile.
#pragma once
#include "common.h"

namespace sfa {

typedef double v4d __attribute__((ext_vector_type(4)));

constexpr int GEMM_THREADS = 256;

// MFMA f64 16x16x4 operand layout (lane l of the wave): A[i][k] at i = l % 16,
// k = l / 16; B[k][j] at j = l % 16, k = l / 16; D[i][j] in register r of lane
// l with i = 4 r + l / 16, j = l % 16 (checked by sfa_mfma_f64_layout_probe).
__device__ inline v4d mfma16(double a, double b, v4d c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}


// C (m x n, ldc) = A (m x k, lda) B (k x n, ldb), all row-major FP64, by the
// whole workgroup (4 waves in a 2 x 2 grid over a BM x BN block tile, K in
// steps of BK).  sA: BK x (BM + 8), sB: BK x (BN + 8) doubles of LDS.
// Out-of-range operand elements load as zero; stores are bounds-checked.
// Each output is one MFMA accumulation chain over K in ascending order, so
// the result does not depend on BM, BN or BK.
template <int BM, int BN, int BK>
__device__ void gemm_tile(const double* __restrict__ A, int64_t lda, const double* __restrict__ B,
                          int64_t ldb, double* __restrict__ C, int64_t ldc, int m, int n, int k,
                          int m0, int n0, double* sA, double* sB)
{
    constexpr int SA = BM + 8, SB = BN + 8;
    constexpr int TI = BM / 32, TJ = BN / 32;
    constexpr int LA = BM * BK / GEMM_THREADS, LB = BK * BN / GEMM_THREADS;
    static_assert(LA >= 1 && LB >= 1 && TI >= 1 && TJ >= 1, "tile too small");
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // per-tile indices: nothing hoisted across the caller's tile loop
    const int lane = tid & 63, wv = tid >> 6;
    const int wi = wv >> 1, wj = wv & 1;
    const int lr = lane & 15, lk = lane >> 4;
    v4d acc[TI][TJ];
#pragma unroll
    for (int a = 0; a < TI; ++a)
#pragma unroll
        for (int b = 0; b < TJ; ++b) acc[a][b] = (v4d){0.0, 0.0, 0.0, 0.0};
    bool rin[TI], cin[TJ];  // this wave's 16 x 16 sub-tiles that intersect C
#pragma unroll
    for (int a = 0; a < TI; ++a) rin[a] = m0 + wi * (BM / 2) + a * 16 < m;
#pragma unroll
    for (int b = 0; b < TJ; ++b) cin[b] = n0 + wj * (BN / 2) + b * 16 < n;
    double ra[LA], rb[LB];
    auto load = [&](int k0) {
#pragma unroll
        for (int r = 0; r < LA; ++r) {
            const int e = tid + GEMM_THREADS * r;
            const int i = e / BK, kk = e % BK;
            const int gi = m0 + i, gk = k0 + kk;
            ra[r] = (gi < m && gk < k) ? A[(int64_t)gi * lda + gk] : 0.0;
        }
#pragma unroll
        for (int r = 0; r < LB; ++r) {
            const int e = tid + GEMM_THREADS * r;
            const int kk = e / BN, j = e % BN;
            const int gk = k0 + kk, gj = n0 + j;
            rb[r] = (gk < k && gj < n) ? B[(int64_t)gk * ldb + gj] : 0.0;
        }
    };
    load(0);
    for (int k0 = 0; k0 < k; k0 += BK) {
        __syncthreads();  // the previous step's fragment reads are done
#pragma unroll
        for (int r = 0; r < LA; ++r) {
            const int e = tid + GEMM_THREADS * r;
            sA[(e % BK) * SA + e / BK] = ra[r];
        }
#pragma unroll
        for (int r = 0; r < LB; ++r) {
            const int e = tid + GEMM_THREADS * r;
            sB[(e / BN) * SB + e % BN] = rb[r];
        }
        __syncthreads();
        if (k0 + BK < k) load(k0 + BK);  // prefetch overlaps the MFMAs
        // MFMAs whose operands are all zero padding are skipped: K steps of 4
        // past k, and 16 x 16 sub-tiles wholly outside C (never stored).  All
        // conditions are wave-uniform; a skipped step would add exact zeros.
#pragma unroll
        for (int s = 0; s < BK / 4; ++s) {
            if (k0 + 4 * s < k) {
                const int kk = 4 * s + lk;
                double af[TI], bf[TJ];
#pragma unroll
                for (int a = 0; a < TI; ++a) af[a] = sA[kk * SA + wi * (BM / 2) + a * 16 + lr];
#pragma unroll
                for (int b = 0; b < TJ; ++b) bf[b] = sB[kk * SB + wj * (BN / 2) + b * 16 + lr];
#pragma unroll
                for (int a = 0; a < TI; ++a)
#pragma unroll
                    for (int b = 0; b < TJ; ++b)
                        if (rin[a] && cin[b]) acc[a][b] = mfma16(af[a], bf[b], acc[a][b]);
            }
        }
    }
#pragma unroll
    for (int a = 0; a < TI; ++a)
#pragma unroll
        for (int b = 0; b < TJ; ++b) {
            const int gj = n0 + wj * (BN / 2) + b * 16 + lr;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gi = m0 + wi * (BM / 2) + a * 16 + 4 * r + lk;
                if (gi < m && gj < n) C[(int64_t)gi * ldc + gj] = acc[a][b][r];
            }
        }
}

// Contractions with a matrix of even and odd functions on symmetric nodes
// (phi_k(-x) = (-1)^k phi_k(x): the Legendre and Chebyshev bases with even
// stencils; cos and sin on the periodic grid), at half the products of the
// plain form: even outputs need the even part of the data only, odd ones the
// odd part.
//   FOLD_ROWS_IN   C[2i+p][n] = sum_{j < X/2} A[2i+p][j] (B[j][n] +- B[X-1-j][n])
//                  (analysis; A M x X, B X x N)
//   FOLD_COLS_IN   C[m][2i+p] = sum_{j <= Y/2} (A[m][j] +- A[m][Y-j]) B[j][2i+p]
//                  (real DFT, columns (re, im) pairs; A M x Y, B Y x (Y+2))
//   FOLD_ROWS_OUT  C[j], C[X-1-j] = E +- O, E, O = sum_i A[j][2i+p] B[2i+p]
//                  (synthesis; A X x M, B M x N)
//   FOLD_COLS_OUT  C[m][j], C[m][Y-j] = E +- O, E, O = sum_i A[m][2i+p] B[2i+p][j]
//                  (inverse real DFT; A M x (Y+2), B (Y+2) x Y)
// A data value that is its own mirror image goes to the even part.  Both
// parities of a BMU x BNU tile (units: rows or columns come in pairs on the
// folded side) are accumulated by the same wave, each output as one MFMA chain
// over K in ascending order, whatever the tile.
enum FoldMode { FOLD_ROWS_IN = 0, FOLD_COLS_IN = 1, FOLD_ROWS_OUT = 2, FOLD_COLS_OUT = 3 };

template <int BMU, int BNU>
struct FoldShape {
    static constexpr int WI = BNU == 16 ? 4 : (BMU >= 32 ? 2 : 1), WJ = 4 / WI;  // waves
    static constexpr int TI = BMU / (16 * WI), TJ = BNU / (16 * WJ);             // 16 x 16 tiles of a wave
    static_assert(TI >= 1 && TJ >= 1, "tile too small for four waves");
    static constexpr int SA = BMU + 1, SB = BNU;  // LDS row pitches
    template <int BK>
    static constexpr int lds_a() { return 2 * BK * SA; }
    template <int BK>
    static constexpr int lds_b() { return 2 * BK * SB; }
};

// m x n: the matrix C as a whole; k: the contracted length (X, Y or M); mu0,
// nu0: the tile's first unit row and column.
template <int MODE, int BMU, int BNU, int BK>
__device__ void fold_tile(const double* __restrict__ A, int64_t lda, const double* __restrict__ B, int64_t ldb,
                          double* __restrict__ C, int64_t ldc, int m, int n, int k, int mu0, int nu0, double* sA,
                          double* sB)
{
    using Sh = FoldShape<BMU, BNU>;
    constexpr int SA = Sh::SA, SB = Sh::SB, TI = Sh::TI, TJ = Sh::TJ;
    constexpr int LA = BMU * BK / GEMM_THREADS, LB = BK * BNU / GEMM_THREADS;
    static_assert(LA >= 1 && LB >= 1, "tile too small");
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // per-tile indices: nothing hoisted across the caller's tile loop
    const int lane = tid & 63, wv = tid >> 6;
    const int wi = wv / Sh::WJ, wj = wv % Sh::WJ;
    const int lr = lane & 15, lk = lane >> 4;
    // units: C's rows and columns (pairs on the folded side), K's steps
    const int mu = MODE == FOLD_ROWS_IN || MODE == FOLD_ROWS_OUT ? (m + 1) / 2 : m;
    const int nu = MODE == FOLD_COLS_IN ? n / 2 : (MODE == FOLD_COLS_OUT ? n / 2 + 1 : n);
    const int ku = MODE == FOLD_COLS_IN ? k / 2 + 1 : (k + 1) / 2;
    v4d acc[2][TI][TJ];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int a = 0; a < TI; ++a)
#pragma unroll
            for (int b = 0; b < TJ; ++b) acc[p][a][b] = (v4d){0.0, 0.0, 0.0, 0.0};
    bool rin[TI], cin[TJ];
#pragma unroll
    for (int a = 0; a < TI; ++a) rin[a] = mu0 + (wi * TI + a) * 16 < mu;
#pragma unroll
    for (int b = 0; b < TJ; ++b) cin[b] = nu0 + (wj * TJ + b) * 16 < nu;
    // the two parities' operands, or a data value and its mirror image (summed
    // when they are stored to LDS: not here, where it would wait for the loads)
    double ra[LA][2], rb[LB][2];
    // Inner steps (all of their units inside K, none its own mirror image) load
    // from pointers that advance by a constant; the others from clamped indices
    // with a select.  No load sits under a branch of its own.  (Indices and
    // clamps in every step cost as much as its MFMAs: leg. 512 x 512 on 258
    // columns 22.6 us a product.)
    const double *pa[LA], *pb[LB], *qb[MODE == FOLD_ROWS_IN ? LB : 1];
    int64_t sa1[LA];  // the odd partner of an A value (FOLD_ROWS_IN: a row on; FOLD_COLS_IN: its mirror image)
#pragma unroll
    for (int r = 0; r < LA; ++r) {
        const int e = tid + GEMM_THREADS * r;
        const int gi = mu0 + e / BK, kk = e % BK, ci = gi < mu ? gi : mu - 1;
        if constexpr (MODE == FOLD_ROWS_IN) {
            pa[r] = A + (int64_t)(2 * ci) * lda + kk;
            sa1[r] = 2 * ci + 1 < m ? lda : 0;
        } else if constexpr (MODE == FOLD_COLS_IN) {
            pa[r] = A + (int64_t)ci * lda + kk;
            sa1[r] = k - 2 * kk;
        } else {
            pa[r] = A + (int64_t)ci * lda + 2 * kk;
            sa1[r] = 1;
        }
    }
#pragma unroll
    for (int r = 0; r < LB; ++r) {
        const int e = tid + GEMM_THREADS * r;
        const int kk = e / BNU, gj = nu0 + e % BNU, cj = gj < nu ? gj : nu - 1;
        if constexpr (MODE == FOLD_ROWS_IN) {
            pb[r] = B + (int64_t)kk * ldb + cj;
            qb[r] = B + (int64_t)(k - 1 - kk) * ldb + cj;
        } else if constexpr (MODE == FOLD_COLS_IN) {
            pb[r] = B + (int64_t)kk * ldb + 2 * cj;
        } else {
            pb[r] = B + (int64_t)(2 * kk) * ldb + cj;
        }
    }
    const int64_t bstep = (MODE == FOLD_ROWS_OUT || MODE == FOLD_COLS_OUT ? 2 * BK : BK) * ldb;
    auto advance = [&]() {
#pragma unroll
        for (int r = 0; r < LA; ++r) {
            pa[r] += MODE == FOLD_ROWS_OUT || MODE == FOLD_COLS_OUT ? 2 * BK : BK;
            if (MODE == FOLD_COLS_IN) sa1[r] -= 2 * BK;
        }
#pragma unroll
        for (int r = 0; r < LB; ++r) {
            pb[r] += bstep;
            if (MODE == FOLD_ROWS_IN) qb[r] -= bstep;
        }
    };
    auto load_inner = [&]() {
#pragma unroll
        for (int r = 0; r < LA; ++r) {
            const double v = pa[r][0], w = pa[r][sa1[r]];
            ra[r][0] = v;
            ra[r][1] = w;
        }
#pragma unroll
        for (int r = 0; r < LB; ++r) {
            const double v = pb[r][0];
            const double w = MODE == FOLD_ROWS_IN ? qb[r][0] : MODE == FOLD_COLS_IN ? pb[r][1] : pb[r][ldb];
            rb[r][0] = v;
            rb[r][1] = w;
        }
    };
    auto load_edge = [&](int k0) {
#pragma unroll
        for (int r = 0; r < LA; ++r) {
            const int e = tid + GEMM_THREADS * r;
            const int gi = mu0 + e / BK, gk = k0 + e % BK;
            const int ci = gi < mu ? gi : mu - 1, ck = gk < ku ? gk : ku - 1;
            const bool in = gi < mu && gk < ku;
            if constexpr (MODE == FOLD_ROWS_IN) {
                const bool in1 = in && 2 * gi + 1 < m;
                const double* q = A + (int64_t)(2 * ci) * lda + ck;
                const double v0 = q[0], v1 = q[2 * ci + 1 < m ? lda : 0];
                ra[r][0] = in ? v0 : 0.0;
                ra[r][1] = in1 ? v1 : 0.0;
            } else if constexpr (MODE == FOLD_COLS_IN) {
                const bool self = ck == 0 || 2 * ck == k;
                const double* q = A + (int64_t)ci * lda;
                const double v = q[ck], w = q[self ? ck : k - ck];
                const double f = self ? 0.5 : 1.0;  // its own mirror image: v to the sum, 0 to the difference
                ra[r][0] = in ? f * v : 0.0;
                ra[r][1] = in ? f * w : 0.0;
            } else {
                const bool in1 = in && 2 * gk + 1 < k;
                const double* q = A + (int64_t)ci * lda + 2 * ck;
                const double v0 = q[0], v1 = q[2 * ck + 1 < k ? 1 : 0];
                ra[r][0] = in ? v0 : 0.0;
                ra[r][1] = in1 ? v1 : 0.0;
            }
        }
#pragma unroll
        for (int r = 0; r < LB; ++r) {
            const int e = tid + GEMM_THREADS * r;
            const int gk = k0 + e / BNU, gj = nu0 + e % BNU;
            const int ck = gk < ku ? gk : ku - 1, cj = gj < nu ? gj : nu - 1;
            const bool in = gk < ku && gj < nu;
            if constexpr (MODE == FOLD_ROWS_IN) {
                const bool self = 2 * ck == k - 1;
                const double v = B[(int64_t)ck * ldb + cj], w = B[(int64_t)(k - 1 - ck) * ldb + cj];
                const double f = self ? 0.5 : 1.0;
                rb[r][0] = in ? f * v : 0.0;
                rb[r][1] = in ? f * w : 0.0;
            } else if constexpr (MODE == FOLD_COLS_IN) {
                const double* q = B + (int64_t)ck * ldb + 2 * cj;
                const double v0 = q[0], v1 = q[1];
                rb[r][0] = in ? v0 : 0.0;
                rb[r][1] = in ? v1 : 0.0;
            } else {
                const bool in1 = in && 2 * gk + 1 < k;
                const double* q = B + (int64_t)(2 * ck) * ldb + cj;
                const double v0 = q[0], v1 = q[2 * ck + 1 < k ? ldb : 0];
                rb[r][0] = in ? v0 : 0.0;
                rb[r][1] = in1 ? v1 : 0.0;
            }
        }
    };
    auto load = [&](int k0) {  // k0 ascending from 0 by BK
        if (k0 + BK < ku && (MODE != FOLD_COLS_IN || k0 > 0)) load_inner();
        else load_edge(k0);
        advance();
    };
    load(0);
    for (int k0 = 0; k0 < ku; k0 += BK) {
        __syncthreads();  // the previous step's fragment reads are done
#pragma unroll
        for (int r = 0; r < LA; ++r) {
            const int e = tid + GEMM_THREADS * r;
            const double v = ra[r][0], w = ra[r][1];
            sA[(e % BK) * SA + e / BK] = MODE == FOLD_COLS_IN ? v + w : v;
            sA[(BK + e % BK) * SA + e / BK] = MODE == FOLD_COLS_IN ? v - w : w;
        }
#pragma unroll
        for (int r = 0; r < LB; ++r) {
            const int e = tid + GEMM_THREADS * r;
            const double v = rb[r][0], w = rb[r][1];
            sB[(e / BNU) * SB + e % BNU] = MODE == FOLD_ROWS_IN ? v + w : v;
            sB[(BK + e / BNU) * SB + e % BNU] = MODE == FOLD_ROWS_IN ? v - w : w;
        }
        __syncthreads();
        if (k0 + BK < ku) load(k0 + BK);  // overlaps the MFMAs
#pragma unroll
        for (int s = 0; s < BK / 4; ++s) {
            if (k0 + 4 * s < ku) {  // wave-uniform; a skipped step would add exact zeros
                const int kk = 4 * s + lk;
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    double af[TI], bf[TJ];
#pragma unroll
                    for (int a = 0; a < TI; ++a) af[a] = sA[(p * BK + kk) * SA + (wi * TI + a) * 16 + lr];
#pragma unroll
                    for (int b = 0; b < TJ; ++b) bf[b] = sB[(p * BK + kk) * SB + (wj * TJ + b) * 16 + lr];
#pragma unroll
                    for (int a = 0; a < TI; ++a)
#pragma unroll
                        for (int b = 0; b < TJ; ++b)
                            if (rin[a] && cin[b]) acc[p][a][b] = mfma16(af[a], bf[b], acc[p][a][b]);
                }
            }
        }
    }
#pragma unroll
    for (int a = 0; a < TI; ++a)
#pragma unroll
        for (int b = 0; b < TJ; ++b) {
            const int gj = nu0 + (wj * TJ + b) * 16 + lr;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gi = mu0 + (wi * TI + a) * 16 + 4 * r + lk;
                if (gi >= mu || gj >= nu) continue;
                const double e = acc[0][a][b][r], o = acc[1][a][b][r];
                if constexpr (MODE == FOLD_ROWS_IN) {
                    C[(int64_t)(2 * gi) * ldc + gj] = e;
                    if (2 * gi + 1 < m) C[(int64_t)(2 * gi + 1) * ldc + gj] = o;
                } else if constexpr (MODE == FOLD_COLS_IN) {
                    C[(int64_t)gi * ldc + 2 * gj] = e;
                    C[(int64_t)gi * ldc + 2 * gj + 1] = o;
                } else if constexpr (MODE == FOLD_ROWS_OUT) {
                    C[(int64_t)gi * ldc + gj] = e + o;
                    if (2 * gi != m - 1) C[(int64_t)(m - 1 - gi) * ldc + gj] = e - o;
                } else {
                    C[(int64_t)gi * ldc + gj] = e + o;
                    if (gj != 0 && 2 * gj != n) C[(int64_t)gi * ldc + n - gj] = e - o;
                }
            }
        }
}

}  // namespace sfa

// Per-line operations of the transforms and their mixed-radix kernel.
#pragma once
#include "fft_mixed.h"

namespace sfa {

// OP_DCT1F / OP_DCT1B: Chebyshev-Gauss-Lobatto scalar product / backward via
// DCT-I (REDFT00) of length n, computed as the complex FFT of the line's even
// extension (length 2(n-1)): the sine terms cancel, so the first n outputs
// are the DCT-I of the real and imaginary parts at once.
// OP_R2CF / OP_C2RF: odd-length R2C / C2R as a full-length complex FFT (real
// input widened; Hermitian spectrum completed on load), the even lengths pack
// pairs of reals instead (OP_R2C / OP_C2R)
enum LineOp {
    OP_C2C = 0, OP_R2C = 1, OP_C2R = 2, OP_DCT2 = 3, OP_DCT3 = 4, OP_DCT1F = 5, OP_DCT1B = 6,
    OP_R2CF = 7, OP_C2RF = 8
};

struct LineArgs {
    const char* in;
    char* out;
    int64_t in_sa, in_s1, in_s2;
    int64_t out_sa, out_s1, out_s2;
    int64_t d1, d2;
    int n;      // logical length along the axis (real length for R2C/C2R)
    int ldn;    // LDS line stride (complex elements)
    int T;      // lines per block
    int in_cplx, out_cplx;
    int t_fast_in, t_fast_out;
    int inv;    // C2C direction
    double scale;
    const double* K2;
    const double2* tw;   // FFT table of length plan.nfft
    const double2* tw2;  // R2C/C2R: table of length n; DCT: quarter table of length n
    FFTPlan plan;
};

// ----------------------------------------------------------------- mixed-radix lines
// The same operations for lengths whose prime factors are at most 13, on the
// in-place passes of fft_mixed.h: the first pass reads global memory itself
// (with the operation's permutation, symmetric extension or pre-twiddle; an
// element that two butterflies need is read twice, from L1), the last one
// writes it, and only the operations that combine outputs k and n - k (R2C,
// DCT-II) or k and k + 2 (a stencil) go through LDS once more.
struct MixArgs {
    const char* in;
    char* out;
    int64_t in_sa, in_s1, in_s2;
    int64_t out_sa, out_s1, out_s2;
    int64_t d1, d2;
    int n;
    int T, shift, t_fast;
    double scale;
    const double* K2;
    const double2* tw;   // FFT table of the plan's length
    const double2* tw2;  // R2C/C2R: table of length n; DCT-II/III: quarter table
    MixPlan plan;
};

template <bool CPLX>
__device__ __forceinline__ double2 mix_ld(const char* base, int64_t off)
{
    if (CPLX) return reinterpret_cast<const double2*>(base)[off];
    return make_double2(reinterpret_cast<const double*>(base)[off], 0.0);
}

template <bool CPLX>
__device__ __forceinline__ void mix_st(char* base, int64_t off, double2 v)
{
    if (CPLX) reinterpret_cast<double2*>(base)[off] = v;
    else reinterpret_cast<double*>(base)[off] = v.x;
}

// This thread's (line, index) pairs of the tile, four at a time: get(t, k, i)
// of all four before put(t, k, i) of the first, so that their loads are in
// flight together (get of an absent pair reads the tile's first).
template <class G, class P>
__device__ __forceinline__ void four_at_a_time(const MixTile& m, int len, int tid, int nth, G get, P put)
{
    MixIter it(m, len, tid, nth);
    while (!it.done()) {
        int t[4], k[4];
        bool ok[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            ok[i] = it.here();
            t[i] = ok[i] ? it.t : 0;
            k[i] = ok[i] ? it.k : 0;
            it.next();
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) get(t[i], k[i], i);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (ok[i]) put(t[i], k[i], i);
    }
}

// COMP: composite basis (the stencil K2) in the Chebyshev operations
template <int OP, bool INV, bool CPLX, bool COMP>
__global__ void __launch_bounds__(256) mix_kernel(MixArgs a)
{
    const int tid = threadIdx.x, nth = blockDim.x;
    const int64_t ntile = (a.d2 + a.T - 1) / a.T;
    const int64_t blk = wide_block(), i1 = blk / ntile;
    if (i1 >= a.d1) return;
    const int64_t t0 = (blk - i1 * ntile) * a.T;
    const MixPlan& pl = a.plan;
    MixTile m;
    m.T = a.T;
    m.Tv = (int)((a.d2 - t0) < a.T ? (a.d2 - t0) : a.T);
    m.shift = a.shift;
    m.t_fast = a.t_fast != 0;
    m.ps = m.t_fast ? a.T : 1;
    m.ts = m.t_fast ? 1 : pl.size();
    const int buf = 0, twT = a.T * pl.size();
    const int ends = twT + pl.n;  // 2 T: first and last value of each line (DCT-III, DCT-I backward)
    const int64_t is2 = a.in_s2, isa = a.in_sa, os2 = a.out_s2, osa = a.out_sa;
    const int64_t ib = i1 * a.in_s1 + t0 * is2, ob = i1 * a.out_s1 + t0 * os2;
    // bases in elements of the arrays' own types
    constexpr bool IC2 = CPLX || OP == OP_C2RF || OP == OP_C2R;  // complex input
    constexpr bool OC2 = (CPLX && OP != OP_C2R) || OP == OP_R2CF || OP == OP_R2C;
    const char* inb = a.in + ib * (IC2 ? 16 : 8);
    char* outb = a.out + ob * (OC2 ? 16 : 8);
    const int n = a.n;
    const double sc = a.scale;
    const double* K2 = a.K2;
    auto ild = [&](int t, int i) { return mix_ld<IC2>(inb, t * is2 + i * isa); };
    auto ost = [&](int64_t off, double2 v) { mix_st<OC2>(outb, off, v); };
    // composite input in the orthogonal basis: u_k (k < n - 2) + K2_{k-2} u_{k-2},
    // read without a branch
    auto ortho = [&](int t, int k) {
        if constexpr (!COMP) return ild(t, k);
        const double2 v = ild(t, k < n - 2 ? k : n - 3), u = ild(t, k >= 2 ? k - 2 : 0);
        const double kk = k >= 2 ? K2[k - 2] : 0.0, on = k < n - 2 ? 1.0 : 0.0;
        return make_double2(on * v.x + kk * u.x, on * v.y + kk * u.y);
    };
    const int nb0 = pl.sub[0];
    const float inv_nb0 = 1.0f / (float)nb0;
    auto in_put = [&](int t, int i, double2 v) { lds_put(buf + mix_in_pos(pl, i, inv_nb0) * m.ps + t * m.ts, v); };

    mix_twiddles(pl, twT, a.tw, tid, nth);
    constexpr bool STAGED = OP == OP_DCT3 || OP == OP_DCT1B;
    if constexpr (OP == OP_DCT3) {
        // V[k] = exp(+i pi k/(2N)) ((a_k + b_{N-k}) + i (b_k - a_{N-k})), a_N = b_N = 0:
        // k and N - k from the same two coefficients
        const int np2 = n / 2 + 1;
        double2 ck[4], cn[4];
        four_at_a_time(m, np2, tid, nth,
            [&](int t, int k, int i) {
                ck[i] = ortho(t, k);
                cn[i] = ortho(t, k == 0 ? 0 : n - k);
            },
            [&](int t, int k, int i) {
                if (k == 0) {
                    lds_put(ends + 2 * t, ck[i]);
                    in_put(t, 0, ck[i]);
                    return;
                }
                const double2 w = cconj(a.tw2[k]), wn = cconj(a.tw2[n - k]);
                in_put(t, k, cmul(w, make_double2(ck[i].x + cn[i].y, ck[i].y - cn[i].x)));
                if (2 * k != n) in_put(t, n - k, cmul(wn, make_double2(cn[i].x + ck[i].y, cn[i].y - ck[i].x)));
            });
    }
    if constexpr (OP == OP_DCT1B) {  // the even extension
        double2 c[4];
        four_at_a_time(m, n, tid, nth,
            [&](int t, int k, int i) {
                c[i] = ortho(t, k);
            },
            [&](int t, int k, int i) {
                in_put(t, k, c[i]);
                if (k > 0 && k < n - 1) in_put(t, 2 * (n - 1) - k, c[i]);
                if (k == 0) lds_put(ends + 2 * t, c[i]);
                if (k == n - 1) lds_put(ends + 2 * t + 1, c[i]);
            });
    }
    if (STAGED) __syncthreads();

    // where input j of line t lies, how far apart neighbours are, input i
    constexpr int W = OP == OP_R2C ? 2 : 1;
    auto lb = [&](int t, int j) -> int64_t {
        if constexpr (STAGED) return buf + j * m.ps + t * m.ts;
        else return t * is2 + W * j * isa;
    };
    auto load = [&](int64_t o, int t, int i) -> double2 {
        if constexpr (STAGED) {
            return lds_get((int)o);
        } else if constexpr (OP == OP_C2C || OP == OP_R2CF) {
            return mix_ld<IC2>(inb, o);
        } else if constexpr (OP == OP_R2C) {
            const double* p = reinterpret_cast<const double*>(inb) + o;
            return make_double2(p[0], p[isa]);
        } else if constexpr (OP == OP_C2RF) {
            // X_k for k <= n/2 from the input, X_{n-k} = conj(X_k) above; Im X_0 dropped
            const bool up = i > n / 2;
            const double2 v = ild(t, up ? n - i : i);
            return make_double2(v.x, i == 0 ? 0.0 : (up ? -v.y : v.y));
        } else if constexpr (OP == OP_C2R) {
            double2 xk = mix_ld<true>(inb, o);
            double2 xc = cconj(ild(t, n / 2 - i));
            if (i == 0) xk.y = xc.y = 0.0;
            const double2 d = cmul(cconj(a.tw2[i]), csub(xk, xc));  // exp(+2 pi i k / n) (..)
            return make_double2(xk.x + xc.x - d.y, xk.y + xc.y + d.x);
        } else if constexpr (OP == OP_DCT2) {
            return ild(t, 2 * i < n ? 2 * i : 2 * (n - 1 - i) + 1);
        } else {  // OP_DCT1F
            return ild(t, i < n ? i : 2 * (n - 1) - i);
        }
    };
    constexpr int WO = OP == OP_C2R ? 2 : 1;
    auto sb = [&](int t, int k) -> int64_t { return t * os2 + WO * k * osa; };
    auto store = [&](int64_t o, int t, int k, int pos, double2 v) {
        if constexpr (OP == OP_C2C || OP == OP_C2RF) {
            ost(o, cscale(v, sc));
        } else if constexpr (OP == OP_R2CF) {
            if (k <= n / 2) ost(o, cscale(v, sc));
        } else if constexpr (OP == OP_C2R) {
            double* p = reinterpret_cast<double*>(outb) + o;
            p[0] = v.x * sc;
            p[osa] = v.y * sc;
        } else if constexpr (OP == OP_DCT3) {
            const double2 c0 = lds_get(ends + 2 * t);
            ost(t * os2 + (2 * k < n ? 2 * k : 2 * (n - 1 - k) + 1) * osa,
                make_double2((0.5 * v.x + 0.5 * c0.x) * sc, (0.5 * v.y + 0.5 * c0.y) * sc));
        } else if constexpr (OP == OP_DCT1B) {
            // u_j = 0.5 Y_j + 0.5 t_0 + 0.5 (-1)^j t_{n-1}
            if (k < n) {
                const double2 c0 = lds_get(ends + 2 * t), c1 = lds_get(ends + 2 * t + 1);
                const double sg = (k & 1) ? -0.5 : 0.5;
                ost(o, make_double2((0.5 * v.x + 0.5 * c0.x + sg * c1.x) * sc,
                                                     (0.5 * v.y + 0.5 * c0.y + sg * c1.y) * sc));
            }
        } else {
            lds_put(buf + pos * m.ps + t * m.ts, v);
        }
    };
    mix_first<INV>(pl, m, buf, twT, tid, nth, lb, STAGED ? (int64_t)pl.P * m.ps : W * isa * nb0, load, sb, WO * osa, store);
    mix_rest<INV>(pl, m, buf, a.tw, tid, nth, sb, WO * osa, store);

    auto at = [&](int t, int k) { return buf + mix_pos(pl, k) * m.ps + t * m.ts; };
    if constexpr (OP == OP_R2C) {
        // X_k = 0.5 (Z_k + conj Z_{h-k}) - 0.5 i w_k (Z_k - conj Z_{h-k}), w_k = exp(-2 pi i k/n):
        // k and h - k from the same two values
        __syncthreads();
        const int h = n / 2, np2 = h / 2 + 1;
        double2 zk[4], zc[4], w[4], wn[4];
        four_at_a_time(m, np2, tid, nth,
            [&](int t, int k, int i) {
                zk[i] = lds_get(at(t, k));
                zc[i] = lds_get(at(t, k == 0 ? 0 : h - k));
                w[i] = a.tw2[k];
                wn[i] = a.tw2[h - k];
            },
            [&](int t, int k, int i) {
                auto X = [&](double2 z, double2 zz, double2 ww) {
                    const double2 c = cconj(zz), d = cmul(ww, csub(z, c));
                    return make_double2(0.5 * (z.x + c.x + d.y) * sc, 0.5 * (z.y + c.y - d.x) * sc);
                };
                ost(t * os2 + k * osa, X(zk[i], zc[i], w[i]));
                if (2 * k != h) ost(t * os2 + (h - k) * osa, X(zc[i], zk[i], wn[i]));
            });
    }
    if constexpr (OP == OP_DCT2) {
        // X_k = Re(w (P + Q)) + i Im(w (P - Q)), P = V_k, Q = conj(V_{N-k}): k and
        // N - k from the same two values, in place where a stencil follows
        __syncthreads();
        const int np2 = n / 2 + 1;
        double2 vk[4], vn[4], w[4], wn[4];
        four_at_a_time(m, np2, tid, nth,
            [&](int t, int k, int i) {
                vk[i] = lds_get(at(t, k));
                vn[i] = lds_get(at(t, k == 0 ? 0 : n - k));
                w[i] = a.tw2[k];
                wn[i] = a.tw2[k == 0 ? 0 : n - k];
            },
            [&](int t, int k, int i) {
                auto X = [&](double2 P, double2 V, double2 ww) {
                    const double2 Q = cconj(V);
                    return make_double2(cmul(ww, cadd(P, Q)).x * sc, cmul(ww, csub(P, Q)).y * sc);
                };
                const double2 x = X(vk[i], vn[i], w[i]);
                const bool two = k > 0 && 2 * k != n;
                const double2 y = X(vn[i], vk[i], wn[i]);
                if constexpr (COMP) {
                    lds_put(at(t, k), x);
                    if (two) lds_put(at(t, n - k), y);
                } else {
                    ost(t * os2 + k * osa, x);
                    if (two) ost(t * os2 + (n - k) * osa, y);
                }
            });
    }
    if constexpr ((OP == OP_DCT2 && COMP) || OP == OP_DCT1F) {
        // stencil s_k + K2_k s_{k+2} (k < n - 2); DCT-I: s_k = sc Y_k
        __syncthreads();
        double2 v[4], u[4];
        double kk[4];
        four_at_a_time(m, n, tid, nth,
            [&](int t, int k, int i) {
                v[i] = lds_get(at(t, k));
                if constexpr (COMP) {
                    u[i] = lds_get(at(t, k < n - 2 ? k + 2 : k));
                    kk[i] = k < n - 2 ? K2[k] : 0.0;
                }
            },
            [&](int t, int k, int i) {
                double2 x = v[i];
                if constexpr (OP == OP_DCT1F) x = cscale(x, sc);
                if constexpr (COMP) {
                    if (k < n - 2) {
                        const double q = OP == OP_DCT1F ? kk[i] * sc : kk[i];
                        x.x += q * u[i].x;
                        x.y += q * u[i].y;
                    }
                }
                ost(t * os2 + k * osa, x);
            });
    }
}

// Arguments of the mixed-radix form; false where the length does not allow it.
// T lines per workgroup: at most 16 (256-byte row segments where lanes run over
// lines) and 76 KB of LDS, which keeps two workgroups on a compute unit
// (240 x 129 lines, 256 x 240 x 129 complex along axis 1: T = 16 55.5 us, T = 8
// 72.6), fewer while the launch has under 512 workgroups, but not below the 8
// that make a segment one 128-byte line.  Against the double-buffered Stockham
// form it replaces (a division per element, two LDS copies beside the passes;
// microseconds, complex along axis 1): 180 x 150 x 101 48.6 -> 22.1, 100^3
// 15.8 -> 8.9, 64 x 360 x 64 33.3 -> 13.7; R2C 180 x 150 x 200 42.2 -> 24.3,
// 256 x 256 x 240 98.0 -> 51.7; DCT-II / DCT-III with stencil along axis 0
// 192 x 96 x 81 34.2 / 38.1 -> 19.4 / 16.6, 256 x 256 x 129 162 / 186 -> 94 / 80.
// Lanes run as the input's layout wants it.  An output laid out the other way is
// stored in pieces of one element per line, at up to a third more than one laid
// out like it (complex, 64 lines x 240 x 65 and back: 12.3 and 11.5 us, contiguous
// to contiguous 8.9; the form above, which staged it in LDS, 24.7, 24.2 and 21.0).
inline bool mix_setup(const LineArgs& la, MixArgs& a, dim3* grid, unsigned* block, size_t* lds_bytes,
                      int most = 16)
{
    const int nf = la.plan.nfft;
    int64_t d1 = la.d1, d2 = la.d2;
    auto absl = [](int64_t v) { return v < 0 ? -v : v; };
    // lines whose two dimensions are one in both arrays
    const bool flat = d1 > 1 && la.in_s1 == d2 * la.in_s2 && la.out_s1 == d2 * la.out_s2;
    if (flat) {
        d2 *= d1;
        d1 = 1;
    }
    a.t_fast = (absl(la.in_s2) < absl(la.in_sa) && d2 > 1) ? 1 : 0;
    if (!make_mix_plan(nf, !a.t_fast, &a.plan)) return false;
    const int64_t line = (int64_t)a.plan.size() * sizeof(double2);
    const int64_t table = (int64_t)nf * sizeof(double2);
    int T = most;  // lines at most
    while (T > 1 && T * line + table > 76 * 1024) T >>= 1;
    while (T > 1 && T >= 2 * d2) T >>= 1;
    while (T > 8 && d1 * ((d2 + T - 1) / T) < 512) T >>= 1;
    a.T = T;
    a.shift = 0;
    while ((1 << a.shift) < T) ++a.shift;
    a.in = la.in;
    a.out = la.out;
    a.in_sa = la.in_sa;
    a.in_s1 = la.in_s1;
    a.in_s2 = la.in_s2;
    a.out_sa = la.out_sa;
    a.out_s1 = la.out_s1;
    a.out_s2 = la.out_s2;
    a.d1 = d1;
    a.d2 = d2;
    a.n = la.n;
    a.scale = la.scale;
    a.K2 = la.K2;
    a.tw = la.tw;
    a.tw2 = la.tw2;
    const size_t lds = (size_t)(T * line + table) + (size_t)2 * T * sizeof(double2);
    if (lds > 160 * 1024) return false;
    const int64_t nblk = d1 * ((d2 + T - 1) / T);
    // a thread per butterfly of the pass that has the most, at most 256; all 256
    // where the workgroups are few, for the steps that go over elements
    int rmin = kMixMaxRadix;
    for (int l = 0; l < a.plan.np; ++l) rmin = a.plan.r[l] < rmin ? a.plan.r[l] : rmin;
    const int64_t nbf = (int64_t)T * nf / rmin;
    *block = nbf >= 256 || nblk < 64 ? 256u : (unsigned)((nbf + 63) / 64 * 64);
    *grid = wide_grid(nblk);
    *lds_bytes = lds;
    return true;
}

template <int OP, bool INV, bool CPLX, bool COMP = false>
int mix_run(const MixArgs& a, dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    auto kfn = mix_kernel<OP, INV, CPLX, COMP>;
    if (lds > 64 * 1024)
        SFA_HIP(hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kfn, grid, block, lds, stream, a);
    SFA_LAUNCH_CHECK();
    return SFA_OK;
}

// one translation unit per group of operations (each holds a body per radix
// and pass)
int mix_run_fft(int op, bool inv, const MixArgs& a, dim3 grid, dim3 block, size_t lds, hipStream_t stream);
int mix_run_real(int op, const MixArgs& a, dim3 grid, dim3 block, size_t lds, hipStream_t stream);
int mix_run_dct2(bool cplx, const MixArgs& a, dim3 grid, dim3 block, size_t lds, hipStream_t stream);
int mix_run_dct3(bool cplx, const MixArgs& a, dim3 grid, dim3 block, size_t lds, hipStream_t stream);
int mix_run_dct1f(bool cplx, const MixArgs& a, dim3 grid, dim3 block, size_t lds, hipStream_t stream);
int mix_run_dct1b(bool cplx, const MixArgs& a, dim3 grid, dim3 block, size_t lds, hipStream_t stream);

// mix_blue.hip: lengths with larger prime factors, up to 2048
bool blue_launch(int op, bool inv, const LineArgs& la, hipStream_t stream, int* rc);

// Launch the mixed-radix form where the length allows it.
inline bool mix_launch(int op, bool inv, const LineArgs& la, hipStream_t stream, int* rc)
{
    MixArgs a;
    dim3 grid;
    unsigned block;
    size_t lds;
    if (!mix_setup(la, a, &grid, &block, &lds)) return blue_launch(op, inv, la, stream, rc);
    const bool c = la.in_cplx != 0;
    switch (op) {
        case OP_C2C: *rc = mix_run_fft(op, inv, a, grid, block, lds, stream); break;
        case OP_R2CF:
        case OP_C2RF:
        case OP_R2C:
        case OP_C2R: *rc = mix_run_real(op, a, grid, block, lds, stream); break;
        case OP_DCT2: *rc = mix_run_dct2(c, a, grid, block, lds, stream); break;
        case OP_DCT3: *rc = mix_run_dct3(c, a, grid, block, lds, stream); break;
        case OP_DCT1F: *rc = mix_run_dct1f(c, a, grid, block, lds, stream); break;
        default: *rc = mix_run_dct1b(c, a, grid, block, lds, stream); break;
    }
    return true;
}

}  // namespace sfa

// Lines of lengths with a prime factor above 13, up to 2048, by Bluestein's
// algorithm (L. Bluestein, A linear filtering approach to the computation of
// discrete Fourier transform, 1970): with c_j = exp(-i pi j^2 / n),
//   X_k = c_k sum_j (x_j c_j) conj(c_{k-j}),
// a convolution, done as two FFTs of a length M >= 2n - 1 with small factors
// (the in-place passes of fft_mixed.h) and a product with the transform of
// conj(c).  Chirp and its transform are computed in extended precision.  It
// replaces a butterfly of the prime radix p at p multiply-adds (and two table
// loads each) per value: C2C along axis 1 of 64 x 313 x 33 385 -> 49 us, 100 x
// 146 x 51 147 -> 45, 218 x 38 x 144 85 -> 59, 64 x 17 x 65 18 -> 12; DCT-II and
// DCT-III of 218 x 38 x 144 along axis 0 405 -> 62; one line of 1284 reals 146 ->
// 27.  Bound by its two transforms of twice the length, at two waves per SIMD.  Inverse transforms run as the conjugate of the forward
// transform of the conjugate, the second FFT likewise, so that one body of
// passes serves all of them.
#include <complex>
#include <map>
#include <mutex>
#include <vector>

#include "mix_line.h"

namespace sfa {

struct BlueArgs {
    MixArgs a;             // plan: of M; tw: of M; n: logical length of the operation
    int nf;                // FFT length
    int op, inv, cplx, comp;
    const double2* chirp;  // c_j, nf entries
    const double2* bhat;   // FFT of conj(c) / M, M entries
};

// Values per thread held between the FFTs: T M <= 16 * 256, and a smaller
// workgroup has a thread for every 16 values at least (mix_setup: one per
// butterfly).
constexpr int BLUE_HOLD = 16;

__global__ void __launch_bounds__(256) blue_kernel(BlueArgs ba)
{
    const MixArgs& a = ba.a;
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
    const int buf = 0, twT = a.T * pl.size(), ends = twT + pl.n;
    const int op = ba.op, n = a.n, nf = ba.nf, M = pl.n;
    const bool ic = ba.cplx || op == OP_C2RF || op == OP_C2R;                    // complex input
    const bool oc = (ba.cplx && op != OP_C2R && op != OP_C2RF) || op == OP_R2CF || op == OP_R2C;  // complex output
    const int64_t is2 = a.in_s2, isa = a.in_sa, os2 = a.out_s2, osa = a.out_sa;
    const char* inb = a.in + (i1 * a.in_s1 + t0 * is2) * (ic ? 16 : 8);
    char* outb = a.out + (i1 * a.out_s1 + t0 * os2) * (oc ? 16 : 8);
    const double sc = a.scale;
    const double* K2 = a.K2;
    const float inv_nb = 1.0f / (float)pl.sub[0];
    const double sgn = ba.inv ? -1.0 : 1.0;
    auto in_put = [&](int t, int i, double2 v) { lds_put(buf + mix_in_pos(pl, i, inv_nb) * m.ps + t * m.ts, v); };
    auto at = [&](int t, int k) { return buf + mix_pos(pl, k) * m.ps + t * m.ts; };

    // 1. (x_j c_j), j < nf, zeros up to M; the operation's own pre-processing
    auto fill = [&](auto CI, auto CC, auto value) {
        constexpr bool IC = decltype(CI)::v != 0, COMP = decltype(CC)::v != 0;
        auto ild = [&](int t, int i) { return mix_ld<IC>(inb, t * is2 + i * isa); };
        auto ortho = [&](int t, int k) {  // composite input in the orthogonal basis
            if constexpr (!COMP) return ild(t, k);
            const double2 v = ild(t, k < n - 2 ? k : n - 3), u = ild(t, k >= 2 ? k - 2 : 0);
            const double kk = k >= 2 ? K2[k - 2] : 0.0, on = k < n - 2 ? 1.0 : 0.0;
            return make_double2(on * v.x + kk * u.x, on * v.y + kk * u.y);
        };
        double2 v[4], c[4];
        four_at_a_time(
            m, M, tid, nth,
            [&](int t, int i, int q) {
                const int j = i < nf ? i : 0;
                v[q] = value(ild, ortho, t, j);
                c[q] = ba.chirp[j];
            },
            [&](int t, int i, int q) {
                in_put(t, i, i < nf ? cmul(make_double2(v[q].x, sgn * v[q].y), c[q]) : make_double2(0.0, 0.0));
            });
        if (op == OP_DCT3 || op == OP_DCT1B)  // first and last value of each line
            for (int e = tid; e < 2 * m.Tv; e += nth) lds_put(ends + e, ortho(e >> 1, (e & 1) ? n - 1 : 0));
    };
    auto by_type = [&](auto value) {
        if (ic && ba.comp) fill(IC<1>{}, IC<1>{}, value);
        else if (ic) fill(IC<1>{}, IC<0>{}, value);
        else if (ba.comp) fill(IC<0>{}, IC<1>{}, value);
        else fill(IC<0>{}, IC<0>{}, value);
    };
    mix_twiddles(pl, twT, a.tw, tid, nth);
    switch (op) {
        case OP_R2C:
            fill(IC<0>{}, IC<0>{}, [&](auto&, auto&, int t, int j) {
                const double* p = reinterpret_cast<const double*>(inb) + t * is2 + 2 * j * isa;
                return make_double2(p[0], p[isa]);
            });
            break;
        case OP_C2RF:
            fill(IC<1>{}, IC<0>{}, [&](auto& ild, auto&, int t, int j) {
                const bool up = j > n / 2;
                const double2 v = ild(t, up ? n - j : j);
                return make_double2(v.x, j == 0 ? 0.0 : (up ? -v.y : v.y));
            });
            break;
        case OP_C2R:
            fill(IC<1>{}, IC<0>{}, [&](auto& ild, auto&, int t, int j) {
                double2 xk = ild(t, j), xc = cconj(ild(t, n / 2 - j));
                if (j == 0) xk.y = xc.y = 0.0;
                const double2 d = cmul(cconj(a.tw2[j]), csub(xk, xc));
                return make_double2(xk.x + xc.x - d.y, xk.y + xc.y + d.x);
            });
            break;
        case OP_DCT2:
            by_type([&](auto& ild, auto&, int t, int j) { return ild(t, 2 * j < n ? 2 * j : 2 * (n - 1 - j) + 1); });
            break;
        case OP_DCT3:
            by_type([&](auto&, auto& ortho, int t, int j) {
                const double2 ck = ortho(t, j);
                double2 cn = ortho(t, j == 0 ? 0 : n - j);
                if (j == 0) cn = make_double2(0.0, 0.0);
                return cmul(cconj(a.tw2[j]), make_double2(ck.x + cn.y, ck.y - cn.x));
            });
            break;
        case OP_DCT1F:
            by_type([&](auto& ild, auto&, int t, int j) { return ild(t, j < n ? j : 2 * (n - 1) - j); });
            break;
        case OP_DCT1B:
            by_type([&](auto&, auto& ortho, int t, int j) { return ortho(t, j < n ? j : 2 * (n - 1) - j); });
            break;
        default:  // OP_C2C, OP_R2CF
            by_type([&](auto& ild, auto&, int t, int j) { return ild(t, j); });
            break;
    }
    // 2. FFT, product with the chirp's transform (conjugated), FFT
#pragma unroll 1
    for (int rep = 0; rep < 2; ++rep) {
        __syncthreads();
        auto none = [](int, int) -> int64_t { return 0; };
        auto back = [&](int64_t, int t, int, int pos, double2 v) { lds_put(buf + pos * m.ps + t * m.ts, v); };
        mix_first<false>(
            pl, m, buf, twT, tid, nth, [&](int t, int j) -> int64_t { return buf + j * m.ps + t * m.ts; },
            (int64_t)pl.P * m.ps, [&](int64_t o, int, int) { return lds_get((int)o); }, none, 0, back);
        mix_rest<false>(pl, m, buf, a.tw, tid, nth, none, 0, back);
        __syncthreads();
        if (rep == 0) {
            double2 hold[BLUE_HOLD];
            MixIter g(m, M, tid, nth);
#pragma unroll
            for (int i = 0; i < BLUE_HOLD; ++i) {
                hold[i] = make_double2(0.0, 0.0);
                if (!g.done() && g.here()) hold[i] = cconj(cmul(lds_get(at(g.t, g.k)), ba.bhat[g.k]));
                g.next();
            }
            __syncthreads();
            MixIter h(m, M, tid, nth);
#pragma unroll
            for (int i = 0; i < BLUE_HOLD; ++i) {
                if (!h.done() && h.here()) in_put(h.t, h.k, hold[i]);
                h.next();
            }
        }
    }
    // 3. X_k = c_k conj(.), conjugated again for an inverse transform; post-processing
    auto val = [&](int t, int k) {
        const double2 v = cmul(ba.chirp[k], cconj(lds_get(at(t, k))));
        return make_double2(v.x, sgn * v.y);
    };
    auto ost = [&](int64_t off, double2 v) {
        if (oc) mix_st<true>(outb, off, v);
        else mix_st<false>(outb, off, v);
    };
    double2 x[4], y[4], w[4], wn[4];
    auto pairs = [&](int len, auto put) {  // k and len - k
        four_at_a_time(
            m, len / 2 + 1, tid, nth,
            [&](int t, int k, int i) {
                x[i] = val(t, k);
                y[i] = val(t, k == 0 ? 0 : len - k);
                w[i] = a.tw2[k];
                wn[i] = a.tw2[op == OP_R2C || k > 0 ? len - k : 0];
            },
            put);
    };
    if (op == OP_R2C) {
        const int h = n / 2;
        pairs(h, [&](int t, int k, int i) {
            auto X = [&](double2 z, double2 zz, double2 ww) {
                const double2 c = cconj(zz), d = cmul(ww, csub(z, c));
                return make_double2(0.5 * (z.x + c.x + d.y) * sc, 0.5 * (z.y + c.y - d.x) * sc);
            };
            ost(t * os2 + k * osa, X(x[i], y[i], w[i]));
            if (2 * k != h) ost(t * os2 + (h - k) * osa, X(y[i], x[i], wn[i]));
        });
    } else if (op == OP_DCT2) {
        pairs(n, [&](int t, int k, int i) {
            auto X = [&](double2 P, double2 V, double2 ww) {
                const double2 Q = cconj(V);
                return make_double2(cmul(ww, cadd(P, Q)).x * sc, cmul(ww, csub(P, Q)).y * sc);
            };
            const double2 p = X(x[i], y[i], w[i]), q = X(y[i], x[i], wn[i]);
            const bool two = k > 0 && 2 * k != n;
            if (ba.comp) {
                lds_put(at(t, k), p);
                if (two) lds_put(at(t, n - k), q);
            } else {
                ost(t * os2 + k * osa, p);
                if (two) ost(t * os2 + (n - k) * osa, q);
            }
        });
    } else {
        const int len = op == OP_R2CF ? n / 2 + 1 : op == OP_DCT1B ? n : nf;
        four_at_a_time(
            m, len, tid, nth, [&](int t, int k, int i) { x[i] = val(t, k); },
            [&](int t, int k, int i) {
                double2 v = x[i];
                if (op == OP_C2R) {
                    double* p = reinterpret_cast<double*>(outb) + t * os2 + 2 * k * osa;
                    p[0] = v.x * sc;
                    p[osa] = v.y * sc;
                } else if (op == OP_DCT3) {
                    const double2 c0 = lds_get(ends + 2 * t);
                    ost(t * os2 + (2 * k < n ? 2 * k : 2 * (n - 1 - k) + 1) * osa,
                        make_double2((0.5 * v.x + 0.5 * c0.x) * sc, (0.5 * v.y + 0.5 * c0.y) * sc));
                } else if (op == OP_DCT1B) {
                    const double2 c0 = lds_get(ends + 2 * t), c1 = lds_get(ends + 2 * t + 1);
                    const double sg = (k & 1) ? -0.5 : 0.5;
                    ost(t * os2 + k * osa, make_double2((0.5 * v.x + 0.5 * c0.x + sg * c1.x) * sc,
                                                        (0.5 * v.y + 0.5 * c0.y + sg * c1.y) * sc));
                } else if (op == OP_DCT1F) {
                    lds_put(at(t, k), cscale(v, sc));
                } else {
                    ost(t * os2 + k * osa, cscale(v, sc));
                }
            });
    }
    if ((op == OP_DCT2 && ba.comp) || op == OP_DCT1F) {  // stencil s_k + K2_k s_{k+2}, k < n - 2
        __syncthreads();
        double kk[4];
        four_at_a_time(
            m, n, tid, nth,
            [&](int t, int k, int i) {
                const bool st = ba.comp && k < n - 2;
                x[i] = lds_get(at(t, k));
                y[i] = lds_get(at(t, st ? k + 2 : k));
                kk[i] = st ? K2[k] : 0.0;
            },
            [&](int t, int k, int i) {
                double2 v = x[i];
                if (ba.comp && k < n - 2) {
                    v.x += kk[i] * y[i].x;
                    v.y += kk[i] * y[i].y;
                }
                ost(t * os2 + k * osa, v);
            });
    }
}

// --------------------------------------------------------------- tables
using cld = std::complex<long double>;

// FFT of x[0], x[s], .. (n of them) into y, by the factors of n (at most 13)
static void host_fft(const cld* x, cld* y, int n, int s, const std::vector<cld>& tw, int tws)
{
    if (n == 1) {
        y[0] = x[0];
        return;
    }
    int p = 2;
    while (n % p) ++p;
    const int q = n / p;
    for (int r = 0; r < p; ++r) host_fft(x + (int64_t)r * s, y + (int64_t)r * q, q, s * p, tw, tws * p);
    const int N = (int)tw.size();
    std::vector<cld> z(p);
    for (int k = 0; k < q; ++k) {
        for (int r = 0; r < p; ++r) z[r] = y[r * q + k] * tw[(int)((int64_t)r * k * tws % N)];
        for (int j = 0; j < p; ++j) {
            cld v = 0;
            for (int r = 0; r < p; ++r) v += z[r] * tw[(int)((int64_t)r * j * (N / p) % N)];
            y[j * q + k] = v;
        }
    }
}

struct BlueTable {
    int M;
    double2* d;  // chirp [nf] | transform of its conjugate [M]
};
static std::mutex g_blue_mu;
static std::map<std::pair<int, int>, BlueTable> g_blue;  // (nf, device)

// Length with factors up to 13 and at least 2 nf - 1: the least M (np + 1), np
// its passes.
static int blue_length(int nf)
{
    int best = 0;
    double cost = 0;
    for (int M = 2 * nf - 1; M <= 4096 && M <= 3 * nf; ++M) {
        MixPlan p;
        if (!make_mix_plan(M, true, &p)) continue;
        const double c = (double)M * (p.np + 1);
        if (!best || c < cost) {
            best = M;
            cost = c;
        }
    }
    return best;
}

static bool blue_table(int nf, BlueTable* out, int* rc)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    std::lock_guard<std::mutex> lk(g_blue_mu);
    auto it = g_blue.find({nf, dev});
    if (it != g_blue.end()) {
        *out = it->second;
        return true;
    }
    const int M = blue_length(nf);
    if (!M) return false;
    if (alloc_forbidden()) {
        *rc = fail(SFA_ERR_ARG, "chirp table of length %d was not built before a no-allocation call", nf);
        return true;
    }
    const long double pi = 3.141592653589793238462643383279502884L;
    std::vector<cld> b(M), f(M), tw(M);
    std::vector<double2> h((size_t)nf + M);
    for (int m = 0; m < M; ++m) tw[m] = cld(cosl(2 * pi * m / M), -sinl(2 * pi * m / M));
    for (int j = 0; j < nf; ++j) {
        const long double t = pi * (long double)((int64_t)j * j % (2 * (int64_t)nf)) / nf;
        const cld c(cosl(t), sinl(t));
        h[j] = make_double2((double)c.real(), (double)-c.imag());
        b[j] = c;
        if (j) b[M - j] = c;
    }
    host_fft(b.data(), f.data(), M, 1, tw, 1);
    for (int k = 0; k < M; ++k) h[nf + k] = make_double2((double)(f[k].real() / M), (double)(f[k].imag() / M));
    BlueTable t{M, nullptr};
    hipError_t e = hipMalloc(&t.d, h.size() * sizeof(double2));
    if (e == hipSuccess) {
        e = hipMemcpy(t.d, h.data(), h.size() * sizeof(double2), hipMemcpyHostToDevice);
        if (e != hipSuccess) (void)hipFree(t.d);
    }
    if (e != hipSuccess) {
        *rc = fail(SFA_ERR_HIP, "chirp table of length %d failed: %s", nf, hipGetErrorString(e));
        return true;
    }
    g_blue[{nf, dev}] = t;
    *out = t;
    return true;
}

// Tables of the complex lines of length nf that no plan of the caller holds:
// a pipeline that is captured into a graph right after its plan was made may
// not allocate them then.
int line_tables(int nf)
{
    SFA_CHECK(fft_table(nf) != nullptr, SFA_ERR_HIP, "table allocation failed");
    MixPlan p;
    if (make_mix_plan(nf, true, &p) || nf > 2048) return SFA_OK;
    int rc = SFA_OK;
    BlueTable tab{0, nullptr};
    if (!blue_table(nf, &tab, &rc)) return SFA_OK;
    SFA_CHECK(rc || fft_table(tab.M) != nullptr, SFA_ERR_HIP, "table allocation failed");
    return rc;
}

bool blue_launch(int op, bool inv, const LineArgs& la, hipStream_t stream, int* rc)
{
    BlueArgs ba;
    MixArgs& a = ba.a;
    const int nf = la.plan.nfft;
    if (nf > 2048) return false;
    *rc = SFA_OK;
    BlueTable tab{0, nullptr};
    if (!blue_table(nf, &tab, rc)) return false;
    if (*rc) return true;
    LineArgs lb = la;
    lb.plan.nfft = tab.M;
    dim3 grid;
    unsigned block;
    size_t lds;
    int most = 16;
    while (most > 1 && most * tab.M > BLUE_HOLD * 256) most >>= 1;
    if (!mix_setup(lb, a, &grid, &block, &lds, most)) return false;
    a.tw = fft_table(tab.M);
    if (!a.tw) {
        *rc = fail(SFA_ERR_HIP, "twiddle table allocation failed");
        return true;
    }
    ba.nf = nf;
    ba.op = op;
    ba.inv = inv;
    ba.cplx = la.in_cplx != 0;
    ba.comp = la.K2 != nullptr;
    ba.chirp = tab.d;
    ba.bhat = tab.d + nf;
    if (lds > 64 * 1024) {
        const hipError_t e =
            hipFuncSetAttribute((const void*)blue_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            *rc = fail(SFA_ERR_HIP, "LDS size %d refused: %s", (int)lds, hipGetErrorString(e));
            return true;
        }
    }
    hipLaunchKernelGGL(blue_kernel, grid, dim3(block), lds, stream, ba);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) *rc = fail(SFA_ERR_HIP, "kernel launch failed: %s", hipGetErrorString(e));
    return true;
}

}  // namespace sfa

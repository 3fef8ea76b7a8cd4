// gfx950 strided line passes (kinetic parts along dimensions >= 1, GSPO
// kinetic split operator, forward/inverse transforms) and H applied to a
// complex128 vector (Operator::Apply).
#include "qdx_gridfft.hpp"
#include "qdx_kernels_common.hpp"

namespace qdx {

// ---------------------------------------------------------------------------
// Strided line pass along dimension `dim` (1 or 2) on X, in place.  A block
// owns a tile of W adjacent dimension-0 positions for one state and one index
// of the remaining dimension; the W lanes of a butterfly touch W adjacent
// words in LDS and W adjacent complex values in memory.
// MODE 0: forward, 1: inverse, 2: forward * T/N inverse,
//      3: forward * exp(-i tau T)/N inverse,
//      4: X = IFFT(T_dim/N_dim FFT(src)), the dimension's part of the
//         separable kinetic operator, 5: X += the same.
// CMP (modes 4 and 5): src and X in the compact 40-bit term storage.
// GEN: as fft_line.
template <class R, int MODE, int P = 8, bool IMAG = false, bool CMP = false, bool GEN = true>
__global__ void __launch_bounds__(512) k_col(GridDev g, int S, int dim, int W, LinePlan p, HamDev<R> h, double tau,
                                              cx<R> *__restrict__ X, const cx<R> *__restrict__ src,
                                              ChebyCtl *ctl, ConvCheck cc, const double *__restrict__ ek) {
    if (ctl && ctl->done) return;
    extern __shared__ __align__(16) char smem_raw[];
    cx<R> *smem = reinterpret_cast<cx<R> *>(smem_raw);
    __shared__ double bc;
    const int N0 = g.N[0];
    const int L = g.N[dim];
    const int TL = L / P;
    const long estride = dim_stride(g, dim);
    const int nother = col_nother(g, dim);
    const int tiles0 = N0 / W;
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int c0 = (b % tiles0) * W;
    const int rest = b / tiles0;
    const int oth = rest % nother;
    const int st = rest / nother;
    const int c = threadIdx.x % W;
    const int lt = threadIdx.x / W;
    const bool active = lt < TL;
    int kk[kMaxDims] = {0, 0, 0, 0};   // k-space index per dimension (dimensions 0 and dim set below)
    const long boff = (long)st * g.size + col_other(g, dim, oth, kk) + c0 + c;   // element of this thread's column
    const long nT = (long)S * g.size;
    LdsLine<R> ln;
    ln.a = smem + c;
    ln.b = smem + (long)W * tw_lds_len(L) + c;
    ln.es = W;
    ln.pad = true;
    cx<R> *twl = smem + (long)2 * W * tw_lds_len(L);
    cx<R> v[P], yv[P];
    const bool tw_in_lds = p.tw_lds;
    auto FFT = [&](int sign) {
        if (tw_in_lds) fft_line<R, P, false, GEN>(v, ln, p, twl, sign, lt, active, kTwLds);
        else fft_line<R, P, false, GEN>(v, ln, p, reinterpret_cast<const cx<R> *>(p.tw), sign, lt, active, kTwMem);
    };

    if (active) {
        const cx<R> *in = MODE >= 4 ? src : X;
#pragma unroll
        for (int q = 0; q < P; ++q) v[q] = tld<CMP>(in, boff + (long)(lt + q * TL) * estride, nT);
        if (MODE == 5) {
#pragma unroll
            for (int q = 0; q < P; ++q) yv[q] = tld<CMP>(X, boff + (long)(lt + q * TL) * estride, nT);
        }
    }
    // kinetic table values of this thread's elements, requested early.
    // Real-time GSPO (mode 3) with ek: the factor exp(-i tau T(k)) / N as
    // inv_n times the product over dimensions of exp(-i tau T_d(k_d)) from
    // the per-state tables ek (state st at 2 st sum_d N_d doubles, dimension
    // d after the tables of the dimensions before it, (re, im) pairs)
    double tq[P];
    cx<double> fq[P];
    const bool etab = MODE == 3 && !IMAG && ek != nullptr;
    if (etab && active) {
        long tot = 0, offd = 0;
        long off[kMaxDims] = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < kMaxDims; ++e) {
            off[e] = tot;
            if (e < g.nd) tot += g.N[e];
            if (e == dim) offd = off[e];
        }
        const double *es = ek + 2 * (long)st * tot;
        kk[0] = c0 + c;
        cx<double> fo = mk<double>(h.inv_n, 0.0);
#pragma unroll
        for (int e = 0; e < kMaxDims; ++e) {
            if (e < g.nd && e != dim) {
                const double *q = es + 2 * (off[e] + kk[e]);
                fo = cmul(fo, mk<double>(q[0], q[1]));
            }
        }
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const double *t = es + 2 * (offd + lt + q * TL);
            fq[q] = cmul(fo, mk<double>(t[0], t[1]));
        }
    } else if (MODE >= 2 && active) {
        const bool has_t = h.tk[st][0] != nullptr;
        kk[0] = c0 + c;
#pragma unroll
        for (int q = 0; q < P; ++q) {
            const int kd = lt + q * TL;
#pragma unroll
            for (int e = 1; e < kMaxDims; ++e)
                if (e == dim) kk[e] = kd;
            if (MODE >= 4) tq[q] = has_t ? (0.0 + h.tk[st][dim][kd]) * h.inv_nd[dim] : 0.0;
            else tq[q] = has_t ? kin_sum<R>(h, st, g, kk) : 0.0;
        }
    }
    if (tw_in_lds) stage_twiddles(twl, p);
    {
        double a;
        if (prev_converged(cc, &bc, &a)) {
            // the previous order ended the series (OCheby.cpp:179-182); the
            // row kernel of this order reads the outcome from ctl.  Every
            // block reaches the same decision, block 0 records it.
            if (MODE == 4 && ctl && b == 0 && threadIdx.x == 0) {
                ctl->done = 1;
                ctl->accnorm = a;
            }
            return;
        }
    }
    FFT(MODE == 1 ? +1 : -1);
    if (MODE >= 2) {
        if (active) {
#pragma unroll
            for (int q = 0; q < P; ++q) {
                const double tt = tq[q];
                if (MODE >= 4) {
                    v[q] = mk<R>((R)((double)v[q].r * tt), (R)((double)v[q].i * tt));
                } else if (MODE == 2) {
                    const double t = tt * h.inv_n;
                    v[q] = mk<R>((R)((double)v[q].r * t), (R)((double)v[q].i * t));
                } else if (IMAG) {
                    // exp(-tau T) / N, imaginary time
                    const double f = exp(-tau * tt) * h.inv_n;
                    v[q] = mk<R>((R)((double)v[q].r * f), (R)((double)v[q].i * f));
                } else if (etab) {
                    v[q] = from_d<R>(cmul(to_d(v[q]), fq[q]));
                } else {
                    // exp(-i tau T) / N (OGSPO.cpp:37-41 folds 1/N into the exponential)
                    double sn, cs;
                    sincos(-tau * tt, &sn, &cs);
                    v[q] = from_d<R>(cmul(to_d(v[q]), mk<double>(cs * h.inv_n, sn * h.inv_n)));
                }
            }
        }
        FFT(+1);
    }
    if (active) {
        if (MODE == 5) {
#pragma unroll
            for (int q = 0; q < P; ++q) v[q] = v[q] + yv[q];
        }
#pragma unroll
        for (int q = 0; q < P; ++q) tst<CMP>(X, boff + (long)(lt + q * TL) * estride, nT, v[q]);
    }
}

// ---------------------------------------------------------------------------
// H applied to a complex128 vector (Operator::Apply): forward row pass,
// strided passes, row epilogue.
template <class R, int S>
__global__ void __launch_bounds__(512) k_row_fwd(GridDev g, LinePlan p0, int rb, const cx<double> *__restrict__ src,
                                                  cx<R> *__restrict__ X) {
    extern __shared__ __align__(16) char smem_raw[];
    RowBlock<R> B(g, rb, S, reinterpret_cast<cx<R> *>(smem_raw), p0);
    const long base = (long)B.st * g.size;
    cx<R> v[8];
    if (B.active) {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = from_d<R>(src[base + B.gidx(q)]);
    }
    B.stage(p0);
    B.fft(v, p0, -1);
    if (B.active) {
#pragma unroll
        for (int q = 0; q < 8; ++q) X[base + B.gidx(q)] = v[q];
    }
}

template <class R, int S, bool ONE_D>
__global__ void __launch_bounds__(512) k_apply_row(GridDev g, HamDev<R> h, LinePlan p0, int rb,
                                                    const cx<double> *__restrict__ src, const cx<R> *__restrict__ X,
                                                    cx<double> *__restrict__ dst) {
    extern __shared__ __align__(16) char smem_raw[];
    RowBlock<R> B(g, rb, S, reinterpret_cast<cx<R> *>(smem_raw), p0);
    const int st = B.st;
    const long base = (long)st * g.size;
    cx<R> v[8];
    if (B.active) {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = ONE_D ? from_d<R>(src[base + B.gidx(q)]) : X[base + B.gidx(q)];
    }
    B.stage(p0);
    const bool has_t = h.tk[st][0] != nullptr;
    if (ONE_D) {
        B.fft(v, p0, -1);
        if (B.active) {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const double t = has_t ? (0.0 + h.tk[st][0][B.lt + q * B.TL]) * h.inv_n : 0.0;
                v[q] = mk<R>((R)((double)v[q].r * t), (R)((double)v[q].i * t));
            }
        }
    }
    B.fft(v, p0, +1);
    if (!B.active) return;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const long gi = B.gidx(q);
        cx<double> hp = has_t ? to_d(v[q]) : mk<double>(0, 0);
#pragma unroll
        for (int j = 0; j < S; ++j) {
            double w = (j == st) ? h.unity[st] : 0.0;
            if (h.W[st][j]) w += (double)h.W[st][j][gi];
            if (h.mu[st][j]) w += h.Edip[st][j] * (double)h.mu[st][j][gi];
            const cx<double> pj = src[(long)j * g.size + gi];
            hp.r += w * pj.r;
            hp.i += w * pj.i;
        }
        if (h.Wi[st]) {   // negative imaginary potential: -i Wi psi
            const double c = (double)h.Wi[st][gi];
            const cx<double> ps = src[base + gi];
            hp.r += c * ps.i;
            hp.i -= c * ps.r;
        }
        dst[base + gi] = hp;
    }
}

template <class R, int P, bool GEN>
static void col_pass_P(hipStream_t s, const GridDev &g, int S, int dim, int mode, const LinePlan &plan,
                       const HamDev<R> &h, double tau, R *X, ChebyCtl *ctl, const ConvCheck &cc, int imag,
                       const double *ek) {
    const int L = g.N[dim];
    const int W = col_tile(g, S, dim, L, sizeof(cx<R>), P);
    const int nb = (g.N[0] / W) * col_nother(g, dim) * S;
    const int threads = std::max(64, round64(W * (L / P)));
    const size_t lds = col_lds_bytes(W, L, sizeof(cx<R>));
    cx<R> *x = reinterpret_cast<cx<R> *>(X);
    LinePlan pl = plan;
    pl.tw_lds = 1;
    const cx<R> *none = nullptr;
    const double *ekp = mode == 3 && !imag ? ek : nullptr;
    auto launch = [&](auto kernel) {
        set_lds(kernel, lds);
        QDX_LAUNCH(kernel, dim3(nb), dim3(threads), lds, s, g, S, dim, W, pl, h, tau, x, none, ctl, cc, ekp);
        QDX_HIP(hipGetLastError());
    };
    switch (mode) {
    case 0: launch(k_col<R, 0, P, false, false, GEN>); break;
    case 1: launch(k_col<R, 1, P, false, false, GEN>); break;
    case 2:   // H psi
        if constexpr (P == 8) launch(k_col<R, 2>);
        else throw std::runtime_error("line pass: mode 0, 1 or 3 at 4 points per thread");
        break;
    default:
        if (!imag) {
            launch(k_col<R, 3, P, false, false, GEN>);
        } else {
            if constexpr (std::is_same<R, double>::value) launch(k_col<R, 3, P, true>);
            else throw std::runtime_error("imaginary time: FP64 only");
        }
        break;
    }
}

template <class R>
void Launch<R>::col_pass(hipStream_t s, const GridDev &g, int S, int dim, int mode, const LinePlan &plan,
                         const HamDev<R> &h, double tau, R *X, ChebyCtl *ctl, const ConvCheck &cc, int imag,
                         const double *ek) {
    const bool gen = plan.odd_prime();
    if (plan.ppt == 4 && gen) col_pass_P<R, 4, true>(s, g, S, dim, mode, plan, h, tau, X, ctl, cc, imag, ek);
    else if (plan.ppt == 4) col_pass_P<R, 4, false>(s, g, S, dim, mode, plan, h, tau, X, ctl, cc, imag, ek);
    else if (gen) col_pass_P<R, 8, true>(s, g, S, dim, mode, plan, h, tau, X, ctl, cc, imag, ek);
    else col_pass_P<R, 8, false>(s, g, S, dim, mode, plan, h, tau, X, ctl, cc, imag, ek);
}

// Mode 4 of k_col by the in-place line filter (qdx_gridfft.hpp): half the LDS
// and half the exchanges of the two Stockham transforms, so that more blocks
// share a CU.  128^3 points: FP64 (67 MB) 32.7 -> 24.0 us, compact terms (42
// MB) 20.5 -> 17.6.  Mode 5 stays with k_col: its larger stride and third
// stream bound it elsewhere (36.5 against 37.6 us here, compact 24.6 against
// 28.6).  FP32: the same on 128^3 points (14.5 against 14.6 us), ahead on others (a
// whole step on 64^3 points 1.03 -> 0.98 ms).
template <class R, bool CMP>
__global__ void __launch_bounds__(256, 3) k_kin_filter(GridDev g, int S, int dim, int W, LinePlan p, int R2, int R3,
                                                       HamDev<R> h, cx<R> *__restrict__ Y,
                                                       const cx<R> *__restrict__ src, ChebyCtl *ctl, ConvCheck cc) {
    if (ctl && ctl->done) return;
    extern __shared__ __align__(16) char smem_raw[];
    __shared__ double bc;
    const int N0 = g.N[0], L = g.N[dim], len = grid_line_len(R2, R3);
    const long estride = dim_stride(g, dim);
    const int nother = col_nother(g, dim), tiles0 = (N0 + W - 1) / W;
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int rest = b / tiles0, oth = rest % nother, st = rest / nother;
    GridAxis<R> A;
    A.m = L / 8;
    A.R2 = R2;
    A.R3 = R3;
    A.RS = grid_rs(R3);
    A.nl = W;
    A.lt = threadIdx.x / W;
    A.a = A.lt / R3;
    A.b = A.lt - A.a * R3;
    const int c = threadIdx.x - A.lt * W, c0 = (b % tiles0) * W + c;
    A.on = A.lt < A.m && c0 < N0;
    int kk[kMaxDims] = {0, 0, 0, 0};
    const long boff = (long)st * g.size + col_other(g, dim, oth, kk) + c0;   // element of this thread's column
    const long nT = (long)S * g.size;
    cx<R> *smem = reinterpret_cast<cx<R> *>(smem_raw), *tw = smem + W * len;
    double *f = reinterpret_cast<double *>(tw + grid_tw_len(A.m));
    A.buf = smem + c;
    A.tw1 = tw;
    A.tw2 = tw + 7 * A.m;
    cx<R> v[8];
    if (A.on) {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = tld<CMP>(src, boff + (long)(A.lt + q * A.m) * estride, nT);
    }
    grid_tables(reinterpret_cast<const cx<R> *>(p.tw), A.m, R3, tw, tw + 7 * A.m);
    grid_factors(h.tk[st][0] ? h.tk[st][dim] : nullptr, h.inv_nd[dim], R2, R3, f);
    {
        double a;
        if (prev_converged(cc, &bc, &a)) {   // as k_col
            if (ctl && b == 0 && threadIdx.x == 0) {
                ctl->done = 1;
                ctl->accnorm = a;
            }
            return;
        }
    }
    __syncthreads();
    grid_filter<false>(v, A, f, [] {}, [] {});
    if (!A.on) return;
#pragma unroll
    for (int q = 0; q < 8; ++q) tst<CMP>(Y, boff + (long)(A.lt + q * A.m) * estride, nT, v[q]);
}

// false: the line or the grid does not suit k_kin_filter (lines of 8 m points
// with small prime factors; at least four adjacent columns per block)
template <class R>
static bool kin_filter(hipStream_t s, const GridDev &g, int S, int dim, const LinePlan &p,
                       const HamDev<R> &h, const R *src, R *Y, ChebyCtl *ctl, const ConvCheck &cc, bool cmp) {
    const int L = g.N[dim], m = L / 8;
    int R2, R3;
    if (L % 8 || !grid_radices(m, R2, R3) || R2 == 11 || R2 == 13 || R2 > 16 || R3 == 11 || R3 == 13) return false;
    int W = 256 / m;
    if (W > 16) W = 16;
    if (W > g.N[0]) W = g.N[0];
    if (W < 4) return false;
    const int nb = ((g.N[0] + W - 1) / W) * col_nother(g, dim) * S;
    const int threads = std::max(64, round64(W * m));
    const size_t lds = ((size_t)W * grid_line_len(R2, R3) + grid_tw_len(m)) * sizeof(cx<R>) +
                       grid_line_len(R2, R3) * sizeof(double);
    auto launch = [&](auto kernel) {
        set_lds(kernel, lds);
        QDX_LAUNCH(kernel, dim3(nb), dim3(threads), lds, s, g, S, dim, W, p, R2, R3, h, reinterpret_cast<cx<R> *>(Y),
                   reinterpret_cast<const cx<R> *>(src), ctl, cc);
        QDX_HIP(hipGetLastError());
    };
    if (cmp) {
        if constexpr (std::is_same<R, double>::value) launch(k_kin_filter<R, true>);
        else throw std::runtime_error("compact terms: FP64 only");
    } else {
        launch(k_kin_filter<R, false>);
    }
    return true;
}

template <class R, int P, bool GEN>
static void kin_pass_P(hipStream_t s, const GridDev &g, int S, int dim, bool accumulate, const LinePlan &plan,
                       const HamDev<R> &h, const R *src, R *Y, ChebyCtl *ctl, const ConvCheck &cc, bool cmp) {
    const int L = g.N[dim];
    const int W = col_tile(g, S, dim, L, sizeof(cx<R>), P);
    const int nb = (g.N[0] / W) * col_nother(g, dim) * S;
    const int threads = std::max(64, round64(W * (L / P)));
    const size_t lds = col_lds_bytes(W, L, sizeof(cx<R>));
    cx<R> *y = reinterpret_cast<cx<R> *>(Y);
    const cx<R> *in = reinterpret_cast<const cx<R> *>(src);
    const double *ekp = nullptr;
    LinePlan pl = plan;
    pl.tw_lds = 1;
    auto launch = [&](auto kernel) {
        set_lds(kernel, lds);
        QDX_LAUNCH(kernel, dim3(nb), dim3(threads), lds, s, g, S, dim, W, pl, h, 0.0, y, in, ctl, cc, ekp);
        QDX_HIP(hipGetLastError());
    };
    if (cmp) {
        if constexpr (std::is_same<R, double>::value) {
            if (accumulate) launch(k_col<R, 5, P, false, true, GEN>);
            else launch(k_col<R, 4, P, false, true, GEN>);
        } else {
            throw std::runtime_error("compact terms: FP64 only");
        }
    } else if (accumulate) {
        launch(k_col<R, 5, P, false, false, GEN>);
    } else {
        launch(k_col<R, 4, P, false, false, GEN>);
    }
}

template <class R>
void Launch<R>::kin_pass(hipStream_t s, const GridDev &g, int S, int dim, bool accumulate, const LinePlan &plan,
                         const HamDev<R> &h, const R *src, R *Y, ChebyCtl *ctl, const ConvCheck &cc, bool cmp,
                         bool filter) {
    if (filter && !accumulate && kin_filter<R>(s, g, S, dim, plan, h, src, Y, ctl, cc, cmp)) return;
    const bool gen = plan.odd_prime();
    if (plan.ppt == 4 && gen) kin_pass_P<R, 4, true>(s, g, S, dim, accumulate, plan, h, src, Y, ctl, cc, cmp);
    else if (plan.ppt == 4) kin_pass_P<R, 4, false>(s, g, S, dim, accumulate, plan, h, src, Y, ctl, cc, cmp);
    else if (gen) kin_pass_P<R, 8, true>(s, g, S, dim, accumulate, plan, h, src, Y, ctl, cc, cmp);
    else kin_pass_P<R, 8, false>(s, g, S, dim, accumulate, plan, h, src, Y, ctl, cc, cmp);
}

template <class R, int S>
static void ham_apply_S(hipStream_t st, const GridDev &g, const HamDev<R> &h, const LinePlan *plans_in,
                        const double *src, double *dst, R *X) {
    LinePlan plans[kMaxDims];
    for (int d = 0; d < g.nd; ++d) plans[d] = plans_in[d];
    RowLaunch r = row_launch<R>(g, S, plans[0]);
    auto s = reinterpret_cast<const cx<double> *>(src);
    auto d = reinterpret_cast<cx<double> *>(dst);
    auto x = reinterpret_cast<cx<R> *>(X);
    if (g.nd == 1) {
        set_lds(k_apply_row<R, S, true>, r.lds);
        QDX_LAUNCH((k_apply_row<R, S, true>), dim3(r.nb), dim3(r.threads), r.lds, st, g, h, plans[0], r.rb, s,
                           x, d);
        QDX_HIP(hipGetLastError());
        return;
    }
    set_lds(k_row_fwd<R, S>, r.lds);
    QDX_LAUNCH((k_row_fwd<R, S>), dim3(r.nb), dim3(r.threads), r.lds, st, g, plans[0], r.rb, s, x);
    QDX_HIP(hipGetLastError());
    // forward transforms along dimensions 1 .. nd-2, the last dimension's
    // FFT * T(k)/N * IFFT, inverse transforms back down to dimension 1
    for (int d = 1; d < g.nd - 1; ++d) Launch<R>::col_pass(st, g, S, d, 0, plans[d], h, 0.0, X, nullptr, ConvCheck());
    Launch<R>::col_pass(st, g, S, g.nd - 1, 2, plans[g.nd - 1], h, 0.0, X, nullptr, ConvCheck());
    for (int d = g.nd - 2; d >= 1; --d) Launch<R>::col_pass(st, g, S, d, 1, plans[d], h, 0.0, X, nullptr, ConvCheck());
    set_lds(k_apply_row<R, S, false>, r.lds);
    QDX_LAUNCH((k_apply_row<R, S, false>), dim3(r.nb), dim3(r.threads), r.lds, st, g, h, plans[0], r.rb, s, x,
                       d);
    QDX_HIP(hipGetLastError());
}

template <class R>
void Launch<R>::ham_apply(hipStream_t s, const GridDev &g, const HamDev<R> &h, const LinePlan *plans,
                          const double *src, double *dst, R *X) {
    QDX_DISPATCH_S(h.S, (ham_apply_S<R, SS>(s, g, h, plans, src, dst, X)));
}

template <class R>
void Launch<R>::line_fft(hipStream_t s, const GridDev &g, int S, int dim, const LinePlan &plan, const double *src,
                         R *X) {
    if (dim == 0) {
        QDX_DISPATCH_S(S, {
            LinePlan p0 = plan;
            RowLaunch r = row_launch<R>(g, SS, p0);
            set_lds(k_row_fwd<R, SS>, r.lds);
            QDX_LAUNCH((k_row_fwd<R, SS>), dim3(r.nb), dim3(r.threads), r.lds, s, g, p0, r.rb,
                       reinterpret_cast<const cx<double> *>(src), reinterpret_cast<cx<R> *>(X));
        });
        QDX_HIP(hipGetLastError());
        return;
    }
    if constexpr (!std::is_same<R, double>::value) throw std::runtime_error("line_fft: FP64 only");
    QDX_HIP(hipMemcpyAsync(X, src, (size_t)S * g.size * 2 * sizeof(double), hipMemcpyDeviceToDevice, s));
    col_pass(s, g, S, dim, 0, plan, HamDev<R>(), 0.0, X, nullptr, ConvCheck());
}

#define QDX_INST_LINES(R)                                                                                      \
    template void Launch<R>::col_pass(hipStream_t, const GridDev &, int, int, int, const LinePlan &,               \
                                      const HamDev<R> &, double, R *, ChebyCtl *, const ConvCheck &, int,           \
                                      const double *);                                                              \
    template void Launch<R>::kin_pass(hipStream_t, const GridDev &, int, int, bool, const LinePlan &,              \
                                      const HamDev<R> &, const R *, R *, ChebyCtl *, const ConvCheck &, bool,       \
                                      bool);                                                                       \
    template void Launch<R>::ham_apply(hipStream_t, const GridDev &, const HamDev<R> &, const LinePlan *,          \
                                       const double *, double *, R *);                                              \
    template void Launch<R>::line_fft(hipStream_t, const GridDev &, int, int, const LinePlan &, const double *, R *);
QDX_INST_LINES(double)
QDX_INST_LINES(float)

}  // namespace qdx

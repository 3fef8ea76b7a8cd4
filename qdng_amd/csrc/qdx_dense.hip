// gfx950 kernels of short 1D lines (up to 64 kDenseBlocks points): whole
// Chebyshev and split-operator runs in one block, with the kinetic operator
// applied as a dense circulant matrix from registers.
//
// A short line is a latency chain: the FFT kernels spend 3.1 us per order on
// 128 points in eight dependent LDS round trips of one half-filled wave.  The
// kinetic operator T = F^-1 diag(T_k) F is a symmetric circulant matrix
// t(i - j), so T phi is 2 N^2 multiply-adds without any chain; for N = 128
// these are 512 cycles of a CU's 64 FP64 lanes.  One radix-2 step halves
// them: with M = N / 2 and the real parities x_e,o(j) = phi(j) +- phi(j + M),
//   (T phi)(i) +- (T phi)(i + M) = sum_j [t(i - j) +- t(i - j + M)] x_e,o(j).
//
// Thread layout: 128 nb threads per state, nb = ceil(M / 32) blocks of 32
// rows of each parity.  tid = q + 8 par + 16 g + 128 blk (+ 128 nb st): rows
// 32 blk + g + 8 r (r < 4) of parity par against the columns q + 8 c (c < 4
// nb), so that the lanes of a read take consecutive LDS words, and a thread's
// 4 x 4 nb matrix elements hold only 4 nb + 3 different values (kept in
// registers).  The eight column lanes are summed by a reduce-scatter over
// DPP moves, which leaves every thread with one real component of one point;
// all that follows (multiplies with the surfaces, recurrence, psi) is done
// there, the other component one lane away.  One barrier per order publishes
// the new term and the partial sums of the break test together.
#include "qdx_gridfft.hpp"
#include "qdx_kernels_common.hpp"
#include "qdx_xsplit.hpp"

namespace qdx {

// position of a thread and the pieces of LDS it uses
template <int NB>
struct DenseLine {
    static constexpr int C = 4 * NB;              // columns per thread
    static constexpr int MP = 32 * NB;            // rows of a parity, padded
    static constexpr int PS = MP + 8;             // parity stride: the two parities on different banks
    static constexpr int T = 128 * NB;            // threads per state
    int q, par, st, wave, i, n, comp, N, M;
    bool own;      // this thread holds component comp of point n
    double tc[C + 3];
    __device__ DenseLine(int N_, const double *tab) {
        const int t = threadIdx.x;
        N = N_;
        M = N >> 1;
        q = t & 7;
        par = (t >> 3) & 1;
        const int g = (t >> 4) & 7;
        st = t / T;
        const int blk = (t - st * T) >> 7;
        wave = t >> 6;
        i = 32 * blk + g + 8 * (2 * (q >> 2) + ((q >> 1) & 1));
        comp = q & 1;
        n = i + par * M;
        own = i < M;
        // tab: [state][parity][N]
        const double *tb = tab + ((long)st * 2 + par) * N;
#pragma unroll
        for (int m = 0; m < C + 3; ++m) {
            int d = 32 * blk + g - q + 8 * (m - (C - 1));
            d %= N;
            if (d < 0) d += N;
            tc[m] = tb[d];
        }
    }
    // own component of T x from the parity vectors xs of this thread's state
    __device__ __forceinline__ double apply(const cx<double> *xs) const {
        double a[4][2] = {};
        const cx<double> *x = xs + par * PS + q;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const cx<double> v = x[8 * c];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                a[r][0] = __builtin_fma(tc[r - c + C - 1], v.r, a[r][0]);
                a[r][1] = __builtin_fma(tc[r - c + C - 1], v.i, a[r][1]);
            }
        }
        return scatter(a);
    }
    // sums over the eight column lanes, each lane keeping its own component,
    // and the two parities put together
    __device__ __forceinline__ double scatter(const double (&a)[4][2]) const {
        const bool b2 = q & 4, b1 = q & 2, b0 = q & 1;
        double h[2][2], s[2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const double keep = b2 ? a[2 + u][c] : a[u][c], send = b2 ? a[u][c] : a[2 + u][c];
                h[u][c] = keep + dpp<kXor7>(send);
            }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const double keep = b1 ? h[1][c] : h[0][c], send = b1 ? h[0][c] : h[1][c];
            s[c] = keep + dpp<kXor2>(send);
        }
        const double y = (b0 ? s[1] : s[0]) + dpp<kXor1>(b0 ? s[0] : s[1]);
        const double o = dpp<kXor8>(y);
        return par ? o - y : y + o;
    }
    // publish the own component p of a term: parity vectors and, for several
    // states, the point itself
    __device__ __forceinline__ void put(double p, cx<double> *xs, cx<double> *full) const {
        const double o = dpp<kXor8>(p);
        if (own) {
            reinterpret_cast<double *>(xs + par * PS + i)[comp] = par ? o - p : p + o;
            if (full) reinterpret_cast<double *>(full + n)[comp] = p;
        }
    }
};

// observables of the state before a step (Reporter.cpp:101-137), per state:
// sum |psi|^2 and sum conj(psi) psi0; red: 3 doubles per wave
__device__ __forceinline__ void dense_obs_put(double ps, double p0, int comp, int wave, double *red) {
    const double p0x = dpp<kXor1>(p0);
    const double n2 = dpp_wave_sum(ps * ps);
    const double ar = dpp_wave_sum(ps * p0);
    const double ai = dpp_wave_sum(comp ? -ps * p0x : ps * p0x);
    if ((threadIdx.x & 63) == 0) {
        red[3 * wave] = n2;
        red[3 * wave + 1] = ar;
        red[3 * wave + 2] = ai;
    }
}

// Chebyshev steps of a 1D line of S states (OCheby::real_time_step, and with
// IMAG imag_time_step, OCheby.cpp:92-297): the operands, break tests and
// orders of the per-order kernels, with every term in FP64.  fields: per step
// the S x S values -E(t) scale; obs (nullable): per step the sums of
// dense_obs_put as qdx_prop_run lays them out; orders: H applications per
// step.  The break test of an order is read beside the next order's product.
// Per order on one CU (128 points): 3.1 -> 0.5 us against the FFT kernel.
template <int NB, int S, bool NIP, bool IMAG>
__global__ void __launch_bounds__(128 * NB * S) k_dense_cheby(HamDev<double> h, DenseRun a, const double *tab,
                                                              const double *__restrict__ coef, int order,
                                                              double offset, double offset_i, double inv_scaling,
                                                              double prec, cx<double> *__restrict__ psi,
                                                              ChebyCtl *ctl, double *__restrict__ partials) {
    using D = DenseLine<NB>;
    __shared__ __align__(16) cx<double> xs[2][S][2 * D::PS];
    __shared__ __align__(16) cx<double> full[2][S > 1 ? S : 1][S > 1 ? 2 * D::MP : 1];
    constexpr int NW = D::T * S / 64;
    __shared__ double red[2][NW], ored[3 * NW];
    D B(a.N, tab);
    const int st = B.st;
    for (int j = threadIdx.x; j < 2 * S * 2 * D::PS; j += blockDim.x) (&xs[0][0][0])[j] = mk<double>(0, 0);
    const long e = (long)st * a.N + B.n;   // this thread's point
    double ps = 0, p0 = 0, Wv[S], Mv[S], wi = 0;
    if (B.own) {
        ps = reinterpret_cast<const double *>(psi + e)[B.comp];
        if (a.psi0) p0 = a.psi0[2 * e + B.comp];
        if (NIP) wi = (offset_i + (h.Wi[0] ? h.Wi[0][B.n] : 0.0)) * inv_scaling;
    }
#pragma unroll
    for (int j = 0; j < S; ++j) {
        Wv[j] = (B.own && h.W[st][j] ? h.W[st][j][B.n] : 0.0) + (j == st ? h.unity[st] : 0.0);
        Mv[j] = B.own && h.mu[st][j] ? h.mu[st][j][B.n] : 0.0;
    }
    const double sgn = B.comp ? -1.0 : 1.0;
    const int lane = threadIdx.x & 63;
    double acc = 0, last_acc = 0, norm0 = 0;
    int last = 1;
    bool broke = false;
    __syncthreads();
    for (int step = 0; step < a.nsteps; ++step) {
        double wv[S];
#pragma unroll
        for (int j = 0; j < S; ++j) {
            const double E = a.fields ? a.fields[((long)step * S + st) * S + j] : a.field0[st * S + j];
            wv[j] = Wv[j] + E * Mv[j];
        }
        double pm1 = ps, pm2 = 0;
        int buf = 0;
        B.put(pm1, xs[0][st], S > 1 ? full[0][st] : nullptr);
        dense_obs_put(ps, p0, B.comp, B.wave, ored);
        lds_barrier();
        norm0 = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) norm0 += ored[3 * w];
        if (a.obs && threadIdx.x < 3 * S) {
            const int s = threadIdx.x / 3, c = threadIdx.x - 3 * s;
            double t = 0;
            for (int w = 0; w < D::T / 64; ++w) t += ored[3 * (s * (D::T / 64) + w) + c];
            double *o = a.obs + (long)step * 4 * S;
            if (c == 0) {
                o[2 * s] = t;
                o[2 * s + 1] = 0;
            } else {
                o[2 * S + 2 * s + c - 1] = t;
            }
        }
        last = 1;
        last_acc = acc = 0;
        broke = false;
        double c0r = coef[0], c0i = coef[1];
        for (int k = 1; k < order; ++k) {
            const double ckr = coef[2 * k], cki = coef[2 * k + 1];
            double hp = B.apply(xs[buf][st]);
            if (k >= 3 && prec > 0) {
                // break test of order k - 1 (OCheby.cpp:179-182, 283-285)
                double t = 0;
#pragma unroll
                for (int w = 0; w < NW; ++w) t += red[buf][w];
                last_acc = acc;
                acc = t;
                if (IMAG ? (k >= 4 && fabs(acc - last_acc) / last_acc < prec) : fabs(norm0 - acc) / norm0 < prec) {
                    broke = true;
                    break;
                }
            }
            last = k;
#pragma unroll
            for (int j = 0; j < S; ++j) {
                double pj = pm1;
                if (S > 1 && j != st) pj = B.own ? reinterpret_cast<const double *>(full[buf][j] + B.n)[B.comp] : 0.0;
                hp += wv[j] * pj;
            }
            double b = (hp - offset * pm1) * inv_scaling;
            if (NIP) b += sgn * wi * dpp<kXor1>(pm1);
            double pk;
            if (IMAG) {
                pk = k == 1 ? -b : -2.0 * b - pm2;
            } else {
                const double bo = sgn * dpp<kXor1>(b);
                pk = k == 1 ? bo : 2.0 * bo + pm2;
            }
            if (!B.own) pk = 0;
            pm2 = pm1;
            pm1 = pk;
            buf ^= 1;
            B.put(pk, xs[buf][st], S > 1 ? full[buf][st] : nullptr);
            if (k == 1) {
                const double px = dpp<kXor1>(ps);
                ps = c0r * ps - sgn * c0i * px;
            }
            ps += ckr * pk - sgn * cki * dpp<kXor1>(pk);
            if (k >= 2 && (prec > 0 || k == order - 1)) {
                const double s = dpp_wave_sum(ps * ps);
                if (lane == 0) red[buf][B.wave] = s;
            }
            lds_barrier();
        }
        if (threadIdx.x == 0 && a.orders) a.orders[step] = last;
        lds_barrier();   // the next step's first writes follow the last reads
    }
    if (!broke && last >= 2) {
        double t = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) t += red[last & 1][w];
        last_acc = acc;
        acc = t;
    }
    if (threadIdx.x == 0) {
        // the outcome of the last step, where the per-order kernels leave it
        constexpr int NS = IMAG ? 3 : 2;
        ctl->norm0 = norm0;
        ctl->done = broke;
        ctl->accnorm = acc;
        ctl->last_order = last;
        partials[2 * kMaxPartials] = norm0;
        const int s0 = last % NS, s1 = (last + NS - 1) % NS;
        partials[(s0 == 2 ? 3 : s0) * kMaxPartials] = acc;
        if (IMAG) partials[(s1 == 2 ? 3 : s1) * kMaxPartials] = last_acc;
    }
    if (B.own) reinterpret_cast<double *>(psi + e)[B.comp] = ps;
}

// Split-operator steps exp(-i tau/2 W) exp(-i tau T) exp(-i tau/2 W) of a 1D
// line (OGSPO.cpp:114-139), W the product of the x-space operators: for one
// state, or several uncoupled ones, a phase per point, whose field part is
// formed once per step (the step's two halves share it); for two coupled
// states the 2 x 2 unitaries of the whole group.  exp(-i tau T) is the dense
// circulant matrix tab (re, im), 4 multiply-adds per element.  psi stays in
// registers over the steps.
// MU: one operator carries a field (one state); CPL: two coupled states.
template <int NB, int S, bool MU, bool CPL>
__global__ void __launch_bounds__(128 * NB * S) k_dense_gspo(XGroupDev<double> pre, XGroupDev<double> post, DenseRun a,
                                                             const double *tabr, const double *tabi,
                                                             cx<double> *__restrict__ psi) {
    using D = DenseLine<NB>;
    static_assert(!MU || S == 1, "field operators act on one state");
    static_assert(!CPL || S == 2, "two coupled states");
    __shared__ __align__(16) cx<double> xs[2][S][2 * D::PS];
    __shared__ __align__(16) cx<double> full[CPL ? 2 : 1][CPL ? 2 * D::MP : 1];
    constexpr int NW = D::T * S / 64;
    __shared__ double ored[2][3 * NW];
    D B(a.N, tabr);
    double ti[D::C + 3];
    {
        const D Bi(a.N, tabi);
#pragma unroll
        for (int m = 0; m < D::C + 3; ++m) ti[m] = Bi.tc[m];
    }
    const int st = B.st;
    for (int j = threadIdx.x; j < 2 * S * 2 * D::PS; j += blockDim.x) (&xs[0][0][0])[j] = mk<double>(0, 0);
    const long e = (long)st * a.N + B.n;
    const double sgn = B.comp ? -1.0 : 1.0;
    double ps = 0, p0 = 0, mu = 0;
    // the x-space groups on this point: phases of the own state (uncoupled),
    // or the full matrices Q = post and this state's row of P = pre
    cx<double> fs = mk<double>(1, 0), P[2], Q[2][2];
    if (B.own) {
        ps = reinterpret_cast<const double *>(psi + e)[B.comp];
        if (a.psi0) p0 = a.psi0[2 * e + B.comp];
        if constexpr (CPL) {
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                cx<double> v[2] = {mk<double>(c == 0, 0), mk<double>(c == 1, 0)}, u[2] = {v[0], v[1]};
                xgroup_point<double, 2>(post, B.n, v);
                Q[0][c] = v[0];
                Q[1][c] = v[1];
                xgroup_point<double, 2>(pre, B.n, u);
                P[c] = st ? u[1] : u[0];
            }
        } else {
            cx<double> v[S];
#pragma unroll
            for (int s = 0; s < S; ++s) v[s] = mk<double>(1, 0);
            for (int o = 0; o < pre.n; ++o) {
                XSplitDev<double> op = pre.op[o];
                if (MU && op.mu[0][0]) {
                    mu = op.tau * op.mu[0][0][B.n];
                    op.mu[0][0] = nullptr;   // the field part is formed per step
                    if (!op.V[0][0]) continue;
                }
                xsplit_point<double, S>(op, B.n, v);
            }
#pragma unroll
            for (int s = 0; s < S; ++s)
                if (s == st) fs = v[s];
        }
    }
    __syncthreads();
    for (int step = 0; step < a.nsteps; ++step) {
        const int buf = step & 1;
        cx<double> f = fs;
        if (MU) {
            double sn, cs;
            sincos(-mu * (a.fields ? a.fields[step] : a.field0[0]), &sn, &cs);
            f = cmul(f, mk<double>(cs, sn));
        }
        if (a.obs) dense_obs_put(ps, p0, B.comp, B.wave, ored[buf]);
        double v;
        if constexpr (CPL) {
            // own row of the pre group on both states of the point
            if (step == 0) {
                if (B.own) reinterpret_cast<double *>(full[st] + B.n)[B.comp] = ps;
                lds_barrier();
            }
            cx<double> w0 = mk<double>(0, 0), w1 = w0;
            if (B.own) {
                w0 = full[0][B.n];
                w1 = full[1][B.n];
                if (step > 0) {
                    const cx<double> y0 = w0, y1 = w1;
                    w0 = cmul(Q[0][0], y0) + cmul(Q[0][1], y1);
                    w1 = cmul(Q[1][0], y0) + cmul(Q[1][1], y1);
                }
            }
            const cx<double> z = cmul(P[0], w0) + cmul(P[1], w1);
            v = B.comp ? z.i : z.r;
        } else {
            v = f.r * ps - sgn * f.i * dpp<kXor1>(ps);
        }
        if (!B.own) v = 0;
        B.put(v, xs[buf][st], nullptr);
        lds_barrier();
        if (a.obs && threadIdx.x < 3 * S) {
            const int s = threadIdx.x / 3, c = threadIdx.x - 3 * s;
            double t = 0;
            for (int w = 0; w < D::T / 64; ++w) t += ored[buf][3 * (s * (D::T / 64) + w) + c];
            double *o = a.obs + (long)step * 4 * S;
            if (c == 0) {
                o[2 * s] = t;
                o[2 * s + 1] = 0;
            } else {
                o[2 * S + 2 * s + c - 1] = t;
            }
        }
        double y;
        {
            double ac[4][2] = {};
            const cx<double> *x = xs[buf][st] + B.par * D::PS + B.q;
#pragma unroll
            for (int c = 0; c < D::C; ++c) {
                const cx<double> w = x[8 * c];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const double tr = B.tc[r - c + D::C - 1], tm = ti[r - c + D::C - 1];
                    ac[r][0] = __builtin_fma(tr, w.r, __builtin_fma(-tm, w.i, ac[r][0]));
                    ac[r][1] = __builtin_fma(tr, w.i, __builtin_fma(tm, w.r, ac[r][1]));
                }
            }
            y = B.scatter(ac);
        }
        if constexpr (CPL) {
            if (B.own) reinterpret_cast<double *>(full[st] + B.n)[B.comp] = y;
            lds_barrier();
            if (B.own) {
                const cx<double> y0 = full[0][B.n], y1 = full[1][B.n];
                const cx<double> z = cmul(st ? Q[1][0] : Q[0][0], y0) + cmul(st ? Q[1][1] : Q[0][1], y1);
                ps = B.comp ? z.i : z.r;
            }
        } else {
            ps = f.r * y - sgn * f.i * dpp<kXor1>(y);
            if (!B.own) ps = 0;
        }
    }
    if (B.own) reinterpret_cast<double *>(psi + e)[B.comp] = ps;
}

// ---------------------------------------------------------------------------
// launchers

// row blocks of a line of N points for S states, 0: the line takes another
// path.  At most 1024 threads (128 nb S).
int dense_blocks(int N, int S, bool gspo) {
    if (N % 2 || N < 8 || S < 1 || S > kMaxStates) return 0;
    int nb = (N + 63) / 64;
    if (nb == 5) nb = 6;
    if (nb == 7) nb = 8;
    const int most = S == 1 ? (gspo ? 6 : 8) : S == 2 ? 4 : 2;
    return nb <= most ? nb : 0;
}

template <int NB, int S>
static void dense_cheby_NS(hipStream_t s, const HamDev<double> &h, const DenseRun &a, const double *tab,
                           const double *coef, int order, double offset, double offset_i, double inv_scaling,
                           double prec, bool nip, bool imag, double *psi, ChebyCtl *ctl, double *partials) {
    auto p = reinterpret_cast<cx<double> *>(psi);
    const dim3 threads(128 * NB * S);
    if (nip) {
        if constexpr (S == 1) {
            if (imag) throw std::runtime_error("negative imaginary potential: real time only");
            QDX_LAUNCH((k_dense_cheby<NB, 1, true, false>), dim3(1), threads, 0, s, h, a, tab, coef, order, offset,
                       offset_i, inv_scaling, prec, p, ctl, partials);
        } else {
            throw std::runtime_error("negative imaginary potential: single-state Hamiltonians only");
        }
    } else if (imag) {
        QDX_LAUNCH((k_dense_cheby<NB, S, false, true>), dim3(1), threads, 0, s, h, a, tab, coef, order, offset, 0.0,
                   inv_scaling, prec, p, ctl, partials);
    } else {
        QDX_LAUNCH((k_dense_cheby<NB, S, false, false>), dim3(1), threads, 0, s, h, a, tab, coef, order, offset, 0.0,
                   inv_scaling, prec, p, ctl, partials);
    }
    QDX_HIP(hipGetLastError());
}

template <int NB, int S>
static void dense_gspo_NS(hipStream_t s, const XGroupDev<double> &pre, const XGroupDev<double> &post,
                          const DenseRun &a, const double *tabr, const double *tabi, bool mu, bool coupled,
                          double *psi) {
    auto p = reinterpret_cast<cx<double> *>(psi);
    const dim3 threads(128 * NB * S);
    if (mu) {
        if constexpr (S == 1)
            QDX_LAUNCH((k_dense_gspo<NB, 1, true, false>), dim3(1), threads, 0, s, pre, post, a, tabr, tabi, p);
        else throw std::runtime_error("field split operators act on one state");
    } else if (coupled) {
        if constexpr (S == 2)
            QDX_LAUNCH((k_dense_gspo<NB, 2, false, true>), dim3(1), threads, 0, s, pre, post, a, tabr, tabi, p);
        else throw std::runtime_error("coupled split operators: two states");
    } else {
        QDX_LAUNCH((k_dense_gspo<NB, S, false, false>), dim3(1), threads, 0, s, pre, post, a, tabr, tabi, p);
    }
    QDX_HIP(hipGetLastError());
}

// CALL with NB and SS as constants
#define QDX_DISPATCH_DENSE(NB_, S_, GSPO_, CALL)                                    \
    switch (S_ * 16 + NB_) {                                                        \
    case 17: { constexpr int NB = 1, SS = 1; CALL; } break;                         \
    case 18: { constexpr int NB = 2, SS = 1; CALL; } break;                         \
    case 19: { constexpr int NB = 3, SS = 1; CALL; } break;                         \
    case 20: { constexpr int NB = 4, SS = 1; CALL; } break;                         \
    case 22: { constexpr int NB = 6, SS = 1; CALL; } break;                         \
    case 24: { constexpr int NB = GSPO_ ? 6 : 8, SS = 1; CALL; } break;             \
    case 33: { constexpr int NB = 1, SS = 2; CALL; } break;                         \
    case 34: { constexpr int NB = 2, SS = 2; CALL; } break;                         \
    case 35: { constexpr int NB = 3, SS = 2; CALL; } break;                         \
    case 36: { constexpr int NB = 4, SS = 2; CALL; } break;                         \
    case 49: { constexpr int NB = 1, SS = 3; CALL; } break;                         \
    case 50: { constexpr int NB = 2, SS = 3; CALL; } break;                         \
    case 65: { constexpr int NB = 1, SS = 4; CALL; } break;                         \
    case 66: { constexpr int NB = 2, SS = 4; CALL; } break;                         \
    default: throw std::runtime_error("dense line kernel: line too long");          \
    }

void launch_dense_cheby(hipStream_t s, int S, const HamDev<double> &h, const DenseRun &a, const double *tab,
                        const double *coef, int order, double offset, double offset_i, double inv_scaling, double prec,
                        bool imag, double *psi, ChebyCtl *ctl, double *partials) {
    const int nb = dense_blocks(a.N, S, false);
    const bool nip = offset_i != 0 || h.Wi[0] != nullptr;
    QDX_DISPATCH_DENSE(nb, S, false, (dense_cheby_NS<NB, SS>(s, h, a, tab, coef, order, offset, offset_i, inv_scaling,
                                                             prec, nip, imag, psi, ctl, partials)));
}

void launch_dense_gspo(hipStream_t s, int S, const XGroupDev<double> &pre, const XGroupDev<double> &post,
                       const DenseRun &a, const double *tabr, const double *tabi, bool mu, bool coupled,
                       double *psi) {
    const int nb = dense_blocks(a.N, S, true);
    QDX_DISPATCH_DENSE(nb, S, true, (dense_gspo_NS<NB, SS>(s, pre, post, a, tabr, tabi, mu, coupled, psi)));
}

}  // namespace qdx

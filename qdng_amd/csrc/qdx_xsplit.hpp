// The x-space split operators of GSPO on one grid point (included by
// qdx_gspo.hip and qdx_dense.hip).
#pragma once

#include "qdx_kernels_common.hpp"

namespace qdx {

// ---------------------------------------------------------------------------
// GSPO x-space split operators on one grid point (all states):
//   psi <- exp(-i tau W(x)) psi, W real symmetric (ODSpace.h:65-69,
//   OGridDipole.cpp:83-87, ODMultistate.cpp:109-159 / TransformMSD.cpp:31-101)
template <class R, int S, bool IMAG = false>
__device__ __forceinline__ void xsplit_point(const XSplitDev<R> &op, long gi, cx<double> (&v)[S]) {
    if (!IMAG && op.U) {   // the table of a time-independent operator
        auto u = [&](int c) {
            const double *q = op.U + 2 * ((long)c * op.n + gi);
            return mk<double>(q[0], q[1]);
        };
        if (S == 2 && op.coupled) {
            const cx<double> u00 = u(0), u01 = u(1), u11 = u(2);
            const cx<double> a0 = cmul(u00, v[0]) + cmul(u01, v[1]);
            const cx<double> a1 = cmul(u01, v[0]) + cmul(u11, v[1]);
            v[0] = a0;
            v[1] = a1;
        } else {
#pragma unroll
            for (int i = 0; i < S; ++i) v[i] = cmul(v[i], u(i));
        }
        return;
    }
    double Wm[S][S];
#pragma unroll
    for (int i = 0; i < S; ++i)
#pragma unroll
        for (int j = 0; j < S; ++j) {
            double w = 0;
            if (op.V[i][j]) w += (double)op.V[i][j][gi];
            if (op.mu[i][j]) w += op.Edip[i][j] * (double)op.mu[i][j][gi];
            Wm[i][j] = w;
        }
    if (!op.coupled || S == 1) {
#pragma unroll
        for (int i = 0; i < S; ++i) {
            if (IMAG) {   // exp(-tau w), imaginary time
                const double f = exp(-op.tau * Wm[i][i]);
                v[i] = mk<double>(v[i].r * f, v[i].i * f);
                continue;
            }
            double sn, cs;
            sincos(-op.tau * Wm[i][i], &sn, &cs);
            v[i] = cmul(v[i], mk<double>(cs, sn));
        }
        return;
    }
    if constexpr (S == 2) {
        if (IMAG) {
            // exp(-tau W) = e^{-tau m} [cosh(tau O) - sinh(tau O)/O (W - m)]
            const double m = 0.5 * (Wm[0][0] + Wm[1][1]);
            const double d = 0.5 * (Wm[0][0] - Wm[1][1]);
            const double b = Wm[0][1];
            const double O = sqrt(d * d + b * b);
            const double ch = cosh(op.tau * O);
            const double sh = O > 0 ? sinh(op.tau * O) / O : op.tau;
            const double e = exp(-op.tau * m);
            const double u00 = e * (ch - sh * d), u11 = e * (ch + sh * d), u01 = -e * sh * b;
            const cx<double> a0 = mk<double>(u00 * v[0].r + u01 * v[1].r, u00 * v[0].i + u01 * v[1].i);
            const cx<double> a1 = mk<double>(u01 * v[0].r + u11 * v[1].r, u01 * v[0].i + u11 * v[1].i);
            v[0] = a0;
            v[1] = a1;
            return;
        }
        // exp(-i tau W) = e^{-i tau m} [cos(tau O) - i sin(tau O)/O (W - m)]
        const double m = 0.5 * (Wm[0][0] + Wm[1][1]);
        const double d = 0.5 * (Wm[0][0] - Wm[1][1]);
        const double b = Wm[0][1];
        const double O = sqrt(d * d + b * b);
        double so, c;
        sincos(op.tau * O, &so, &c);
        const double sc = O > 0 ? so / O : op.tau;
        double sm, cm;
        sincos(-op.tau * m, &sm, &cm);
        const cx<double> ph = mk<double>(cm, sm);
        const cx<double> u00 = mk<double>(c, -sc * d), u11 = mk<double>(c, sc * d);
        const cx<double> u01 = mk<double>(0, -sc * b);
        const cx<double> a0 = cmul(u00, v[0]) + cmul(u01, v[1]);
        const cx<double> a1 = cmul(u01, v[0]) + cmul(u11, v[1]);
        v[0] = cmul(ph, a0);
        v[1] = cmul(ph, a1);
    }
}

template <class R, int S, bool IMAG = false>
__device__ __forceinline__ void xgroup_point(const XGroupDev<R> &grp, long gi, cx<double> (&v)[S]) {
    for (int o = 0; o < grp.n; ++o) xsplit_point<R, S, IMAG>(grp.op[o], gi, v);
}

}  // namespace qdx

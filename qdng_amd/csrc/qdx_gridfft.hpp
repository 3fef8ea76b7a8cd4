// Line filters of the persistent grid kernels and of the kinetic pass of larger
// grids: IFFT . diag(f) . FFT of lines of N = 8 m points, 8 points per thread.
// Also the DPP and barrier helpers that the dense 1D kernels share.
//
// With n = n1 m + n2 and k = k1 + 8 k2 the transform is a radix-8 stage over
// n1 on registers (thread lt owns the points lt + q m), a twiddle, and for
// each k1 an m-point transform over n2, taken as m = R2 R3 in two stages
// through LDS.  Forward stages decimate in frequency and the inverse ones
// undo them in reverse order, so every butterfly writes the places it read:
// one LDS buffer, one barrier between stages, no reordering, and the factors
// f are applied in registers between the two middle stages.  The inverse runs
// on swapped real and imaginary parts, which makes it the same forward
// butterflies.  Bound by LDS latency (one wave per SIMD: 8 reads of 16 bytes
// take 470 cycles, the butterfly behind them 330; in a run on 512 x 512 points
// vector instructions issue in 22 % of the wave cycles, and bank conflicts take
// 0.3 cycles per LDS instruction).  Against the Stockham
// stages of fft_line (4 points per thread, two buffers, run-time strides) the
// filter of four 512-point lines per block went from 5.7 to 4.4 us; an order
// of a Chebyshev series on 240 x 176 points from 29.2 to 16.5 us.
#pragma once

#include "qdx_kernels_common.hpp"

namespace qdx {

// a barrier that orders LDS only: global accesses in flight stay so
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// value of another lane by a DPP control word
template <int CTRL>
__device__ __forceinline__ double dpp(double x) {
    const int lo = __double2loint(x), hi = __double2hiint(x);
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, CTRL, 0xf, 0xf, false),
                            __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}
constexpr int kXor1 = 0xB1;          // quad_perm [1, 0, 3, 2]
constexpr int kXor2 = 0x4E;          // quad_perm [2, 3, 0, 1]
constexpr int kXor7 = 0x141;         // row_half_mirror
constexpr int kXor15 = 0x140;        // row_mirror
constexpr int kXor8 = 0x128;         // row_ror:8

// sum over the wave, in every lane: 16-lane rows by DPP, then the four rows
// (six dependent LDS permutes in wave_sum)
__device__ __forceinline__ double dpp_wave_sum(double v) {
    v += dpp<kXor1>(v);
    v += dpp<kXor2>(v);
    v += dpp<kXor7>(v);
    v += dpp<kXor15>(v);
    const int lo = __double2loint(v), hi = __double2hiint(v);
    double t = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        t += __hiloint2double(__builtin_amdgcn_readlane(hi, 16 * r), __builtin_amdgcn_readlane(lo, 16 * r));
    return t;
}

// cos and sin of 2 pi k / r, k = 1, 2, ...
template <int r>
struct Roots;
// An opaque zero.  Constants read at an index that holds it are loaded (scalar)
// where they are used: as literals the compiler hoists them out of the order
// loop for every radix at once, hundreds of scalar registers that spill.
__device__ __forceinline__ int opaque_zero() {
    int z = 0;
    asm volatile("" : "+s"(z));
    return z;
}
template <>
struct Roots<9> {
    static constexpr double c[] = {
        0.76604444311897803520, 0.17364817766693034885, -0.50000000000000000000, -0.93969262078590838405};
    static constexpr double s[] = {
        0.64278760968653932632, 0.98480775301220805937, 0.86602540378443864676, 0.34202014332566873304};
};
template <>
struct Roots<16> {
    static constexpr double c[] = {
        0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.00000000000000000000,
        -0.38268343236508977173, -0.70710678118654752440, -0.92387953251128675613, -1.00000000000000000000,
        -0.92387953251128675613};
    static constexpr double s[] = {
        0.38268343236508977173, 0.70710678118654752440, 0.92387953251128675613, 1.00000000000000000000,
        0.92387953251128675613, 0.70710678118654752440, 0.38268343236508977173, 0.00000000000000000000,
        -0.38268343236508977173};
};
// the same of odd primes as device data: cosines, then sines
#define QDX_PRIME_ROOTS(r_, ...)                                                   \
    __constant__ const double k_roots64_##r_[] = {__VA_ARGS__};                     \
    __constant__ const float k_roots32_##r_[] = {__VA_ARGS__};                      \
    template <>                                                                     \
    __device__ __forceinline__ const double *prime_roots<r_, double>() {            \
        return k_roots64_##r_;                                                      \
    }                                                                               \
    template <>                                                                     \
    __device__ __forceinline__ const float *prime_roots<r_, float>() {              \
        return k_roots32_##r_;                                                      \
    }
template <int r, class R>
__device__ const R *prime_roots();
QDX_PRIME_ROOTS(5, 0.30901699437494742410, -0.80901699437494742410, 0.95105651629515357212, 0.58778525229247312917)
QDX_PRIME_ROOTS(7, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624,
                0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048)
QDX_PRIME_ROOTS(11, 0.84125353283118116886, 0.41541501300188642553, -0.14231483827328514044,
                -0.65486073394528506406, -0.95949297361449738989, 0.54064081745559758211,
                0.90963199535451837141, 0.98982144188093273238, 0.75574957435425828377, 0.28173255684142969771)
QDX_PRIME_ROOTS(13, 0.88545602565320989590, 0.56806474673115580251, 0.12053668025532305335, -0.35460488704253562597,
                -0.74851074817110109863, -0.97094181742605202716, 0.46472317204376854566,
                0.82298386589365639458, 0.99270887409805399280, 0.93501624268541482344, 0.66312265824079520238,
                0.23931566428755776715)
QDX_PRIME_ROOTS(17, 0.93247222940435580457, 0.73900891722065911592, 0.44573835577653826740, 0.09226835946330199524,
                -0.27366299007208286354, -0.60263463637925638918, -0.85021713572961415213,
                -0.98297309968390177828, 0.36124166618715294874, 0.67369564364655721171, 0.89516329135506232207,
                0.99573417629503452187, 0.96182564317281907041, 0.79801722728023950333, 0.52643216287735580024,
                0.18374951781657033157)
QDX_PRIME_ROOTS(19, 0.94581724170063467902, 0.78914050939639359922, 0.54694815812242687471, 0.24548548714079914892,
                -0.08257934547233232460, -0.40169542465296945752, -0.67728157162574107476,
                -0.87947375120648907139, -0.98636130340272237360, 0.32469946920468348741,
                0.61421271268966781744, 0.83716647826252857481, 0.96940026593933041674, 0.99658449300666984982,
                0.91577332665505743992, 0.73572391067313162477, 0.47594739303707354443, 0.16459459028073389414)
QDX_PRIME_ROOTS(23, 0.96291728734779929502, 0.85441940454648855255, 0.68255314321865408287, 0.46006503773115212604,
                0.20345601305263378988, -0.06824241336467097592, -0.33487961217098615196,
                -0.57668032211486714125, -0.77571129070441980704, -0.91721130150545301784,
                -0.99068594603633075234, 0.26979677115702427125, 0.51958395003543357813, 0.73083596427812410165,
                0.88788521840237523498, 0.97908408768232287563, 0.99766876919053919845, 0.94226092211882049562,
                0.81696989301044201697, 0.63108794432605278937, 0.39840108984624145800, 0.13616664909624659076)
QDX_PRIME_ROOTS(29, 0.97662055571008668321, 0.90757541967095705362, 0.79609306570564374600, 0.64738628478182763918,
                0.46840844069979013922, 0.26752833852922082119, 0.05413890858541752615, -0.16178199655276472654,
                -0.37013815533991435686, -0.56118706536238236927, -0.72599549192313085814,
                -0.85685717616758924452, -0.94765317118280244427, -0.99413795715435960896,
                0.21497044021102406718, 0.41988910156026457697, 0.60517421519376516592, 0.76216205512763646326,
                0.88351204444602292283, 0.96354999251922296004, 0.99853341385112386457, 0.98682652254152615177,
                0.92897671981679144179, 0.82768899815689055614, 0.68769945885342329308, 0.51555385717702173971,
                0.31930153013597997320, 0.10811901842394176303)
QDX_PRIME_ROOTS(31, 0.97952994125249449394, 0.91895781162023062913, 0.82076344120727632636, 0.68896691907568656780,
                0.52896401032696245737, 0.34730525284482028554, 0.15142777750457666366, -0.05064916883871271228,
                -0.25065253225872053931, -0.44039415155763430952, -0.61210598254766284415,
                -0.75875812269279090191, -0.87434661614458211883, -0.95413925640004885148,
                -0.99486932339189514632, 0.20129852008866007914, 0.39435585511331858010, 0.57126821509479227916,
                0.72479278722911995887, 0.84864425749475095046, 0.93775213214708045843, 0.98846832432811139916,
                0.99871650717105280715, 0.96807711886620430515, 0.89780453957074165714, 0.79077573693769858208,
                0.65137248272222220745, 0.48530196253108102521, 0.29936312297335795401, 0.10116832198743217779)
#undef QDX_PRIME_ROOTS

// X[u] = sum_t x[t] exp(-2 pi i t u / RR) for an odd prime RR by the sums and
// differences of the pairs t, RR - t; put(u, X[u]) takes the results as they
// come
template <int RR, class R, class Put>
__device__ __forceinline__ void prime_dft(const cx<R> *x, Put put) {
    constexpr int H = (RR - 1) / 2;
    const R *cs = prime_roots<RR, R>() + opaque_zero();
    R cw[2 * H];
#pragma unroll
    for (int t = 0; t < 2 * H; ++t) cw[t] = cs[t];
    cx<R> s[H], d[H], y0 = x[0];
    const cx<R> x0 = x[0];
#pragma unroll
    for (int t = 0; t < H; ++t) {
        s[t] = x[t + 1] + x[RR - 1 - t];
        d[t] = x[t + 1] - x[RR - 1 - t];
        y0 = y0 + s[t];
    }
    put(0, y0);
#pragma unroll
    for (int u = 1; u <= H; ++u) {
        cx<R> a = x0, b = mk<R>(0, 0);
#pragma unroll
        for (int t = 0; t < H; ++t) {
            const int q = (u * (t + 1)) % RR;
            const R c = cw[(q <= H ? q : RR - q) - 1];
            const R w = q <= H ? cw[H + q - 1] : -cw[H + RR - q - 1];
            a.r = __builtin_fma(c, s[t].r, a.r);
            a.i = __builtin_fma(c, s[t].i, a.i);
            b.r = __builtin_fma(w, d[t].r, b.r);
            b.i = __builtin_fma(w, d[t].i, b.i);
        }
        // a - i b and a + i b
        put(u, mk<R>(a.r + b.i, a.i - b.r));
        put(RR - u, mk<R>(a.r - b.i, a.i + b.r));
    }
}

// the same for any radix, natural order, in place
template <int RR, class R>
struct Dft {
    static __device__ __forceinline__ void run(cx<R> *x) {
        prime_dft<RR, R>(x, [&](int u, cx<R> y) { x[u] = y; });
    }
};
// exp(-2 pi i q / RR) on x
template <int RR, class R>
__device__ __forceinline__ cx<R> root_mul(cx<R> x, int q) {
    constexpr int H = sizeof(Roots<RR>::c) / sizeof(double);
    if (q == 0) return x;
    return cmul(x, q <= H ? mk<R>((R)Roots<RR>::c[q - 1], (R)-Roots<RR>::s[q - 1])
                          : mk<R>((R)Roots<RR>::c[RR - q - 1], (R)Roots<RR>::s[RR - q - 1]));
}
template <class R>
struct Dft<1, R> {
    static __device__ __forceinline__ void run(cx<R> *) {}
};
#define QDX_DFT_BFLY(RR_)                                                                        \
    template <class R>                                                                           \
    struct Dft<RR_, R> {                                                                         \
        static __device__ __forceinline__ void run(cx<R> *x) { Bfly<RR_, R>::run(x, -1); }       \
    };
QDX_DFT_BFLY(2)
QDX_DFT_BFLY(3)
QDX_DFT_BFLY(4)
QDX_DFT_BFLY(8)
#undef QDX_DFT_BFLY
// coprime A, B: t = B t1 + A t2, u = the remainders u1 mod A, u2 mod B
template <int A, int B, class R>
struct DftCoprime {
    static __device__ __forceinline__ void run(cx<R> *x) {
        constexpr int RR = A * B;
        cx<R> y[A][B];
#pragma unroll
        for (int t2 = 0; t2 < B; ++t2) {
            cx<R> z[A];
#pragma unroll
            for (int t1 = 0; t1 < A; ++t1) z[t1] = x[(B * t1 + A * t2) % RR];
            Dft<A, R>::run(z);
#pragma unroll
            for (int u1 = 0; u1 < A; ++u1) y[u1][t2] = z[u1];
        }
#pragma unroll
        for (int u1 = 0; u1 < A; ++u1) {
            Dft<B, R>::run(y[u1]);
#pragma unroll
            for (int u = 0; u < RR; ++u)
                if (u % A == u1) x[u] = y[u1][u % B];
        }
    }
};
// A x A: t = t1 A + t2, u = u1 + A u2
template <int A, class R>
struct DftSquare {
    static __device__ __forceinline__ void run(cx<R> *x) {
        cx<R> y[A][A];
#pragma unroll
        for (int t2 = 0; t2 < A; ++t2) {
            cx<R> z[A];
#pragma unroll
            for (int t1 = 0; t1 < A; ++t1) z[t1] = x[t1 * A + t2];
            Dft<A, R>::run(z);
#pragma unroll
            for (int u1 = 0; u1 < A; ++u1) y[u1][t2] = root_mul<A * A>(z[u1], u1 * t2);
        }
#pragma unroll
        for (int u1 = 0; u1 < A; ++u1) {
            Dft<A, R>::run(y[u1]);
#pragma unroll
            for (int u2 = 0; u2 < A; ++u2) x[u1 + A * u2] = y[u1][u2];
        }
    }
};
template <class R>
struct Dft<6, R> : DftCoprime<2, 3, R> {};
template <class R>
struct Dft<10, R> : DftCoprime<2, 5, R> {};
template <class R>
struct Dft<12, R> : DftCoprime<4, 3, R> {};
template <class R>
struct Dft<14, R> : DftCoprime<2, 7, R> {};
template <class R>
struct Dft<15, R> : DftCoprime<3, 5, R> {};
template <class R>
struct Dft<9, R> : DftSquare<3, R> {};
template <class R>
struct Dft<16, R> : DftSquare<4, R> {};

// One axis of a filter as a thread sees it.  Place (k1, a, b) of a line,
// a < R2, b < R3, is element ((k1 R2 + a) RS + b) nl of the line's buffer, RS
// = R3 made odd (consecutive butterflies of the R3 stage fall on different
// banks); nl lines are interleaved.
template <class R>
struct GridAxis {
    int m, R2, R3, RS, nl;
    int lt, a, b;         // n2 of the thread's points, lt = a R3 + b
    bool on;              // it has points of a line
    cx<R> *buf;           // its line
    const cx<R> *tw1;     // exp(-2 pi i k1 n2 / N) at (k1 - 1) m + n2
    const cx<R> *tw2;     // exp(-2 pi i a b / m) at a R3 + b
};
__host__ __device__ constexpr int grid_rs(int R3) { return R3 | 1; }
// elements of one line's buffer (and of a factor table)
__host__ __device__ constexpr int grid_line_len(int R2, int R3) { return 8 * R2 * grid_rs(R3); }
// elements of the twiddle tables
__host__ __device__ constexpr int grid_tw_len(int m) { return 7 * m + m; }

// tables of an axis from tab = exp(-2 pi i q / N), by the whole block
template <class R>
__device__ __forceinline__ void grid_tables(const cx<R> *tab, int m, int R3, cx<R> *tw1, cx<R> *tw2) {
    const int N = 8 * m;
    for (int i = threadIdx.x; i < 7 * m; i += blockDim.x) {
        const int k1 = i / m + 1, n2 = i % m;
        tw1[i] = tab[(k1 * n2) % N];
    }
    for (int i = threadIdx.x; i < m; i += blockDim.x) tw2[i] = tab[(8 * (i / R3) * (i % R3)) % N];
}
// factors f[k] (already scaled by g) at the places of k, by the whole block
__device__ __forceinline__ double scaled_factor(double f, double g) { return f * g; }
__device__ __forceinline__ cx<double> scaled_factor(cx<double> f, double g) { return mk<double>(f.r * g, f.i * g); }
template <class F>
__device__ __forceinline__ void grid_factors(const F *f, double g, int R2, int R3, F *dst) {
    const int RS = grid_rs(R3), m = R2 * R3;
    for (int i = threadIdx.x; i < 8 * m; i += blockDim.x) {
        const int k1 = i / m, a = (i % m) / R3, b = i % R3;
        dst[(k1 * R2 + a) * RS + b] = f ? scaled_factor(f[k1 + 8 * (a + R2 * b)], g) : F{};
    }
}

template <class R>
__device__ __forceinline__ cx<R> swapped(cx<R> a) {
    return mk<R>(a.i, a.r);
}
// the factor of a filter at a place: real (T) or complex (exp(-i tau T))
template <class R>
__device__ __forceinline__ cx<R> factor_mul(cx<R> x, double f) {
    return mk<R>((R)((double)x.r * f), (R)((double)x.i * f));
}
template <class R>
__device__ __forceinline__ cx<R> factor_mul(cx<R> x, cx<double> f) {
    return from_d<R>(cmul(to_d(x), f));
}

// Loads that are needed later are issued ahead of the butterflies (the
// compiler would read each twiddle right before its product, one LDS round
// trip after the other).
__device__ __forceinline__ void loads_first() { __builtin_amdgcn_sched_barrier(0); }

// stage over a: butterflies (k1, b), with the twiddle after it (forward) or
// before it (inverse)
template <int RR, class R>
__device__ __forceinline__ void grid_stage2(const GridAxis<R> &A, bool inv) {
    const int st = A.RS * A.nl, w3 = A.R3;
    int k1 = A.a, b = A.b;
    asm volatile("" : "+v"(k1), "+v"(b));   // addresses are formed here, not kept for every radix
    const cx<R> *tw = A.tw2 + b;
#pragma unroll 1
    for (; k1 < 8; k1 += RR) {
        cx<R> *p = A.buf + (k1 * RR * A.RS + b) * A.nl;
        cx<R> x[RR];
#pragma unroll
        for (int t = 0; t < RR; ++t) x[t] = p[t * st];
        if constexpr (RR >= 11 && RR % 2 && RR != 15) {
            // results go out one by one (registers)
            if (inv) {
#pragma unroll
                for (int t = 1; t < RR; ++t) x[t] = cmul(x[t], tw[t * w3]);
            }
            prime_dft<RR, R>(x, [&](int u, cx<R> y) { p[u * st] = inv || u == 0 ? y : cmul(y, tw[u * w3]); });
        } else {
            constexpr bool PRE = RR <= 8;   // (registers)
            cx<R> w[PRE ? RR : 1];
            if (PRE) {
#pragma unroll
                for (int t = 1; t < RR; ++t) w[t] = tw[t * w3];
                loads_first();
            }
            if (inv) {
#pragma unroll
                for (int t = 1; t < RR; ++t) x[t] = cmul(x[t], PRE ? w[PRE ? t : 0] : tw[t * w3]);
            }
            Dft<RR, R>::run(x);
            if (!inv) {
#pragma unroll
                for (int t = 1; t < RR; ++t) x[t] = cmul(x[t], PRE ? w[PRE ? t : 0] : tw[t * w3]);
            }
#pragma unroll
            for (int t = 0; t < RR; ++t) p[t * st] = x[t];
        }
    }
}
// stages over b with the factors between them: butterflies (k1, a)
template <int RR, class R, class F>
__device__ __forceinline__ void grid_stage3(const GridAxis<R> &A, const F *f) {
    const int rs = grid_rs(RR);
    int j = A.lt;
    asm volatile("" : "+v"(j));
#pragma unroll 1
    for (; j < 8 * A.R2; j += A.m) {
        cx<R> *p = A.buf + j * rs * A.nl;
        const F *g = f + j * rs;
        cx<R> x[RR];
        constexpr bool PRE = RR <= 8;
        F fx[PRE ? RR : 1];
#pragma unroll
        for (int t = 0; t < RR; ++t) x[t] = p[t * A.nl];
        if (PRE) {
#pragma unroll
            for (int t = 0; t < RR; ++t) fx[t] = g[t];
            loads_first();
        }
#pragma unroll 1
        for (int half = 0; half < 2; ++half) {
            Dft<RR, R>::run(x);
            if (half == 0) {
#pragma unroll
                for (int t = 0; t < RR; ++t) x[t] = swapped(factor_mul(x[t], PRE ? fx[PRE ? t : 0] : g[t]));
            }
        }
#pragma unroll
        for (int t = 0; t < RR; ++t) p[t * A.nl] = x[t];
    }
}

// v <- IFFT f FFT v (unnormalised: f holds 1/N).  Every thread of the block
// calls it.  f: the factors of the line's state.  PRIMES: radices of primes
// above 7 occur (instances of their own: they need more registers).  before, after: called ahead
// of and behind the barrier that follows the first stage through LDS.
template <bool PRIMES, class R, class F, class Before, class After>
__device__ __forceinline__ void grid_filter(cx<R> (&v)[8], const GridAxis<R> &A, const F *f, Before before,
                                            After after) {
    cx<R> *p = A.buf + (A.a * A.RS + A.b) * A.nl;
    const int st = A.R2 * A.RS * A.nl;
    const cx<R> *tw = A.tw1 + A.lt;
    cx<R> w[8];
    if (A.on) {
#pragma unroll
        for (int q = 1; q < 8; ++q) w[q] = tw[(q - 1) * A.m];
        loads_first();
        Bfly<8, R>::run(v, -1);
#pragma unroll
        for (int q = 1; q < 8; ++q) v[q] = cmul(v[q], w[q]);
#pragma unroll
        for (int q = 0; q < 8; ++q) p[q * st] = v[q];
    }
    lds_barrier();
#define QDX_STAGE2(RR_) \
    case RR_: grid_stage2<RR_, R>(A, inv); break;
#define QDX_STAGE3(RR_) \
    case RR_: grid_stage3<RR_, R>(A, f); break;
#define QDX_STAGE2P(RR_) \
    case RR_: if constexpr (PRIMES) grid_stage2<RR_, R>(A, inv); break;
#define QDX_STAGE3P(RR_) \
    case RR_: if constexpr (PRIMES) grid_stage3<RR_, R>(A, f); break;
#pragma unroll 1
    for (int inv = 0; inv < 2; ++inv) {
        if (A.R2 > 1) {
            if (A.on) {
                switch (A.R2) {
                    QDX_STAGE2(2)
                    QDX_STAGE2(3)
                    QDX_STAGE2(4)
                    QDX_STAGE2(5)
                    QDX_STAGE2(6)
                    QDX_STAGE2(7)
                    QDX_STAGE2(8)
                    QDX_STAGE2(9)
                    QDX_STAGE2(10)
                    QDX_STAGE2P(11)
                    QDX_STAGE2(12)
                    QDX_STAGE2P(13)
                    QDX_STAGE2(14)
                    QDX_STAGE2(15)
                    QDX_STAGE2(16)
                    QDX_STAGE2P(17)
                    QDX_STAGE2P(19)
                    QDX_STAGE2P(23)
                    QDX_STAGE2P(29)
                    QDX_STAGE2P(31)
                default: break;
                }
            }
            if (inv == 0) before();
            lds_barrier();
            if (inv == 0) after();
        }
        if (inv) break;
        if (A.on) {
            switch (A.R3) {
                QDX_STAGE3(1)
                QDX_STAGE3(2)
                QDX_STAGE3(3)
                QDX_STAGE3(4)
                QDX_STAGE3(5)
                QDX_STAGE3(6)
                QDX_STAGE3(7)
                QDX_STAGE3(8)
                QDX_STAGE3(9)
                QDX_STAGE3(10)
                QDX_STAGE3P(11)
                QDX_STAGE3(12)
                QDX_STAGE3P(13)
                QDX_STAGE3(14)
                QDX_STAGE3(15)
            default: grid_stage3<16, R>(A, f); break;
            }
        }
        if (A.R2 == 1) before();
        lds_barrier();
        if (A.R2 == 1) after();
    }
#undef QDX_STAGE2
#undef QDX_STAGE3
#undef QDX_STAGE2P
#undef QDX_STAGE3P
    if (A.on) {
#pragma unroll
        for (int q = 1; q < 8; ++q) w[q] = tw[(q - 1) * A.m];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = p[q * st];
        loads_first();
#pragma unroll
        for (int q = 1; q < 8; ++q) v[q] = cmul(v[q], w[q]);
        Bfly<8, R>::run(v, -1);
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = swapped(v[q]);
    }
}

}  // namespace qdx

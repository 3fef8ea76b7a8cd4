// gfx950 persistent kernels of 2D grids that fit the chip's registers: whole
// Chebyshev and split-operator runs in one launch.
//
// A 2D grid of up to 2^19 points times states is bound by latency when every
// order is two launches (row kernel and column pass): each of them reads its
// operands back from memory, fills the chip with only two waves per SIMD and
// drains (512 x 512 points, two states: 36 us per order in FP64, 25 in FP32;
// here 19.5 and 14, of which the two filters take 9 and the two exchanges of
// 8.4 MB 7).  Here every block keeps its rows of psi, phi_{k-1}, phi_{k-2} and of
// the surfaces in registers over all orders and steps; only the kinetic part
// along dimension 1 travels: phi_{k-1} to the owners of the columns, its
// filtered lines back to the owners of the rows.
//
// Block b owns rows [b rb, (b + 1) rb) of every state and the columns
// [b cw, (b + 1) cw) of every state; lanes run over the lines first (row: l =
// r S + st, column: l = c S + st), then over the points of a line.  The two
// exchange buffers hold one chunk of S rb cw values per (row block, column
// block) pair, column-block major for phi (A) and row-block major for the way
// back (B), so that both sides move whole chunks.
//
// Order of an iteration: store phi to A, filter the own rows along dimension 0
// (hides the exchange), signaling on the way, wait for all row blocks, load the own
// columns, filter, store to B, signal, wait for all column blocks, load,
// epilogue.  Chunks move with agent-scope (sc1) stores and loads, which go
// past the XCDs' private L2s: no cache write-back or invalidation is needed,
// only the store counter before the block's flag is raised.  Flags hold
// epochs that grow over all launches of a propagator.
//
// All blocks have to be on the chip together: there are at most as many as
// CUs, each fits a CU by itself, and the host lets no more such launches run at a
// time, per device and process, than their blocks have CUs.  (Cooperative
// launches would say so to the runtime, but they cost 20 us more, and once a
// process has made one its other streams run slower: a batch of jobs 34 -> 45
// ms.)  Other processes on the
// GPU can still hold CUs, so every wait is bounded (kGridWait): a block that
// gives up leaves, the others follow, and the host, which keeps psi until the
// launch is known to be complete, runs its steps again order by order.
#include "qdx_gridfft.hpp"
#include "qdx_xsplit.hpp"

namespace qdx {

// bound of one wait in ticks of the 100 MHz wall clock: 0.1 s
constexpr unsigned long long kGridWait = 10000000ull;

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
constexpr int kAgentScope = 16;   // sc1 of the buffer instructions' cache policy

// a place past the end of every exchange buffer: the buffer instructions read 0
// there (S N <= 2^19 values of 16 bytes; 16 times this stays below 2^31)
constexpr int kGridNowhere = 0x7ffffff;

// exchange buffer with agent-scope accesses of whole complex values
template <class R>
struct GridX {
    __amdgpu_buffer_rsrc_t r;
    __device__ GridX(void *p, long n)
        : r(__builtin_amdgcn_make_buffer_rsrc(p, 0, (int)(n * (long)sizeof(cx<R>)), 0x00020000)) {}
    __device__ __forceinline__ void st(int i, cx<R> v) const {
        if constexpr (sizeof(R) == 8)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, i * 16, 0, kAgentScope);
        else
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, i * 8, 0, kAgentScope);
    }
    __device__ __forceinline__ cx<R> ld(int i) const {
        if constexpr (sizeof(R) == 8)
            return __builtin_bit_cast(cx<R>, __builtin_amdgcn_raw_buffer_load_b128(r, i * 16, 0, kAgentScope));
        else
            return __builtin_bit_cast(cx<R>, __builtin_amdgcn_raw_buffer_load_b64(r, i * 8, 0, kAgentScope));
    }
};

// this thread's stores have reached the coherence point
__device__ __forceinline__ void grid_drain() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Flags and partial sums are kept in kGridCopies copies: a block writes all of
// them in one store instruction and reads only the copy of its group (b mod
// 8, the blocks of one XCD).  One copy polled by every wave of 256 blocks took
// 4 us to pass a barrier, 1.1 us with 32 blocks.
constexpr int kGridCopies = 8;
constexpr int kGridCopyBytes = kGridBlocks * 4 + 4 * kGridBlocks * 8 + 256;   // flags, four slots of partial sums
static_assert(kGridCopies * kGridCopyBytes <= (int)kGridSyncBytes, "sync area");
__device__ __forceinline__ unsigned *grid_flags(char *sync, int copy) {
    return reinterpret_cast<unsigned *>(sync + copy * kGridCopyBytes);
}
__device__ __forceinline__ double *grid_slot(char *sync, int copy, int slot) {
    return reinterpret_cast<double *>(sync + copy * kGridCopyBytes + kGridBlocks * 4) + slot * kGridBlocks;
}

// by wave 0: this block's flag
__device__ __forceinline__ void grid_signal(char *sync, unsigned epoch) {
    if (threadIdx.x < kGridCopies)
        __hip_atomic_store(grid_flags(sync, threadIdx.x) + blockIdx.x, epoch, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
// by wave 0: this block's partial sum, also where the host looks for it
__device__ __forceinline__ void grid_put(char *sync, int slot, double v, double *partials) {
    if (threadIdx.x < kGridCopies)
        __hip_atomic_store(grid_slot(sync, threadIdx.x, slot) + blockIdx.x, v, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    else if (threadIdx.x == kGridCopies)
        partials[slot * kMaxPartials + blockIdx.x] = v;
}

// by wave 0: waits until the first n blocks' flags have reached epoch; false
// after kGridWait.  n <= kGridBlocks.
__device__ __forceinline__ bool grid_wait(char *sync, int n, unsigned epoch) {
    const unsigned *flags = grid_flags(sync, blockIdx.x % kGridCopies);
    const int lane = threadIdx.x & 63;
    unsigned long long t0 = 0;
    for (bool first = true;; first = false) {
        unsigned f[kGridBlocks / 64];
#pragma unroll
        for (int i = 0; i < kGridBlocks / 64; ++i)
            f[i] = lane + 64 * i < n
                       ? __hip_atomic_load(flags + lane + 64 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                       : epoch;
        bool good = true;
#pragma unroll
        for (int i = 0; i < kGridBlocks / 64; ++i) good = good && (int)(f[i] - epoch) >= 0;
        if (__all(good)) break;
        if (first) t0 = wall_clock64();
        else if (wall_clock64() - t0 > kGridWait) return false;
    }
    asm volatile("" ::: "memory");   // loads of the exchanged data stay behind
    return true;
}

// by wave 0: sum of the first n blocks' partials, the same in every block; lane 0
__device__ __forceinline__ double grid_sum(char *sync, int slot, int n) {
    const double *p = grid_slot(sync, blockIdx.x % kGridCopies, slot);
    const int lane = threadIdx.x & 63;
    double a[kGridBlocks / 64], t = 0;
#pragma unroll
    for (int i = 0; i < kGridBlocks / 64; ++i)
        a[i] = lane + 64 * i < n ? __hip_atomic_load(p + lane + 64 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                 : 0.0;
#pragma unroll
    for (int i = 0; i < kGridBlocks / 64; ++i) t += a[i];
    return dpp_wave_sum(t);
}

// A block's rows and columns: what each of its threads owns of them, where
// that sits in the exchange buffers, and the filters' tables in LDS.
template <class R, int S>
struct GridBlock {
    int b, N0, N1, n, nrb, ncb;
    bool row, col;          // this block owns rows / columns
    int rst, cst;           // state of this thread's row / column
    int gi0, gi1;           // grid points of the row's and the column's first element (the others m0 and m1 N0 apart)
    int rA[8], rB[8], cA[8], cB[8];   // places of the row's and the column's elements in A and B
    GridAxis<R> ax[2];
    const double *f[2];     // the factor tables, per state
    // need: the axes whose filters run (bits 0 and 1)
    __device__ GridBlock(const GridShape &g, const LinePlan &p0, const LinePlan &p1, cx<R> *smem, int need = 3) {
        b = blockIdx.x;
        N0 = p0.L;
        N1 = p1.L;
        n = N0 * N1;
        nrb = g.nrb;
        ncb = g.ncb;
        row = b < nrb;
        col = b < ncb;
        const int rb = g.rb, cw = g.cw, chunk = S * rb * cw, tid = threadIdx.x;
        // neighbouring columns share cache lines: keep them on one XCD
        const int cb = col ? xcd_remap(b, ncb) : b;
        const int len0 = grid_line_len(g.R2[0], g.R3[0]), len1 = grid_line_len(g.R2[1], g.R3[1]);
        const int lines = max(rb * S * len0, cw * S * len1);
        cx<R> *tw = smem + lines;
        for (int d = 0; d < 2; ++d) {
            GridAxis<R> &A = ax[d];
            A.m = (d ? N1 : N0) / 8;
            A.R2 = g.R2[d];
            A.R3 = g.R3[d];
            A.RS = grid_rs(A.R3);
            A.nl = (d ? cw : rb) * S;
            A.lt = tid / A.nl;
            A.a = A.lt / A.R3;
            A.b = A.lt - A.a * A.R3;
            A.buf = smem + (tid - A.lt * A.nl);
            if (d == 0 || N1 != N0) {
                if (N1 == N0 || (need >> d) & 1)
                    grid_tables(reinterpret_cast<const cx<R> *>(d ? p1.tw : p0.tw), A.m, A.R3, tw, tw + 7 * A.m);
                A.tw1 = tw;
                A.tw2 = tw + 7 * A.m;
                tw += grid_tw_len(A.m);
            } else {
                A.tw1 = ax[0].tw1;
                A.tw2 = ax[0].tw2;
            }
        }
        f[0] = reinterpret_cast<double *>(tw);
        f[1] = f[0] + S * len0;
        const int lr = tid - ax[0].lt * ax[0].nl, r = lr / S, lc = tid - ax[1].lt * ax[1].nl, c = lc / S;
        rst = lr - r * S;
        cst = lc - c * S;
        ax[0].on = row && ax[0].lt < ax[0].m && b * rb + r < N1;
        ax[1].on = col && ax[1].lt < ax[1].m && cb * cw + c < N0;
        gi0 = (b * rb + r) * N0 + ax[0].lt;
        gi1 = ax[1].lt * N0 + cb * cw + c;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int x = ax[0].lt + q * ax[0].m, xb = x / cw, xc = x - xb * cw;
            rA[q] = (xb * nrb + b) * chunk + (xc * rb + r) * S + rst;
            rB[q] = (b * ncb + xb) * chunk + (r * cw + xc) * S + rst;
            if (!ax[0].on) rB[q] = kGridNowhere;
            const int y = ax[1].lt + q * ax[1].m, yb = y / rb, yr = y - yb * rb;
            cA[q] = !ax[1].on ? kGridNowhere : (cb * nrb + yb) * chunk + (c * rb + yr) * S + cst;
            cB[q] = (yb * ncb + cb) * chunk + (yr * cw + c) * S + cst;
        }
    }
    __device__ int gi(int q) const { return gi0 + q * ax[0].m; }
    // the axis of the filter `ph` as this thread takes part in it
    __device__ GridAxis<R> axis(int ph) const {
        GridAxis<R> A = ax[0];
        if (ph) A = ax[1];
        return A;
    }
};

// Per-state observables of the state before a step (Reporter.cpp:101-137), o:
// this thread's share of sum |psi|^2 and sum conj(psi) psi0, as one partial sum
// per block; put_norm: the block's norm also goes to the break test (slot 2).
template <int S>
__device__ __forceinline__ void grid_observe(const GridRun &a, int step, int st, const double (&o)[3],
                                             double (*red)[3 * S], bool put_norm, double *partials) {
    const int tid = threadIdx.x, wave = tid >> 6, nw = (blockDim.x + 63) >> 6;
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double v = dpp_wave_sum(s == st ? o[c] : 0.0);
            if ((tid & 63) == 0) red[wave][3 * s + c] = v;
        }
    lds_barrier();
    if (tid < 3 * S) {
        double v = 0;
        for (int w = 0; w < nw; ++w) v += red[w][tid];
        a.obsp[((long)step * 3 * S + tid) * gridDim.x + blockIdx.x] = v;
    }
    if (wave == 0 && put_norm) {
        double v = 0;
        for (int s = 0; s < S; ++s)
            for (int w = 0; w < nw; ++w) v += red[w][3 * s];
        grid_put(a.sync, 2, v, partials);
    }
}

// Chebyshev steps of a 2D grid (OCheby::real_time_step, and with IMAG
// imag_time_step, OCheby.cpp:92-297): the operands, break tests and orders of
// the per-order kernels.  partials: slots of the per-order kernels, one value
// per row block.  NIP: negative imaginary potential (one state).
// PRIMES: radices of primes above 7.  One instance holds the butterflies of all of
// them, so it spills (116 to 212 bytes of scratch per lane here, 0.8 to 1.1 kB in
// k_gspo_grid with two states); it is ahead of the per-order kernels all the same
// (240 x 176 points: a Chebyshev order 40 -> 14 us, a split-operator step of two
// coupled states 53 -> 23; 232 x 248: 297 -> 28 and 394 -> 38).
template <class R, int S, bool IMAG, bool NIP, bool PRIMES>
__global__ void __launch_bounds__(256) k_cheby_grid(GridRun a, GridShape g, HamDev<R> h, LinePlan p0, LinePlan p1,
                                                    const double *__restrict__ coef, int order, double offset,
                                                    double offset_i, double inv_scaling, double prec,
                                                    const cx<double> *__restrict__ psi, ChebyCtl *ctl,
                                                    double *__restrict__ partials) {
    extern __shared__ __align__(16) char smem_raw[];
    __shared__ double red[4][3 * S], bc;
    __shared__ int bad;
    __shared__ const R *Wp[S][S], *Mp[S][S];   // (scalar registers are short in the order loop)
    const int tid = threadIdx.x, wave = tid >> 6, nw = (blockDim.x + 63) >> 6;
    const GridBlock<R, S> B(g, p0, p1, reinterpret_cast<cx<R> *>(smem_raw));
    const int st = B.rst;
    const bool on = B.ax[0].on;
    if (tid == 0) {
#pragma unroll
        for (int i = 0; i < S; ++i)
#pragma unroll
            for (int j = 0; j < S; ++j) {
                Wp[i][j] = h.W[i][j];
                Mp[i][j] = h.mu[i][j];
            }
    }
    const double uni = st ? h.unity[S - 1] : h.unity[0];
    for (int s = 0; s < S; ++s) {
        const int len0 = grid_line_len(g.R2[0], g.R3[0]), len1 = grid_line_len(g.R2[1], g.R3[1]);
        grid_factors(h.tk[s][0], h.inv_nd[0], g.R2[0], g.R3[0], const_cast<double *>(B.f[0]) + s * len0);
        grid_factors(h.tk[s][1], h.inv_nd[1], g.R2[1], g.R3[1], const_cast<double *>(B.f[1]) + s * len1);
    }
    if (tid == 0) bad = 0;
    const long nx = (long)S * g.nrb * g.rb * g.ncb * g.cw;
    const GridX<R> XA(a.A, nx), XB(a.B, nx);
    cx<double> ps[8];
    double wi[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        ps[q] = on ? psi[(long)st * B.n + B.gi(q)] : mk<double>(0, 0);
        if (NIP) wi[q] = on ? (offset_i + (h.Wi[0] ? (double)h.Wi[0][B.gi(q)] : 0.0)) * inv_scaling : 0.0;
    }
    constexpr int NS = IMAG ? 3 : 2;
    auto slot = [](int k) { return k % NS == 2 ? 3 : k % NS; };
    unsigned epoch = a.epoch;
    double norm0 = 0, acc = 0, last_acc = 0;
    int last = 1;
    bool broke = false;
    __syncthreads();
    for (int step = 0; step < a.nsteps; ++step) {
        double wv[S][8];
#pragma unroll
        for (int j = 0; j < S; ++j) {
            const double E = a.fields ? a.fields[((long)step * S + st) * S + j] : a.field0[st * S + j];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                double w = j == st ? uni : 0.0;
                if (on && Wp[st][j]) w += (double)Wp[st][j][B.gi(q)];
                if (on && Mp[st][j]) w += E * (double)Mp[st][j][B.gi(q)];
                wv[j][q] = w;
            }
        }
        cx<R> pm1[8], pm2[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            pm1[q] = from_d<R>(ps[q]);
            pm2[q] = mk<R>(0, 0);
        }
        double o[3] = {0, 0, 0};
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            o[0] += ps[q].r * ps[q].r + ps[q].i * ps[q].i;
            if (a.psi0 && on) {
                const cx<double> z = reinterpret_cast<const cx<double> *>(a.psi0)[(long)st * B.n + B.gi(q)];
                o[1] += ps[q].r * z.r + ps[q].i * z.i;
                o[2] += ps[q].r * z.i - ps[q].i * z.r;
            }
        }
        grid_observe<S>(a, step, st, o, red, B.row, partials);
        last = 1;
        broke = false;
        acc = last_acc = 0;
        for (int k = 1; k < order; ++k) {
            const cx<double> ck = mk<double>(coef[2 * k], coef[2 * k + 1]);
            cx<R> x[8], v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                x[q] = pm1[q];
                if (on) XA.st(B.rA[q], pm1[q]);
            }
            ++epoch;
#pragma unroll 1
            for (int ph = 0; ph < 2; ++ph) {
                if (ph ? B.col : B.row) {
                    // the block's flag goes up inside the row filter, once its stores have landed
                    grid_filter<PRIMES>(x, B.axis(ph), ph ? B.f[1] + B.cst * grid_line_len(g.R2[1], g.R3[1])
                                                  : B.f[0] + st * grid_line_len(g.R2[0], g.R3[0]),
                                [&] { if (ph == 0) grid_drain(); },
                                [&] { if (ph == 0 && wave == 0) grid_signal(a.sync, epoch); });
                } else {
                    lds_barrier();   // publishes bc
                }
                if (ph) break;
#pragma unroll
                for (int q = 0; q < 8; ++q) v[q] = x[q];
                if (wave == 0 && !grid_wait(a.sync, B.nrb, epoch) && tid == 0) bad = 1;
                lds_barrier();
                if (bad) break;
#pragma unroll
                for (int q = 0; q < 8; ++q) x[q] = XA.ld(B.cA[q]);   // 0 for threads without a column
                // sum |psi|^2 of the step start or of order k - 1
                if (wave == 0 && (k == 1 || (k >= 3 && prec > 0))) {
                    const double s = grid_sum(a.sync, k == 1 ? 2 : slot(k - 1), B.nrb);
                    if (tid == 0) bc = s;
                }
            }
            if (bad) {
                if (tid == 0) *a.status = 1;
                return;
            }
            if (k == 1) norm0 = bc;
            if (k >= 3 && prec > 0) {
                // break test of order k - 1 (OCheby.cpp:179-182, 283-285)
                last_acc = acc;
                acc = bc;
                if (IMAG ? (k >= 4 && fabs(acc - last_acc) / last_acc < prec) : fabs(norm0 - acc) / norm0 < prec) {
                    broke = true;
                    break;
                }
            }
            last = k;
            if (B.ax[1].on) {
#pragma unroll
                for (int q = 0; q < 8; ++q) XB.st(B.cB[q], x[q]);
            }
            grid_drain();
            lds_barrier();
            ++epoch;
            if (wave == 0) {
                if (B.col) grid_signal(a.sync, epoch);
                if (B.row && !grid_wait(a.sync, B.ncb, epoch) && tid == 0) bad = 1;
            }
            lds_barrier();
            if (bad) {
                if (tid == 0) *a.status = 1;
                return;
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) x[q] = XB.ld(B.rB[q]);   // 0 for threads without a row
            const double two = k == 1 ? 1.0 : 2.0;   // phi_1 = (H - offset) phi_0 / R * (-i); pm2 = 0 there
            double sum = 0;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                cx<double> hp = to_d(v[q]) + to_d(x[q]);
                const cx<double> p = to_d(pm1[q]);
#pragma unroll
                for (int j = 0; j < S; ++j) {
                    // the other state's value sits one lane away
                    cx<double> pj = p;
                    if constexpr (S == 2) {
                        const cx<R> o = mk<R>(dpp<kXor1>(pm1[q].r), dpp<kXor1>(pm1[q].i));
                        if (j != st) pj = to_d(o);
                    }
                    hp.r += wv[j][q] * pj.r;
                    hp.i += wv[j][q] * pj.i;
                }
                cx<double> bb = mk<double>((hp.r - offset * p.r) * inv_scaling, (hp.i - offset * p.i) * inv_scaling);
                if (NIP) {
                    bb.r += wi[q] * p.i;
                    bb.i -= wi[q] * p.r;
                }
                const cx<double> mm = to_d(pm2[q]);
                cx<double> pk;
                if (IMAG) pk = mk<double>(-two * bb.r - mm.r, -two * bb.i - mm.i);
                else pk = mk<double>(two * bb.i + mm.r, -two * bb.r + mm.i);
                if (k == 1) ps[q] = cmul(mk<double>(coef[0], coef[1]), ps[q]);
                ps[q] = ps[q] + cmul(ck, pk);
                sum += ps[q].r * ps[q].r + ps[q].i * ps[q].i;
                pm2[q] = pm1[q];
                pm1[q] = from_d<R>(pk);
            }
            if (k >= 2 && (prec > 0 || k == order - 1)) {
                const double s = dpp_wave_sum(sum);
                if ((tid & 63) == 0) red[wave][0] = s;
                lds_barrier();
                if (B.row && wave == 0) {
                    double t = 0;
                    for (int w = 0; w < nw; ++w) t += red[w][0];
                    grid_put(a.sync, slot(k), t, partials);
                }
            }
        }
        if (B.b == 0 && tid == 0 && a.orders) a.orders[step] = last;
        lds_barrier();   // the next step's first writes to red follow the last reads
    }
    if (B.b == 0 && tid == 0) {
        ctl->norm0 = norm0;
        ctl->done = broke;
        ctl->accnorm = acc;
        ctl->last_order = last;
    }
    if (on) {
#pragma unroll
        for (int q = 0; q < 8; ++q) reinterpret_cast<cx<double> *>(a.out)[(long)st * B.n + B.gi(q)] = ps[q];
    }
}

// Split-operator steps exp(-i tau/2 W) exp(-i tau T) exp(-i tau/2 W) of a 2D
// grid (OGSPO.cpp:114-139), W the product of the x-space operators: a phase per
// point, whose field part (MU, one state) is formed per step, or (CPL) one 2 x 2
// unitary of two coupled states.  exp(-i tau T) is a filter along each
// dimension, in either order: steps that begin in the row layout filter along
// dimension 0, hand the lines over and end in the column layout, where the
// next step begins (its number's parity says where: single steps give the bits
// of a run).  One exchange per step; the x-space tables and psi0 sit in
// registers in both layouts.  Waiting for one launch costs more than a single
// step, which is two ordinary launches of the same kernel instead (a.part 1:
// up to the exchange, 2: the rest, psi in place).  Per step on 512 x 512 points, two coupled states,
// observables included: 41 -> 16.2 us against the column and the row pass.
template <class R, int S, bool MU, bool CPL, bool PRIMES>
__global__ void __launch_bounds__(256) k_gspo_grid(GridRun a, GridShape g, XGroupDev<R> pre, LinePlan p0, LinePlan p1,
                                                   const double *__restrict__ ek, double inv0, double inv1,
                                                   const cx<double> *__restrict__ psi) {
    static_assert(!MU || S == 1, "field operators act on one state");
    static_assert(!CPL || S == 2, "two coupled states");
    extern __shared__ __align__(16) char smem_raw[];
    __shared__ double red[4][3 * S];
    __shared__ int bad;
    const int tid = threadIdx.x, wave = tid >> 6;
    const bool begin = a.first & 1;                    // the layout of psi before the first step
    const bool later = begin != (a.part == 2);         // ... and of the part's filter
    const int need = a.part ? 1 << later : 3;
    const GridBlock<R, S> B(g, p0, p1, reinterpret_cast<cx<R> *>(smem_raw), need);
    // factors exp(-i tau T_d(k)) / N_d; ek: per state the tables of both
    // dimensions, (re, im)
    cx<double> *fac = reinterpret_cast<cx<double> *>(const_cast<double *>(B.f[0]));
    const int len0 = grid_line_len(g.R2[0], g.R3[0]), len1 = grid_line_len(g.R2[1], g.R3[1]);
    for (int s = 0; s < S; ++s) {
        const cx<double> *e = reinterpret_cast<const cx<double> *>(ek) + (long)s * (B.N0 + B.N1);
        if (need & 1) grid_factors(e, inv0, g.R2[0], g.R3[0], fac + s * len0);
        if (need & 2) grid_factors(e + B.N0, inv1, g.R2[1], g.R3[1], fac + S * len0 + s * len1);
    }
    const cx<double> *f0 = fac + B.rst * len0, *f1 = fac + S * len0 + B.cst * len1;
    if (tid == 0) bad = 0;
    const long nx = (long)S * g.nrb * g.rb * g.ncb * g.cw;
    const GridX<R> XA(a.A, nx), XB(a.B, nx);
    const bool on0 = B.ax[0].on, on1 = B.ax[1].on;
    const int st0 = B.rst, st1 = B.cst;
    // this thread's points in both layouts: the x-space group (own state and,
    // coupled, the other one; of a field operator mu tau) and psi0
    struct Layout {
        cx<double> u[8], w[CPL ? 8 : 1], z[8];
        double mu[MU ? 8 : 1];
    } L0, L1;
    // the usual group, one operator with a table, is read in one go (point by
    // point the eight reads wait for each other)
    const bool table = !MU && pre.n == 1 && pre.op[0].U;
    auto load = [&](Layout &L, bool on, int st, auto gi) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            L.u[q] = mk<double>(1, 0);
            L.z[q] = mk<double>(0, 0);
            if constexpr (CPL) L.w[q] = mk<double>(0, 0);
            if constexpr (MU) L.mu[q] = 0;
        }
        if (!on) return;
        if (a.psi0) {
#pragma unroll
            for (int q = 0; q < 8; ++q) L.z[q] = reinterpret_cast<const cx<double> *>(a.psi0)[(long)st * B.n + gi(q)];
        }
        if (table) {
            const cx<double> *U = reinterpret_cast<const cx<double> *>(pre.op[0].U);
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                L.u[q] = U[(long)(CPL ? 2 * st : st) * B.n + gi(q)];
                if constexpr (CPL) L.w[q] = U[B.n + gi(q)];
            }
            return;
        }
        if constexpr (MU && !PRIMES) {
            // a field and tables, operator by operator for the same reason (a
            // single step on 512 x 512 points 59 -> 54 us, 64 x 64 49 -> 43; with
            // PRIMES the registers do not suffice, 240 x 176 points 18 -> 22)
            for (int o = 0; o < pre.n; ++o) {
                XSplitDev<R> op = pre.op[o];
                if (op.mu[0][0]) {
                    R m[8];
#pragma unroll
                    for (int q = 0; q < 8; ++q) m[q] = op.mu[0][0][gi(q)];
#pragma unroll
                    for (int q = 0; q < 8; ++q) L.mu[q] = op.tau * (double)m[q];
                    op.mu[0][0] = nullptr;   // the field part is formed per step
                    if (!op.V[0][0]) continue;
                }
                if (op.U) {
                    const cx<double> *U = reinterpret_cast<const cx<double> *>(op.U);
                    cx<double> t[8];
#pragma unroll
                    for (int q = 0; q < 8; ++q) t[q] = U[gi(q)];
#pragma unroll
                    for (int q = 0; q < 8; ++q) L.u[q] = cmul(L.u[q], t[q]);
                    continue;
                }
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    cx<double> v[1] = {L.u[q]};
                    xsplit_point<R, 1>(op, gi(q), v);
                    L.u[q] = v[0];
                }
            }
            return;
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const long i = gi(q);
            if constexpr (CPL) {
                cx<double> v[2] = {mk<double>(st == 0, 0), mk<double>(st == 1, 0)};
                xgroup_point<R, 2>(pre, i, v);   // a symmetric matrix
                L.u[q] = st ? v[1] : v[0];
                L.w[q] = st ? v[0] : v[1];
            } else {
                cx<double> v[S];
#pragma unroll
                for (int s = 0; s < S; ++s) v[s] = mk<double>(1, 0);
                for (int o = 0; o < pre.n; ++o) {
                    XSplitDev<R> op = pre.op[o];
                    if constexpr (MU) {
                        if (op.mu[0][0]) {
                            L.mu[q] = op.tau * (double)op.mu[0][0][i];
                            op.mu[0][0] = nullptr;   // the field part is formed per step
                            if (!op.V[0][0]) continue;
                        }
                    }
                    xsplit_point<R, S>(op, i, v);
                }
                L.u[q] = S == 2 && st ? v[S - 1] : v[0];
            }
        }
    };
    const int gr = B.gi0, gc = B.gi1, m0 = B.ax[0].m, sc = B.ax[1].m * B.N0;
    if (need & 1) load(L0, on0, st0, [&](int q) { return (long)(gr + q * m0); });
    if (need & 2) load(L1, on1, st1, [&](int q) { return (long)gc + (long)q * sc; });
    // the x-space group on x
    auto apply = [&](const Layout &L, cx<R>(&x)[8], double E) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            cx<double> u = L.u[q];
            if constexpr (MU) {
                double sn, cs;
                sincos(-L.mu[q] * E, &sn, &cs);
                u = cmul(u, mk<double>(cs, sn));
            }
            cx<double> y = cmul(u, to_d(x[q]));
            if constexpr (CPL) y = y + cmul(L.w[q], to_d(mk<R>(dpp<kXor1>(x[q].r), dpp<kXor1>(x[q].i))));
            x[q] = from_d<R>(y);
        }
    };
    auto observe = [&](const Layout &L, const cx<R>(&x)[8], double(&o)[3]) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const cx<double> p = to_d(x[q]);
            o[0] += p.r * p.r + p.i * p.i;
            o[1] += p.r * L.z[q].r + p.i * L.z[q].i;
            o[2] += p.r * L.z[q].i - p.i * L.z[q].r;
        }
    };
    cx<R> x[8];
    bool cols = later;   // the layout of x
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        x[q] = mk<R>(0, 0);
        if (a.part == 2) {
            x[q] = cols ? XA.ld(B.cA[q]) : XB.ld(B.rB[q]);
        } else if (cols) {
            if (on1) x[q] = from_d<R>(psi[(long)st1 * B.n + gc + (long)q * sc]);
        } else if (on0) {
            x[q] = from_d<R>(psi[(long)st0 * B.n + gr + q * m0]);
        }
    }
    unsigned epoch = a.epoch;
    __syncthreads();
    // two half steps per step, each with one filter
#pragma unroll 1
    for (int half = a.part == 2; half < 2 * a.nsteps; ++half) {
        const int step = half >> 1;
        const bool second = half & 1;
        const double E = MU ? (a.fields ? a.fields[step] : a.field0[0]) : 0.0;
        if (!second) {
            if (a.observe) {
                double o[3] = {0, 0, 0};
                if (cols) observe(L1, x, o);
                else observe(L0, x, o);
                grid_observe<S>(a, step, cols ? st1 : st0, o, red, false, nullptr);
            }
            if (cols) apply(L1, x, E);
            else apply(L0, x, E);
        }
        if (cols ? B.col : B.row)
            grid_filter<PRIMES>(x, B.axis(cols), cols ? f1 : f0, [] {}, [] {});
        if (second) {
            if (cols) apply(L1, x, E);
            else apply(L0, x, E);
            continue;
        }
        // hand over to the other layout
        if (cols) {
            if (on1) {
#pragma unroll
                for (int q = 0; q < 8; ++q) XB.st(B.cB[q], x[q]);
            }
        } else if (on0) {
#pragma unroll
            for (int q = 0; q < 8; ++q) XA.st(B.rA[q], x[q]);
        }
        if (a.part == 1) return;
        grid_drain();
        lds_barrier();
        ++epoch;
        if (wave == 0) {
            if (cols ? B.col : B.row) grid_signal(a.sync, epoch);
            if ((cols ? B.row : B.col) && !grid_wait(a.sync, cols ? B.ncb : B.nrb, epoch) && tid == 0) bad = 1;
        }
        lds_barrier();
        if (bad) {
            if (tid == 0) *a.status = 1;
            return;
        }
        if (cols) {
#pragma unroll
            for (int q = 0; q < 8; ++q) x[q] = XB.ld(B.rB[q]);   // 0 for threads without a row
        } else {
#pragma unroll
            for (int q = 0; q < 8; ++q) x[q] = XA.ld(B.cA[q]);
        }
        cols = !cols;
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        cx<double> *out = reinterpret_cast<cx<double> *>(a.out);
        if (cols) {
            if (on1) out[(long)st1 * B.n + gc + (long)q * sc] = to_d(x[q]);
        } else if (on0) {
            out[(long)st0 * B.n + gr + q * m0] = to_d(x[q]);
        }
    }
}

// The Lanczos vectors and the tridiagonal matrix of one short iterative Lanczos
// step on a 2D grid (OSIL::BuildLZB, OSIL.cpp:79-190; real or imaginary time):
// q_0 = psi, q_{k+1} = (H - alpha_k) q_k - beta_{k-1} q_{k-1}, normalised, until
// the error estimate ends it.  H q as in k_cheby_grid; the two sums of an
// iteration go round over the blocks' partial sums.  res: psinorm^2, the
// number of iterations, alpha[order], beta[order] (norms).  Every vector is
// stored once, for the combination that follows.  An iteration on 192 x 256
// points took 84 us with launches and host round trips for each sum, 22 us here.
template <int S, bool PRIMES>
__global__ void __launch_bounds__(256) k_sil_grid(GridRun a, GridShape g, HamDev<double> h, LinePlan p0, LinePlan p1,
                                                  SilVectors qv, int order, double dt, double err_max, double weight,
                                                  const cx<double> *__restrict__ psi, double *__restrict__ res) {
    extern __shared__ __align__(16) char smem_raw[];
    __shared__ double red[4], bc;
    __shared__ int bad;
    using C = cx<double>;
    const int tid = threadIdx.x, wave = tid >> 6, nw = (blockDim.x + 63) >> 6;
    const GridBlock<double, S> B(g, p0, p1, reinterpret_cast<C *>(smem_raw));
    const int st = B.rst;
    const bool on = B.ax[0].on;
    const int len0 = grid_line_len(g.R2[0], g.R3[0]), len1 = grid_line_len(g.R2[1], g.R3[1]);
    for (int s = 0; s < S; ++s) {
        grid_factors(h.tk[s][0], h.inv_nd[0], g.R2[0], g.R3[0], const_cast<double *>(B.f[0]) + s * len0);
        grid_factors(h.tk[s][1], h.inv_nd[1], g.R2[1], g.R3[1], const_cast<double *>(B.f[1]) + s * len1);
    }
    if (tid == 0) bad = 0;
    const long nx = (long)S * g.nrb * g.rb * g.ncb * g.cw;
    const GridX<double> XA(a.A, nx), XB(a.B, nx);
    const double uni = st ? h.unity[S - 1] : h.unity[0];
    C cur[8], prev[8];
    double wv[S][8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        cur[q] = on ? psi[(long)st * B.n + B.gi(q)] : mk<double>(0, 0);
        prev[q] = mk<double>(0, 0);
#pragma unroll
        for (int j = 0; j < S; ++j) {
            double w = j == st ? uni : 0.0;
            if (on && h.W[st][j]) w += h.W[st][j][B.gi(q)];
            if (on && h.mu[st][j]) w += h.Edip[st][j] * h.mu[st][j][B.gi(q)];
            wv[j][q] = w;
        }
    }
    unsigned epoch = a.epoch;
    // sum over the grid of v, in every thread; false: gave up
    auto total = [&](double v, int slot, double &out) {
        const double s = dpp_wave_sum(v);
        if ((tid & 63) == 0) red[wave] = s;
        lds_barrier();
        ++epoch;
        if (wave == 0) {
            double t = 0;
            for (int w = 0; w < nw; ++w) t += red[w];
            if (B.row) {
                if (tid < kGridCopies)
                    __hip_atomic_store(grid_slot(a.sync, tid, slot) + B.b, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                grid_drain();
                grid_signal(a.sync, epoch);
            }
            if (!grid_wait(a.sync, B.nrb, epoch)) {
                if (tid == 0) bad = 1;
            } else {
                const double r = grid_sum(a.sync, slot, B.nrb);
                if (tid == 0) bc = r;
            }
        }
        lds_barrier();
        out = bc;
        return !bad;
    };
    auto norm2 = [&](const C(&x)[8]) {
        double t = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) t += x[q].r * x[q].r + x[q].i * x[q].i;
        return t;
    };
    __syncthreads();
    bool ok = true;
    double psin = 0, alpha = 0, beta0 = 0, beta1 = 0, beta2 = 0, pdt = 1, prod = 1;
    ok = total(norm2(cur), 0, psin);
    const double psinorm = sqrt(psin * weight);
    // iteration it: H q_{it-1}, alpha_{it-1}, q_it, beta_{it-1}; it = order: only
    // the last diagonal element
    int it = 1;
    for (; ok; ++it) {
        C x[8], v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            x[q] = cur[q];
            if (on) XA.st(B.rA[q], cur[q]);
        }
        ++epoch;
#pragma unroll 1
        for (int ph = 0; ph < 2; ++ph) {
            if (ph ? B.col : B.row)
                grid_filter<PRIMES>(x, B.axis(ph), ph ? B.f[1] + B.cst * len1 : B.f[0] + st * len0,
                                    [&] { if (ph == 0) grid_drain(); },
                                    [&] { if (ph == 0 && wave == 0) grid_signal(a.sync, epoch); });
            if (ph) break;
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = x[q];
            if (wave == 0 && !grid_wait(a.sync, B.nrb, epoch) && tid == 0) bad = 1;
            lds_barrier();
            if (bad) break;
#pragma unroll
            for (int q = 0; q < 8; ++q) x[q] = XA.ld(B.cA[q]);   // 0 for threads without a column
        }
        if (bad) break;
        if (B.ax[1].on) {
#pragma unroll
            for (int q = 0; q < 8; ++q) XB.st(B.cB[q], x[q]);
        }
        grid_drain();
        lds_barrier();
        ++epoch;
        if (wave == 0) {
            if (B.col) grid_signal(a.sync, epoch);
            if (B.row && !grid_wait(a.sync, B.ncb, epoch) && tid == 0) bad = 1;
        }
        lds_barrier();
        if (bad) break;
        double dot = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            C hp = v[q] + XB.ld(B.rB[q]);   // 0 for threads without a row
#pragma unroll
            for (int j = 0; j < S; ++j) {
                C pj = cur[q];
                if constexpr (S == 2) {   // the other state's value sits one lane away
                    const C o = mk<double>(dpp<kXor1>(cur[q].r), dpp<kXor1>(cur[q].i));
                    if (j != st) pj = o;
                }
                hp.r += wv[j][q] * pj.r;
                hp.i += wv[j][q] * pj.i;
            }
            v[q] = hp;
            dot += cur[q].r * hp.r + cur[q].i * hp.i;
        }
        if (!total(dot, 1, alpha)) break;
        alpha *= weight;
        if (B.b == 0 && tid == 0) res[2 + it - 1] = alpha;
        if (it == order) break;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            C w = mk<double>(v[q].r - alpha * cur[q].r, v[q].i - alpha * cur[q].i);
            w.r -= beta1 * prev[q].r;
            w.i -= beta1 * prev[q].i;
            v[q] = w;
        }
        // error estimate dt^(it-2) beta_0 prod beta_i / i over 1 <= i <= it - 3,
        // before this iteration's norm is known (OSIL.cpp:128-135)
        double err = 0;
        if (it >= 2) {
            if (it > 2) pdt *= dt;
            if (it > 3) prod *= beta2 / (it - 3);
            err = fabs(pdt * beta0 * prod);
        }
        beta2 = beta1;
        double b2;
        if (!total(norm2(v), 0, b2)) break;
        beta1 = sqrt(b2 * weight);
        if (it == 1) beta0 = beta1;
        if (B.b == 0 && tid == 0) res[2 + order + it - 1] = beta1;
        const double f = 1 / beta1;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            prev[q] = cur[q];
            cur[q] = mk<double>(v[q].r * f, v[q].i * f);
            if (on) reinterpret_cast<C *>(qv.q[it])[(long)st * B.n + B.gi(q)] = cur[q];
        }
        if (it >= 2 && err < err_max * psinorm) break;
    }
    if (bad) {
        if (tid == 0) *a.status = 1;
        return;
    }
    if (B.b == 0 && tid == 0) {
        res[0] = psin;
        res[1] = it;
    }
}

// psi <- c_0 psi + sum over 0 < i < n of c_i q_i
__global__ void __launch_bounds__(256) k_sil_combine(SilVectors qv, SilCoeffs c, int n, long len,
                                                     cx<double> *__restrict__ psi) {
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < len; e += (long)gridDim.x * 256) {
        cx<double> y = cmul(mk<double>(c.c[0], c.c[1]), psi[e]);
#pragma unroll 4
        for (int i = 1; i < n; ++i)
            y = y + cmul(mk<double>(c.c[2 * i], c.c[2 * i + 1]), reinterpret_cast<const cx<double> *>(qv.q[i])[e]);
        psi[e] = y;
    }
}

// the status of a launch of k_sil_grid to the host
__global__ void k_grid_report(GridRun a, volatile int *report) { *report = *a.status; }

// After a run: psi from its staging copy and the observables of each step
// (blocks past ncopy, one per step: 4 S doubles as qdx_prop_run lays them
// out); nothing when the run gave up.  report: host-visible status.
__global__ void __launch_bounds__(256) k_grid_finish(GridRun a, int S, long n, int nb, int ncopy,
                                                     cx<double> *__restrict__ psi, double *__restrict__ obs,
                                                     volatile int *report) {
    const int status = *a.status;
    if (blockIdx.x == 0 && threadIdx.x == 0) *report = status;
    if (status) return;
    if ((int)blockIdx.x < ncopy) {
        const cx<double> *out = reinterpret_cast<const cx<double> *>(a.out);
        for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < S * n; i += (long)ncopy * 256) psi[i] = out[i];
        return;
    }
    const int step = blockIdx.x - ncopy, wave = threadIdx.x >> 6;
    for (int o = wave; o < 3 * S; o += 4) {
        const double *p = a.obsp + ((long)step * 3 * S + o) * nb;
        double t = 0;
        for (int i = threadIdx.x & 63; i < nb; i += 64) t += p[i];
        t = wave_sum(t);
        if ((threadIdx.x & 63) == 0) {
            const int s = o / 3, c = o - 3 * s;
            double *d = obs + (long)step * 4 * S;
            if (c == 0) {
                d[2 * s] = t;
                d[2 * s + 1] = 0;
            } else {
                d[2 * S + 2 * s + c - 1] = t;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// launchers

// Points of a block's lines, at least: one wave of 8 each.  A short line is a
// latency chain, so it goes to as many CUs as there are lines (an order of
// 64 x 64 points takes 9.4 us with 512 points per block, 10.1 with 1024, 11.8
// with 2048; 256 x 256 12.0, 12.5, 14.6; 240 x 176 16.5, 17.2, 18.7).
constexpr int kGridFill = 512;

// factor: bytes of a filter's factor (8 real, 16 complex)
static size_t grid_lds_bytes(const GridShape &g, int N0, int N1, int S, size_t elem, size_t factor) {
    const size_t l0 = grid_line_len(g.R2[0], g.R3[0]), l1 = grid_line_len(g.R2[1], g.R3[1]);
    const size_t tw = grid_tw_len(N0 / 8) + (N1 == N0 ? 0 : grid_tw_len(N1 / 8));
    return (std::max(g.rb * S * l0, g.cw * S * l1) + tw) * elem + S * (l0 + l1) * factor;
}

// m = R2 R3 for a line of 8 m points: the stages' radices (see grid_filter),
// the pair with the fewest multiply-adds per point and passes; false when
// there is none
bool grid_radices(int m, int &R2, int &R3) {
    auto dft = [](int r) {   // operations of a butterfly, about
        if (r == 1) return 0.0;
        double c = 0;
        int n = r;
        for (int p : {2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31})
            while (n % p == 0) {
                n /= p;
                c += p == 2 ? 2.0 : p == 3 ? 4.0 : p - 1.0;
            }
        return n > 1 ? -1.0 : c * r;
    };
    double best = 0;
    R2 = 0;
    for (int r3 = 1; r3 <= 16; ++r3) {
        if (m % r3) continue;
        const int r2 = m / r3;
        const bool prime = r2 == 17 || r2 == 19 || r2 == 23 || r2 == 29 || r2 == 31;
        if (r2 > 16 && !prime) continue;
        // butterflies of one thread times their cost (twiddles: 4 operations),
        // LDS accesses included
        auto stage = [&](int r) { return ((8 + r - 1) / r) * (dft(r) + 12.0 * r + 40.0); };
        const double c = (r2 > 1 ? stage(r2) + 60.0 : 0.0) + stage(r3);
        if (!R2 || c < best) {
            best = c;
            R2 = r2;
            R3 = r3;
        }
    }
    return R2 > 0;
}

bool grid_shape(int N0, int N1, int S, int cus, bool gspo, GridShape &g) {
    if (S < 1 || S > 2 || N0 % 8 || N1 % 8 || N0 < 8 || N1 < 8) return false;
    if (!grid_radices(N0 / 8, g.R2[0], g.R3[0]) || !grid_radices(N1 / 8, g.R2[1], g.R3[1])) return false;
    for (int d = 0; d < 2; ++d)
        for (int r : {g.R2[d], g.R3[d]}) g.primes = g.primes || r == 11 || r == 13 || r > 16;
    const int most = std::min(cus, kGridBlocks);
    // lines per block: at most 256 threads at 8 points each and no more
    // blocks than CUs; the fewest lines with kGridFill points
    auto pick = [&](int lines, int L) {
        int best = 0;
        for (int r = 1; r <= lines && r * S * L <= 2048; ++r) {
            if ((lines + r - 1) / r > most) continue;
            best = r;
            if (r * S * L >= kGridFill) break;
        }
        return best;
    };
    g.rb = pick(N1, N0);
    g.cw = pick(N0, N1);
    if (!g.rb || !g.cw) return false;
    g.nrb = (N1 + g.rb - 1) / g.rb;
    g.ncb = (N0 + g.cw - 1) / g.cw;
    g.blocks = std::max(g.nrb, g.ncb);
    g.threads = std::max(64, round64(std::max(g.rb * S * (N0 / 8), g.cw * S * (N1 / 8))));
    // the 160 KiB of a CU (the tables of two long lines may not fit)
    return grid_lds_bytes(g, N0, N1, S, 16, gspo ? 16 : 8) <= kLdsBytes - 1024;
}

size_t grid_exchange_len(const GridShape &g, int S) { return (size_t)S * g.nrb * g.rb * g.ncb * g.cw; }

template <class R>
void launch_cheby_grid(hipStream_t s, int S, const HamDev<R> &h, const GridShape &g, const GridRun &a,
                       const LinePlan &p0, const LinePlan &p1, const double *coef, int order, double offset,
                       double offset_i, double inv_scaling, double prec, bool imag, const double *psi, ChebyCtl *ctl,
                       double *partials) {
    const size_t lds = grid_lds_bytes(g, p0.L, p1.L, S, sizeof(cx<R>), sizeof(double));
    auto cp = reinterpret_cast<const cx<double> *>(psi);
    const bool nip = offset_i != 0 || h.Wi[0] != nullptr;
#define QDX_GRID(S_, IMAG_, NIP_)                     \
    do {                                              \
        if (g.primes) QDX_GRIDP(S_, IMAG_, NIP_, true); \
        else QDX_GRIDP(S_, IMAG_, NIP_, false);       \
    } while (0)
#define QDX_GRIDP(S_, IMAG_, NIP_, PR_)                                                                        \
    do {                                                                                                       \
        set_lds(k_cheby_grid<R, S_, IMAG_, NIP_, PR_>, lds);                                                   \
        QDX_LAUNCH((k_cheby_grid<R, S_, IMAG_, NIP_, PR_>), dim3(g.blocks), dim3(g.threads), lds, s, a, g, h,  \
                   p0, p1, coef, order, offset, nip ? offset_i : 0.0, inv_scaling, prec, cp, ctl, partials);   \
    } while (0)
    if (nip) {
        if (S != 1 || imag) throw std::runtime_error("negative imaginary potential: one state, real time only");
        QDX_GRID(1, false, true);
    } else if (imag) {
        if constexpr (std::is_same<R, double>::value) {
            if (S == 1) QDX_GRID(1, true, false);
            else QDX_GRID(2, true, false);
        } else {
            throw std::runtime_error("imaginary time: FP64 only");
        }
    } else if (S == 1) {
        QDX_GRID(1, false, false);
    } else {
        QDX_GRID(2, false, false);
    }
#undef QDX_GRID
#undef QDX_GRIDP
    QDX_HIP(hipGetLastError());
}
template void launch_cheby_grid(hipStream_t, int, const HamDev<double> &, const GridShape &, const GridRun &,
                                const LinePlan &, const LinePlan &, const double *, int, double, double, double, double,
                                bool, const double *, ChebyCtl *, double *);
template void launch_cheby_grid(hipStream_t, int, const HamDev<float> &, const GridShape &, const GridRun &,
                                const LinePlan &, const LinePlan &, const double *, int, double, double, double, double,
                                bool, const double *, ChebyCtl *, double *);

template <class R>
void launch_gspo_grid(hipStream_t s, int S, const GridShape &g, const GridRun &a, const XGroupDev<R> &pre, bool mu,
                      bool coupled, const LinePlan &p0, const LinePlan &p1, const double *ek, double inv0, double inv1,
                      const double *psi) {
    const size_t lds = grid_lds_bytes(g, p0.L, p1.L, S, sizeof(cx<R>), 16);
    auto cp = reinterpret_cast<const cx<double> *>(psi);
    auto launch = [&](auto kernel) {
        set_lds(kernel, lds);
        QDX_LAUNCH(kernel, dim3(g.blocks), dim3(g.threads), lds, s, a, g, pre, p0, p1, ek, inv0, inv1, cp);
        QDX_HIP(hipGetLastError());
    };
#define QDX_GRID(S_, MU_, CPL_)                                                                                  \
    do {                                                                                                         \
        if (g.primes) launch(k_gspo_grid<R, S_, MU_, CPL_, true>);                                               \
        else launch(k_gspo_grid<R, S_, MU_, CPL_, false>);                                                       \
    } while (0)
    if (mu) QDX_GRID(1, true, false);
    else if (coupled) QDX_GRID(2, false, true);
    else if (S == 1) QDX_GRID(1, false, false);
    else QDX_GRID(2, false, false);
#undef QDX_GRID
}
template void launch_gspo_grid(hipStream_t, int, const GridShape &, const GridRun &, const XGroupDev<double> &, bool,
                               bool, const LinePlan &, const LinePlan &, const double *, double, double,
                               const double *);
template void launch_gspo_grid(hipStream_t, int, const GridShape &, const GridRun &, const XGroupDev<float> &, bool,
                               bool, const LinePlan &, const LinePlan &, const double *, double, double,
                               const double *);

void launch_sil_grid(hipStream_t s, int S, const HamDev<double> &h, const GridShape &g, const GridRun &a,
                     const LinePlan &p0, const LinePlan &p1, const SilVectors &q, int order, double dt, double err,
                     double weight, const double *psi, double *res, int *report) {
    const size_t lds = grid_lds_bytes(g, p0.L, p1.L, S, 16, sizeof(double));
    auto cp = reinterpret_cast<const cx<double> *>(psi);
    auto launch = [&](auto kernel) {
        set_lds(kernel, lds);
        QDX_LAUNCH(kernel, dim3(g.blocks), dim3(g.threads), lds, s, a, g, h, p0, p1, q, order, dt, err, weight, cp, res);
        QDX_HIP(hipGetLastError());
    };
    if (S == 1 && g.primes) launch(k_sil_grid<1, true>);
    else if (S == 1) launch(k_sil_grid<1, false>);
    else if (g.primes) launch(k_sil_grid<2, true>);
    else launch(k_sil_grid<2, false>);
    QDX_LAUNCH(k_grid_report, dim3(1), dim3(1), 0, s, a, report);
    QDX_HIP(hipGetLastError());
}

void launch_sil_combine(hipStream_t s, const SilVectors &q, const SilCoeffs &c, int n, long len, double *psi) {
    const int nb = (int)std::min<long>(2048, (len + 255) / 256);
    QDX_LAUNCH(k_sil_combine, dim3(nb), dim3(256), 0, s, q, c, n, len, reinterpret_cast<cx<double> *>(psi));
    QDX_HIP(hipGetLastError());
}

void launch_grid_finish(hipStream_t s, int S, long n, const GridShape &g, const GridRun &a, double *psi, double *obs,
                        int *report) {
    const int ncopy = (int)std::min<long>(1024, (S * n + 255) / 256);
    QDX_LAUNCH(k_grid_finish, dim3(ncopy + (obs ? a.nsteps : 0)), dim3(256), 0, s, a, S, n, g.blocks, ncopy,
               reinterpret_cast<cx<double> *>(psi), obs, report);
    QDX_HIP(hipGetLastError());
}

}  // namespace qdx

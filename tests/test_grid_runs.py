"""2D grids whose runs stay in registers (qdx_grid.hip) against the per-order
kernels, which qdx_ctx_set_line_points(8) selects: the smallest lines, unequal
sides (more row blocks than column blocks and the reverse), several lines per
block, sides with odd prime factors, the largest grid of the rule and the
first beyond it; both kinds of time, fields, the negative imaginary potential,
runs and single steps.  Both evaluate the same series in FP64: an H
application differs by a few 1e-16 of the kinetic range, a series of order k
by about k times that, so 1e-11 bounds a few steps of at most a few hundred
orders; the series lengths are equal.  In FP32 both round each term to 2^-24
and carry that through the same recurrence: 1e-5 over these short series."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(b)


def box(N0, N1, S, laser=False, nip=False, coupled=True, nt=12):
    p = cases.Problem([N0, N1], [-6.0, -5.0], [6.0, 5.0], nstates=S)
    x, y = p.axes()
    one = np.ones(np.broadcast_shapes(x.shape, y.shape))
    for s in range(S):
        p.kinetic(s, [1500.0 + 300 * s, 2500.0 - 200 * s])
        p.potential(s, s, np.minimum(0.03 * (1 + 0.3 * s) * ((x - 0.2 * s) ** 2 + y ** 2) + 0.01 * s, 1.0))
    if S > 1 and coupled:
        p.potential(0, 1, 0.02 * np.exp(-x ** 2 - (y - 0.3) ** 2))
    if laser:
        p.dipole(1 if S > 1 else 0, 0, one * x * np.exp(-x ** 2 / 8), 0.01 * np.cos(0.3 * np.arange(nt)))
    if nip:
        p.gobbler(0, 0, rp={0: 4.0}, order=5, gain=0.02, nip=True)
    g = np.exp(-(x - 0.4) ** 2 - (y + 0.2) ** 2 + 0.8j * x - 0.3j * y)
    p.psi0 = cases.normalized(p, np.stack([(1 - 0.2j * s) * g for s in range(S)]))
    return p


def both(make, steps, run):
    import qdng_amd as Q
    out = []
    for points in (0, 8):
        c = Q.Context(0)
        try:
            c.set_line_points(points)
            p, U = make(c)
            w, w0 = p.gpu_wf(c), p.gpu_wf(c)
            if run:
                n2, ac, nh, _ = U.run(w, 1, steps, w0)
            else:
                st = [U.apply(w, 1 + i) for i in range(steps)]
                n2, ac, nh = [s.norm2 for s in st], [w.overlap(w0)], [s.n_hpsi for s in st]
            out.append((w.download(), np.array(n2), np.array(ac), list(nh)))
            del U, w, w0
        finally:
            c.close()
    return out


def check(pair, tol=1e-11):
    (a, na, aa, ha), (b, nb, ab, hb) = pair
    assert ha == hb
    assert rel(a, b) < tol
    assert np.max(np.abs(na - nb) / nb) < tol and np.max(np.abs(aa - ab)) < tol * max(1.0, np.max(np.abs(ab)))


SHAPES = [(8, 8, 1), (8, 16, 2), (24, 8, 1), (40, 56, 2), (104, 88, 1), (16, 768, 1), (768, 16, 2), (64, 64, 1),
          (240, 176, 1), (232, 248, 2), (256, 256, 1), (128, 384, 2), (768, 512, 1), (512, 512, 2), (768, 768, 2)]


@pytest.mark.parametrize("N0,N1,S", SHAPES)
@pytest.mark.parametrize("laser", [False, True])
def test_cheby(N0, N1, S, laser):
    import qdng_amd as Q
    print("[gpu case] grid cheby", N0, N1, S, laser, flush=True)

    def make(c):
        p = box(N0, N1, S, laser)
        return p, Q.Cheby(p.gpu_ham(c), 2.0, prec=1e-12)
    check(both(make, 4, True))
    check(both(make, 2, False))


@pytest.mark.parametrize("precision,tol", [("fp32", 1e-5), ("compact", 5e-8)])
@pytest.mark.parametrize("N0,N1,S", [(8, 16, 1), (240, 176, 1), (512, 512, 2)])
def test_reduced(N0, N1, S, precision, tol):
    import qdng_amd as Q
    print("[gpu case] grid", precision, N0, N1, S, flush=True)

    def make(c):
        p = box(N0, N1, S, S == 1)
        return p, Q.Cheby(p.gpu_ham(c), 2.0, prec=1e-10, precision=precision)
    check(both(make, 4, True), tol)


@pytest.mark.parametrize("N0,N1,S", [(16, 8, 1), (104, 88, 2), (256, 256, 1)])
def test_imaginary_time(N0, N1, S):
    import qdng_amd as Q
    print("[gpu case] grid imaginary", N0, N1, S, flush=True)

    def make(c):
        p = box(N0, N1, S)
        H = p.gpu_ham(c)
        lo, hi = H.bounds()
        return p, Q.Cheby(H, 3.0 / (hi - lo), prec=1e-10, imag=True)
    # the series cancels down to exp(-R dt) = e^-3 of its terms
    check(both(make, 3, False))


@pytest.mark.parametrize("N0,N1", [(40, 24), (256, 128)])
def test_nip_backward_fixed_series(N0, N1):
    import qdng_amd as Q
    print("[gpu case] grid nip / backward / prec 0", N0, N1, flush=True)

    def nip(c):
        p = box(N0, N1, 1, nip=True)
        return p, Q.Cheby(p.gpu_ham(c), 2.0)
    check(both(nip, 3, True))

    def back(c):
        p = box(N0, N1, 1, laser=True)
        U = Q.Cheby(p.gpu_ham(c), 2.0, prec=0.0)
        U.backward()
        return p, U
    check(both(back, 3, True))


def test_long_run_and_own_autocorrelation(ctx):
    """More orders than one launch takes; a psi0 that is psi itself follows
    the propagation."""
    import qdng_amd as Q
    p = box(32, 24, 1, laser=True, nt=300)
    U = Q.Cheby(p.gpu_ham(ctx), 2.0, prec=1e-12)
    w, ref, w0 = p.gpu_wf(ctx), p.gpu_wf(ctx), p.gpu_wf(ctx)
    n2, ac, nh, _ = U.run(w, 0, 250, w0)
    for i in range(250):
        U.apply(ref, i)
    assert np.array_equal(w.download(), ref.download())
    assert len(nh) == 250 and min(nh) > 3
    n2, ac, _, _ = U.run(w, 0, 3, w)
    assert np.allclose(ac, n2, rtol=1e-12)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-11), ("fp32", 1e-5)])
@pytest.mark.parametrize("N0,N1,S,laser,coupled", [
    (8, 8, 1, False, False), (8, 16, 2, False, True), (104, 88, 1, True, False), (40, 56, 2, False, False),
    (16, 768, 1, True, False), (768, 16, 2, False, True), (240, 176, 1, True, False), (232, 248, 2, False, True),
    (256, 256, 1, False, False), (768, 512, 1, True, False), (512, 512, 2, False, True), (768, 768, 2, False, True)])
def test_gspo(N0, N1, S, laser, coupled, precision, tol):
    """Runs of odd and even length from an odd step on, single steps, the
    observables in both layouts."""
    import qdng_amd as Q
    print("[gpu case] grid gspo", N0, N1, S, laser, coupled, precision, flush=True)

    def make(c):
        p = box(N0, N1, S, laser, coupled=coupled)
        ops = [p.gpu_split_op(c, [k]) for k in (("kin", "pot", "dip") if laser else ("kin", "pot"))]
        return p, Q.GSPO(ops, 2.0, precision=precision)
    check(both(make, 5, True), tol)
    check(both(make, 8, True), tol)
    check(both(make, 3, False), tol)


def test_gspo_steps_and_runs_agree(ctx):
    """Single steps give the bits of a run longer than one launch; backward
    steps lead back; a psi0 that is psi itself stands for the initial state."""
    import qdng_amd as Q
    p = box(40, 24, 1, laser=True, nt=2100)
    G = Q.GSPO([p.gpu_split_op(ctx, [k]) for k in ("kin", "pot", "dip")], 0.5)
    w, ref, w0 = p.gpu_wf(ctx), p.gpu_wf(ctx), p.gpu_wf(ctx)
    _, ac, _, _ = G.run(w, 0, 2060, w0)
    for i in range(2060):
        G.apply(ref, i)
    assert np.array_equal(w.download(), ref.download())
    self = p.gpu_wf(ctx)
    _, ac_self, _, _ = G.run(self, 0, 50, self)
    assert np.allclose(ac_self, ac[:50], rtol=1e-11)
    G.backward()
    G.run(w, 2059, 1)
    G.run(w, 2058, 1)
    G.backward(False)
    G.run(w, 2058, 2)
    assert rel(w.download(), ref.download()) < 1e-12


@pytest.mark.parametrize("imag", [False, True])
@pytest.mark.parametrize("N0,N1,S,order", [(8, 8, 1, 20), (40, 24, 2, 20), (16, 768, 1, 5), (192, 256, 1, 20),
                                           (232, 88, 2, 32), (104, 88, 1, 3), (64, 64, 1, 33)])
def test_lanczos(N0, N1, S, order, imag):
    """Converged and truncated series, one more vector than the kernel takes.
    The Lanczos vectors lose their orthogonality at rounding level over the
    order, by far less than 1e-10 of the state."""
    import qdng_amd as Q
    print("[gpu case] grid lanczos", N0, N1, S, order, imag, flush=True)

    def make(c):
        p = box(N0, N1, S, laser=not imag)
        H = p.gpu_ham(c)
        lo, hi = H.bounds()
        return p, Q.SIL(H, 2.0 / (hi - lo), order=order, imag=imag)
    check(both(make, 3, True), 1e-10)
    check(both(make, 2, False), 1e-10)


# every radix of the line filter's two stages that the shapes above leave out
# (R2 5, 7, 9, 13 to 17, 19, 23; R3 9, 14, 15), along either dimension
RADICES = [(160, 72), (168, 112), (144, 120), (336, 16), (600, 16), (16, 1024), (136, 184), (152, 208)]


@pytest.mark.parametrize("N0,N1", [s for n in RADICES for s in (n, n[::-1])])
@pytest.mark.parametrize("kind", ["cheby", "gspo"])
def test_against_the_oracle(N0, N1, kind):
    """The oracle's bounds of the other propagator tests."""
    import qdng_amd as Q
    from oracle import oracle as O
    print("[gpu case] grid oracle", N0, N1, kind, flush=True)
    c = Q.Context(0)
    try:
        p = box(N0, N1, 1, True)
        w, psi = p.gpu_wf(c), p.psi0.copy()
        if kind == "cheby":
            lo, hi = p.gpu_ham(c).bounds()
            dt = 20.0 / (hi - lo)
            _, _, nh, _ = Q.Cheby(p.gpu_ham(c), dt, prec=1e-12).run(w, 0, 3)
            U = O.Cheby(p.oracle_ham(), dt, prec=1e-12)
            assert list(nh) == [U.step(psi, i) for i in range(3)]
        else:
            kinds = ("kin", "pot", "dip")
            Q.GSPO([p.gpu_split_op(c, [k]) for k in kinds], 2.0).run(w, 0, 3)
            U = O.GSPO([p.oracle_split_op([k]) for k in kinds], 2.0, 1)
            for i in range(3):
                U.step(psi, i)
        assert c.persistent_stats() == (1, 0)
        assert rel(w.download(), psi) < (1e-10 if kind == "cheby" else 1e-12)
        del w
    finally:
        c.close()


@pytest.mark.parametrize("N,kind,precision", [(N, k, q) for N, k in [
    ([64, 24], "cheby"), ([64, 24], "gspo"), ([64, 24], "sil"), ([128], "cheby"), ([128], "gspo"), ([16, 64, 16], "cheby")]
    for q in (("fp64",) if k == "sil" else ("fp64", "fp32"))])
def test_a_set_plan_is_used(N, kind, precision):
    """A radix plan that the caller set for a side selects the kernels that
    transform by plans, as 4 or 8 line points do: here the same kernels, so the
    same bits."""
    import qdng_amd as Q
    print("[gpu case] set plan", N, kind, precision, flush=True)

    def run(plan, points):
        c = Q.Context(0)
        try:
            c.set_line_points(points)
            if plan:
                c.set_radix_plan(64 if 64 in N else 128, plan, precision)
            p = cases.Problem(N, [-6.0] * len(N), [6.0] * len(N))
            x = p.axes()
            r2 = sum(a ** 2 for a in x)
            p.kinetic(0, [1500.0] * len(N))
            p.potential(0, 0, np.minimum(0.03 * r2, 1.0))
            p.psi0 = cases.normalized(p, np.exp(-r2 + 0.5j * x[0]))
            if kind == "gspo":
                U = Q.GSPO([p.gpu_split_op(c, [k]) for k in ("kin", "pot")], 1.0, precision=precision)
            else:
                H = p.gpu_ham(c)
                lo, hi = H.bounds()
                U = Q.SIL(H, 2.0 / (hi - lo)) if kind == "sil" else \
                    Q.Cheby(H, 20.0 / (hi - lo), prec=1e-10, precision=precision)
            w = p.gpu_wf(c)
            U.run(w, 0, 2)
            launches = c.persistent_stats()[0]
            out = w.download()
            del U, w
            return out, launches
        finally:
            c.close()

    plan = [4, 4, 4] if 64 in N else [4, 8, 4]
    points = 8 if len(N) == 1 and kind == "gspo" else 4
    a, na = run(plan, 0)
    b, nb = run(plan, points)
    d, nd = run(None, 0)
    assert na == nb == 0
    assert nd > 0 or len(N) != 2
    assert np.array_equal(a, b)
    assert not np.array_equal(a, d) and rel(a, d) < (1e-11 if precision == "fp64" else 1e-5)


def propagator(c, kind, precision="fp64", nt=12):
    """(problem, propagator) on 40 x 24 points (two blocks), a few orders per step"""
    import qdng_amd as Q
    laser = kind not in ("imag", "gspo2")
    p = box(40, 24, 2 if kind == "gspo2" else 1, laser, nt=nt)
    if kind.startswith("gspo"):
        ops = [p.gpu_split_op(c, [k]) for k in (("kin", "pot", "dip") if laser else ("kin", "pot"))]
        return p, Q.GSPO(ops, 0.5, precision=precision)
    H = p.gpu_ham(c)
    lo, hi = H.bounds()
    if kind == "sil":
        return p, Q.SIL(H, 2.0 / (hi - lo))
    return p, Q.Cheby(H, 3.0 / (hi - lo), prec=1e-12, precision=precision, imag=kind == "imag")


# The steps of a launch that gave up are those of the per-order kernels: the
# bounds of the comparisons above.  FP32 split operator: each step rounds psi to
# 2^-24 about five times, 3e-7, which adds up like a random walk over 2100 steps
# to 1.4e-5; 1e-4 leaves a factor of seven.
@pytest.mark.parametrize("skip", [0, 1])
@pytest.mark.parametrize("kind,precision,steps,tol", [
    ("cheby", "fp64", 300, 1e-11), ("cheby", "fp32", 300, 1e-4), ("cheby", "compact", 300, 5e-7),
    ("gspo", "fp64", 2100, 1e-11), ("gspo", "fp32", 2100, 1e-4), ("gspo2", "fp64", 2100, 1e-11),
    ("gspo2", "fp32", 2100, 1e-4), ("sil", "fp64", 3, 1e-10)])
def test_launch_that_gives_up_in_a_run(kind, precision, steps, tol, skip):
    """A launch of a run of several gives up (the first or the second): its
    steps go by the per-order kernels, the launches behind it are persistent
    again, and the report is whole."""
    import qdng_amd as Q
    print("[gpu case] grid give-up", kind, precision, steps, skip, flush=True)
    out = []
    for points in (0, 8):
        c = Q.Context(0)
        try:
            c.set_line_points(points)
            p, U = propagator(c, kind, precision, steps + 2)
            w, w0 = p.gpu_wf(c), p.gpu_wf(c)
            c.set_short_launches(skip, 1)
            n2, ac, nh, _ = U.run(w, 1, steps, w0)
            out.append((w.download(), np.array(n2), np.array(ac), list(nh)))
            launches, missed = c.persistent_stats()
            assert (missed == 1 and launches >= 2) if points == 0 else launches == 0
            del U, w, w0
        finally:
            c.close()
    check(out, tol)


@pytest.mark.parametrize("kind,precision,tol", [("cheby", "fp64", 1e-11), ("cheby", "compact", 5e-8),
                                                ("cheby", "fp32", 1e-5), ("imag", "fp64", 1e-11)])
def test_single_steps_that_give_up(kind, precision, tol):
    """Three misses in a row: 64 steps go by the per-order kernels, then the
    launches are tried again."""
    import qdng_amd as Q
    print("[gpu case] grid give-up, single steps", kind, precision, flush=True)
    c, d = Q.Context(0), Q.Context(0)
    try:
        d.set_line_points(8)
        p, U = propagator(c, kind, precision, 80)
        _, V = propagator(d, kind, precision, 80)
        w, v = p.gpu_wf(c), p.gpu_wf(d)
        c.set_short_launches(0, 3)
        want = [1, 2, 3] + [3] * 64 + [4, 5]
        for i, n in enumerate(want):
            assert U.apply(w, i).n_hpsi == V.apply(v, i).n_hpsi
            assert c.persistent_stats() == (n, min(n, 3))
            if i in (0, 3, 68):
                assert rel(w.download(), v.download()) < tol * (i + 1)
            w.normalize()
            v.normalize()
        del U, V, w, v
    finally:
        c.close()
        d.close()


def test_short_launch_arguments(ctx):
    import qdng_amd as Q
    for bad in [(-1, 1), (0, -1)]:
        with pytest.raises(Q.QdxError):
            ctx.set_short_launches(*bad)


def test_threads():
    """Four contexts in four threads, two grids that share the chip and two
    that need all of it: the bits of runs one after the other, no launch gives
    up."""
    import threading

    import qdng_amd as Q
    print("[gpu case] grid threads", flush=True)
    shapes = [(64, 64, 1, "cheby"), (256, 64, 1, "gspo"), (512, 512, 2, "cheby"), (256, 256, 1, "sil")]

    def start(N0, N1, S, kind):
        c = Q.Context(0)
        p = box(N0, N1, S)
        H = p.gpu_ham(c)
        lo, hi = H.bounds()
        if kind == "gspo":
            U = Q.GSPO([p.gpu_split_op(c, [k]) for k in ("kin", "pot")], 0.5)
        else:
            U = Q.SIL(H, 2.0 / (hi - lo)) if kind == "sil" else Q.Cheby(H, 20.0 / (hi - lo), prec=1e-10)
        return c, U, p.gpu_wf(c), p.gpu_wf(c)

    def work(prog, out):
        c, U, w, w0 = prog
        w.copy_from(w0)
        for i in range(6):
            U.run(w, i * 20, 20, w0)
        out.append(w.download())

    progs = [start(*s) for s in shapes]
    try:
        alone, together = [[] for _ in shapes], [[] for _ in shapes]
        for g, o in zip(progs, alone):
            work(g, o)
        threads = [threading.Thread(target=work, args=a) for a in zip(progs, together)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert all(np.array_equal(a, b) for a, b in zip(alone, together))
        assert all(g[0].persistent_stats()[1] == 0 for g in progs)
    finally:
        ctxs = [g[0] for g in progs]
        progs.clear()
        for c in ctxs:
            c.close()

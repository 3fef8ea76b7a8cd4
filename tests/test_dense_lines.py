"""Short 1D lines with the kinetic operator as a dense circulant matrix
(qdx_dense.hip) against the line-transform kernels, which
qdx_ctx_set_line_points(8) selects, at the edges of the row blocks (N = 64 nb
and 8 more), for every number of states, both kinds of time, the negative
imaginary potential, fields, runs and single steps.  Both evaluate the same
series in FP64: an H application differs by a few 1e-16 of the kinetic range,
a series of order k by about k times that, so 1e-11 bounds a few steps of a
few hundred orders; the series lengths are equal."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu
TOL = 1e-11


def rel(a, b):
    return np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(b)


def line(N, S, laser=False, coupled=True, nip=False, nt=12):
    p = cases.Problem([N], [-6.0], [6.0], nstates=S)
    x = p.axes()[0]
    for s in range(S):
        if s != 2:   # the third state has no kinetic term
            p.kinetic(s, 1500.0 + 300 * s)
        p.potential(s, s, np.minimum(0.03 * (1 + 0.3 * s) * (x - 0.2 * s) ** 2 + 0.01 * s, 1.0))
    if S > 1 and coupled:
        p.potential(0, 1, 0.02 * np.exp(-x ** 2))
    if laser:
        E = 0.01 * np.cos(0.3 * np.arange(nt))
        p.dipole(1 if S > 1 else 0, 0, x * np.exp(-x ** 2 / 8), E)
    if nip:
        p.gobbler(0, 0, rp={0: 4.0}, order=5, gain=0.02, nip=True)
    g = np.exp(-(x - 0.4) ** 2 + 0.8j * x)
    p.psi0 = cases.normalized(p, np.concatenate([(1 - 0.2j * s) * g for s in range(S)]))
    return p


def both(make, steps, run):
    """(final state, norms, autocorrelations, counts) by the dense and by the
    line-transform kernels."""
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


def check(pair):
    (a, na, aa, ha), (b, nb, ab, hb) = pair
    assert ha == hb
    assert rel(a, b) < TOL
    assert np.max(np.abs(na - nb) / nb) < TOL and np.max(np.abs(aa - ab)) < TOL * max(1.0, np.max(np.abs(ab)))


@pytest.mark.parametrize("N,S", [(8, 1), (64, 1), (72, 1), (128, 1), (136, 1), (256, 1), (264, 1), (384, 1), (392, 1),
                                 (440, 1), (512, 1), (16, 2), (128, 2), (200, 2), (256, 2), (40, 3), (128, 3),
                                 (64, 4), (120, 4)])
@pytest.mark.parametrize("laser", [False, True])
def test_cheby(N, S, laser):
    import qdng_amd as Q
    print("[gpu case] dense cheby", N, S, laser, flush=True)

    def make(c):
        p = line(N, S, laser)
        return p, Q.Cheby(p.gpu_ham(c), 2.0, prec=1e-12)
    check(both(make, 5, True))
    check(both(make, 2, False))


@pytest.mark.parametrize("N,S", [(64, 1), (200, 1), (256, 2), (512, 1), (128, 4)])
def test_cheby_imaginary_time(N, S):
    import qdng_amd as Q
    print("[gpu case] dense imaginary", N, S, flush=True)

    def make(c):
        p = line(N, S)
        H = p.gpu_ham(c)
        lo, hi = H.bounds()
        return p, Q.Cheby(H, 3.0 / (hi - lo), prec=1e-10, imag=True)
    # the series cancels down to exp(-R dt) = e^-3 of its terms
    check(both(make, 3, False))


@pytest.mark.parametrize("N", [72, 256, 512])
def test_cheby_nip_backward_fixed_series(N):
    import qdng_amd as Q
    print("[gpu case] dense nip / backward / prec 0", N, flush=True)

    def nip(c):
        p = line(N, 1, nip=True)
        return p, Q.Cheby(p.gpu_ham(c), 2.0)
    check(both(nip, 3, True))

    def back(c):
        p = line(N, 1, laser=True)
        U = Q.Cheby(p.gpu_ham(c), 2.0, prec=0.0)
        U.backward()
        return p, U
    check(both(back, 3, True))


@pytest.mark.parametrize("N,S,laser,coupled", [(8, 1, False, False), (64, 1, True, False), (200, 1, True, False),
                                               (256, 1, False, False), (384, 1, True, False), (72, 2, False, True),
                                               (256, 2, False, True), (256, 2, False, False), (128, 4, False, False)])
def test_gspo(N, S, laser, coupled):
    import qdng_amd as Q
    print("[gpu case] dense gspo", N, S, laser, coupled, flush=True)

    def make(c):
        p = line(N, S, laser, coupled)
        ops = [p.gpu_split_op(c, [k]) for k in (("kin", "pot", "dip") if laser else ("kin", "pot"))]
        return p, Q.GSPO(ops, 2.0)
    check(both(make, 9, True))
    check(both(make, 1, False))


def test_clock_beyond_the_field(ctx):
    """The steps before the last field value run, then the error is raised."""
    import qdng_amd as Q
    p = line(128, 1, laser=True, nt=4)
    U = Q.Cheby(p.gpu_ham(ctx), 2.0)
    w, ref = p.gpu_wf(ctx), p.gpu_wf(ctx)
    with pytest.raises(Q.QdxError):
        U.run(w, 0, 6)
    U.run(ref, 0, 4)
    assert np.array_equal(w.download(), ref.download())


@pytest.mark.parametrize("N,S,kind,steps", [(512, 1, "cheby", 250), (256, 2, "cheby", 400), (128, 4, "cheby", 400),
                                            (384, 1, "gspo", 9000), (256, 2, "gspo", 6000)])
def test_launches_are_short(N, S, kind, steps):
    """A long run comes in launches of about 10 ms: another context's
    persistent launch waits 0.1 s for the CU.  Twice that covers a clock
    that has not ramped up."""
    import qdng_amd as Q
    print("[gpu case] dense launch length", N, S, kind, flush=True)
    c = Q.Context(0)
    try:
        p = line(N, S)
        if kind == "cheby":
            H = p.gpu_ham(c)
            lo, hi = H.bounds()
            U = Q.Cheby(H, 50.0 / (hi - lo), prec=1e-10)
        else:
            U = Q.GSPO([p.gpu_split_op(c, [k]) for k in ("kin", "pot")], 0.5)
        w = p.gpu_wf(c)
        c.profile(True)
        U.run(w, 0, steps)
        n, ms = c.kernel_time(Q.K_CHEBY_ROW if kind == "cheby" else Q.K_GSPO_ROW)
        c.profile(False)
        assert ms > 20.0, "the run is too short to need two launches"
        assert ms / n < 20.0
        del U, w
    finally:
        c.close()

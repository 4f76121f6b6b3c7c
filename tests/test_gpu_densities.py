"""Moments, momentum expectation values and the energy from the densities
along the axes (k_marginal) against numpy's transforms, at the shortest and
longest axes, fewer pencils than a workgroup holds, more tiles than
workgroups, and a packet far from the origin in x and k (whose second
moments would cancel if they were not taken about the mean)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(2,), (16,), (4096,), (2, 2), (4096, 2), (8, 4096), (64, 512), (2, 4, 2), (16, 2, 256), (128, 64, 32),
          (32, 256, 128)]


@pytest.mark.parametrize("shape", SHAPES)
def test_observables_match_numpy(shape):
    from atus2_amd import hip
    d = len(shape)
    L = [9.0, 8.0, 7.0][:d]
    dx, dk = [l / n for l, n in zip(L, shape)], [2 * np.pi / l for l in L]
    rng = np.random.default_rng(2)
    ax = lambda v, a: v.reshape([-1 if b == a else 1 for b in range(d)])
    x = [ax((np.arange(n) - n // 2) * dx[a], a) for a, n in enumerate(shape)]
    k = [ax(((np.arange(n) + n // 2) % n - n // 2) * dk[a], a) for a, n in enumerate(shape)]
    psis = []
    for c in range(2):
        p = 1e-3 * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
        g = np.ones(shape, complex)
        for a, n in enumerate(shape):
            # a packet at x = L/4, k at half the band
            g = g * np.exp(-((x[a] - L[a] / 4) / (0.05 * L[a])) ** 2 + 1j * (n // 4) * dk[a] * x[a])
        psis.append(p + g)
    V = rng.uniform(0, 3, (2,) + shape)
    gs, alpha = [2.0, 0.7, 0.5, 1.5], [0.5, 0.3, 0.2][:d]
    ar, ark = np.prod(dx), np.prod(dk)
    dens = [np.abs(p) ** 2 for p in psis]
    spec = [np.abs(np.fft.fftn(p)) ** 2 * (ar / (2 * np.pi) ** (d / 2)) ** 2 for p in psis]
    e = sum(ark * np.sum(sum(alpha[a] * k[a] ** 2 for a in range(d)) * s) for s in spec)
    e += sum(ar * np.sum((V[i] + 0.5 * (gs[2 * i] * dens[0] + gs[2 * i + 1] * dens[1])) * dens[i]) for i in range(2))
    # sums of positive terms over at most 2^20 points and transforms of at
    # most 12 stages per axis: 1e-13; first moments may cancel, so they are
    # held against the sums of their absolute terms
    with hip.Context(shape, dx, dk, 2) as ctx:
        for c in range(2):
            ctx.upload(c, psis[c])
            ctx.set_potential(c, V[c])
        ctx.set_g(gs)
        ctx.set_alpha(alpha)
        assert abs(ctx.energy() / e - 1) < 1e-13
        for c in range(2):
            ek, m = ctx.expval_k(c), ctx.moments(c)
            N = ar * dens[c].sum()
            assert abs(m["N"] / N - 1) < 1e-13
            ph = np.sum(np.angle(psis[c]) * dens[c])
            assert abs(m["phase"] * dens[c].sum() - ph) < 1e-13 * np.sum(np.abs(np.angle(psis[c])) * dens[c])
            for a in range(d):
                for got, q, w in ((ek[a], k[a], ark * spec[c]), (m["k"][a], k[a], ark * spec[c] / N),
                                  (m["x"][a], x[a], ar * dens[c] / N)):
                    assert abs(got - np.sum(q * w)) < 1e-13 * np.sum(np.abs(q) * w)
                for got, q, w, mu in ((m["k2"][a], k[a], ark * spec[c] / N, m["k"][a]),
                                      (m["x2"][a], x[a], ar * dens[c] / N, m["x"][a])):
                    # the mean's own error enters to first order times the
                    # remaining first moment about it
                    assert abs(got / np.sum((q - mu) ** 2 * w) - 1) < 1e-12


@pytest.mark.parametrize("shape", [(64,), (32, 16), (16, 8, 64)])
def test_mu_with_inconsistent_dk(orc, shape):
    from atus2_amd import hip
    d = len(shape)
    g = orc.make_grid(shape, L=[8.0, 7.0, 6.0][:d])
    for a in range(d):
        g.dk[a] *= 1.02
    rng = np.random.default_rng(3)
    psi = [rng.standard_normal(shape) + 1j * rng.standard_normal(shape) for _ in range(2)]
    V = [rng.uniform(0, 2, shape) for _ in range(2)]
    gs = np.array([[3.0, 1.0], [0.5, 2.0]])
    S = orc.SobSolver(g, psi, V, gs, [0.5, 0.4], stepsize=0.01)
    with hip.Context.from_grid(g, 2) as ctx:
        for i in range(2):
            ctx.upload(i, psi[i])
            ctx.set_potential(i, V[i])
        ctx.set_g(gs.ravel())
        ctx.sob_setup([0.5, 0.4], 0.01)
        assert np.allclose(ctx.sob_mu(), S.mu(), rtol=1e-12, atol=0)


@pytest.mark.parametrize("c", [0.1, 0.3, 1 / 3])
def test_long_axes_add_no_error(c):
    # 4096 equal densities one after another in a double are off by hundreds
    # of units of 2^-53 (N and the second moment); the sums here are exact up
    # to a handful of roundings of their results
    from fractions import Fraction as Fr
    from atus2_amd import hip
    n, dx = 4096, 0.013
    with hip.Context((n,), [dx], [2 * np.pi / (n * dx)], 1) as ctx:
        ctx.upload(0, np.full(n, c, np.complex128))
        m = ctx.moments(0)
    d, x = Fr(c * c), [Fr((j - n // 2) * dx) for j in range(n)]
    mu = sum(x) / n
    u = Fr(1, 2 ** 53)
    assert abs(Fr(m["N"]) / (Fr(dx) * d * n) - 1) < 4 * u
    assert abs(Fr(m["x2"][0]) / (sum((q - mu) ** 2 for q in x) / n) - 1) < 8 * u


@pytest.mark.parametrize("c", [0.1, 0.7])
def test_phase_sum_in_a_tree(c):
    # 2^21 equal terms: 8 of a pencil, 2 tiles and 8 levels of a workgroup in
    # a double, the rest in long double; atan2, the density, their product,
    # the quotient by the sum and N's factor add a rounding or two each.  One
    # after another in the workgroup and over the workgroups they are 43-48
    # units off
    from fractions import Fraction as Fr
    from atus2_amd import hip
    shape, dx = (128, 128, 128), 0.125
    with hip.Context(shape, [dx] * 3, [2 * np.pi / 16] * 3, 1) as ctx:
        ctx.upload(0, np.full(shape, c + 1j * c))
        m = ctx.moments(0)
    total = Fr(m["phase"]) * Fr(m["N"]) / Fr(dx) ** 3
    ref = Fr(np.pi / 4) * 2 * Fr(c) ** 2 * 2 ** 21
    assert abs(total / ref - 1) < Fr(8 + 1 + 8 + 7, 2 ** 53)

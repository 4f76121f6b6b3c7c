"""The passes of the Sobolev loop at the edges of their ranges, against the
oracle: the shortest axes and fewer columns than a wavefront, long axes, 1D
grids from the shortest to the longest pencil, more partial sums than one
workgroup takes, two wave functions, and a transform pair whose dk is not
2 pi / (n dx)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# a transform and its inverse leave a few rounding errors per stage (12
# stages at most), an iteration three of them: 1e-14 of the state's norm per
# iteration.  The residual is a difference of terms of its own size here
# (the starts are far from converged).
ITS = 3
TOL = ITS * 1e-14


@pytest.mark.parametrize("nw", [1, 2])
@pytest.mark.parametrize("shape", [(2,), (8,), (16,), (256,), (4096,), (2, 2), (4, 2, 2), (64, 4), (4, 4096), (2048, 8),
                                   (8, 16, 64), (32, 2, 16), (16, 512, 2)])
def test_iterations_match_oracle(orc, shape, nw):
    _compare(orc, shape, nw, 1.0, ITS)


def test_many_partial_sums(orc):
    # 2048 workgroups along axis 0: their sums take a launch of their own
    _compare(orc, (512, 64, 128), 1, 1.0, 1)


@pytest.mark.parametrize("shape", [(64,), (16, 32), (8, 16, 16)])
def test_inconsistent_dk(orc, shape):
    _compare(orc, shape, 1, 1.01, ITS)


def _compare(orc, shape, nw, stretch, its):
    from atus2_amd import hip
    d = len(shape)
    g = orc.make_grid(shape, L=[8.0, 7.0, 6.0][:d])
    for a in range(d):
        g.dk[a] *= stretch
    rng = np.random.default_rng(3)
    xs = orc.coords_x(g)
    V = [0.3 * (i + 1) * sum((1 + 0.2 * a) * x ** 2 for a, x in enumerate(xs)) * np.ones(shape) for i in range(nw)]
    psi = []
    for i in range(nw):
        p = np.exp(-sum(x ** 2 for x in xs) / (3.0 + i)) * np.ones(shape)
        psi.append((p + 0.01 * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))).astype(np.complex128))
    gs = [12.0] if nw == 1 else [12.0, 4.0, 3.0, 9.0]
    alpha = [0.5, 0.4][:nw]
    S = orc.SobSolver(g, psi, V, np.reshape(gs, (nw, nw)), alpha, stepsize=0.01)
    S.renormalize()
    with hip.Context.from_grid(g, nw) as ctx:
        for i in range(nw):
            ctx.upload(i, psi[i])
            ctx.set_potential(i, V[i])
        ctx.set_g(gs)
        ctx.sob_setup(alpha, 0.01)
        ctx.sob_renormalize()
        done, r, log = ctx.sob_iterate(its)
        assert done == its
        for k in range(its):
            ref = S.iterate()
            assert abs(log[k, 3] / ref - 1) < 1e-12, k
            assert bool(log[k, 2]) == bool(S.s.renormalised)
        assert r == log[-1, 3]
        for i in range(nw):
            e = np.linalg.norm(ctx.download(i) - S.psi[i]) / np.linalg.norm(S.psi[i])
            assert e < TOL, (i, e)
        assert np.allclose(ctx.sob_mu(), S.mu(), rtol=1e-12, atol=0)

"""The V pass of two components that holds both in one thread (states above 80
MiB, or 16 values per thread tuned at any size), between the first and the
last step of a block, over the lengths of the last axis."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LARGE = [(512, 512, 16), (1024, 64, 64), (4096, 1024), (2048, 2048), (1024, 4096)]  # 128 MiB of state
SMALL = [(16, 2), (4, 8, 8), (16, 4, 32), (64, 128), (32, 512), (8, 1024), (4, 2048), (4, 4096)]


def _blocks_match(orc, shape, rm, kind):
    from atus2_amd import hip
    d = len(shape)
    L = [40.0, 30.0, 36.0][:d]
    g = orc.make_grid(shape, L=L)
    xs = orc.coords_x(g)
    rng = np.random.default_rng(12)
    env = np.exp(-0.5 * sum((x / (3.0 + a)) ** 2 for a, x in enumerate(xs))) * np.ones(shape)
    psis = [(w * env + 1e-3 * rng.standard_normal(shape)).astype(np.complex128) for w in (1.0, 0.4)]
    gs, dt, alpha, lk = [8.0, 6.0, 6.0, 7.0], 1e-3, [0.5] * d, 6 * np.pi / L[0]
    par = dict(beta0=0.02, deltaL=[0.0, 0.7], amp0=5.0, laser_k=lk, laser_domh=8.0, laser_dk=0.05)
    pots = [(0.01 * (c + 1) * sum(x ** 2 for x in xs)) * np.ones(shape) for c in range(2)] if kind == "freeprop" else None
    amp = (lambda t: 1.0 - t) if kind == "bragg_ad" else None
    S = orc.RTSolver(g, psis, gs, alpha, dt=dt, pots=pots, amp=amp, **par)
    S.block({"bragg_ad": orc.BRAGG_AD, "freeprop": orc.FREEPROP, "freeprop_if": orc.FREEPROP_IF}[kind], 3)
    las = hip.laser(**dict(par, deltaL=tuple(par["deltaL"])))
    with hip.Context.from_grid(g, 2) as ctx:
        for f in hip.KFAM:
            ctx.tune(f, rm)
        for c in range(2):
            ctx.upload(c, psis[c])
            if pots:
                ctx.set_potential(c, pots[c])
        ctx.set_g(gs)
        ctx.set_alpha(alpha)
        ctx.run_block({"bragg_ad": hip.STEP_BRAGG_AD, "freeprop": hip.STEP_FREEPROP, "freeprop_if": hip.STEP_FREEPROP_IF}[kind],
                      dt, 3, 0.0, las, amp)
        err = np.sqrt(sum(np.linalg.norm(ctx.download(c) - S.psis[c]) ** 2 for c in range(2)) /
                      sum(np.linalg.norm(S.psis[c]) ** 2 for c in range(2)))
    # three steps of at most six transforms; the Bragg exponential loses
    # digits where the coupling nearly vanishes
    assert err < (1e-11 if kind == "bragg_ad" else 1e-13), err


@pytest.mark.parametrize("rm", [8, 16])
@pytest.mark.parametrize("shape", LARGE)
def test_large_states(orc, shape, rm):
    _blocks_match(orc, shape, rm, "bragg_ad")


@pytest.mark.parametrize("kind", ["bragg_ad", "freeprop", "freeprop_if"])
@pytest.mark.parametrize("shape", SMALL)
def test_sixteen_values_at_any_size(orc, shape, kind):
    _blocks_match(orc, shape, 16, kind)


@pytest.mark.parametrize("batch", [False, True])
def test_the_tuned_values_reach_the_pass(batch):
    # the plans of 8 and 16 values round differently, and nothing else here
    # depends on the family's setting
    from atus2_amd import hip
    shape, out = (64, 128), []
    rng = np.random.default_rng(1)
    psi = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    for rm in (8, 16):
        with (hip.BatchContext(shape, [0.1, 0.1], [0.5, 0.5], 1) if batch else
              hip.Context(shape, [0.1, 0.1], [0.5, 0.5], 2)) as ctx:
            ctx.tune("vfuse", rm)
            for c in range(2):
                ctx.upload(c, psi)
            ctx.set_alpha([0.5, 0.5])
            las = hip.laser(amp0=1.0, laser_k=1.0, laser_domh=1.0)
            if batch:
                ctx.set_runs([[1.0, 0.9, 0.9, 1.0]], [las])
                ctx.run_batch_block(hip.STEP_BRAGG_AD, 1e-3, 4, 0.0)
            else:
                ctx.set_g([1.0, 0.9, 0.9, 1.0])
                ctx.run_block(hip.STEP_BRAGG_AD, 1e-3, 4, 0.0, las)
            out.append(ctx.download(0))
    assert not np.array_equal(out[0], out[1])
    assert np.linalg.norm(out[0] - out[1]) < 1e-11 * np.linalg.norm(out[0])

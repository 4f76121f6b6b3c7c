"""Blocks of several components (k_vcomp in 2D/3D, k_bcomp in 1D) against the
same steps taken one at a time (half kinetic, V, kinetic, ... by
atus_v_step / atus_v_step_ds and atus_kinetic), at the shortest and longest
last axes of their ranges, the lengths beyond them that take the separate
passes, odd workgroup fills and one or two species."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NK = 4
# the two sides do the same operations, rounded differently at most where
# multiply-adds are fused: some 50 rounding errors of 1.1e-16 per step and
# point at the worst.  The closed-form Bragg exponentials lose up to three
# digits near the nodes of the coupling.
TOL, TOL_BRAGG = NK * 5e-15, NK * 5e-12

KINDS = [("freeprop", 2, True), ("freeprop", 3, False), ("freeprop", 4, True), ("if", 2, True), ("if", 3, False),
         ("if", 4, False), ("if2", 2, True), ("if2", 4, True), ("ds", 4, True), ("double", 3, False),
         ("num", 2, True), ("num", 3, False), ("raman", 3, False), ("raman", 4, False)]


@pytest.mark.parametrize("kind,nc,two", KINDS + [("freeprop", 2, False), ("if", 2, False), ("bragg", 2, False)])
@pytest.mark.parametrize("shape", [(2, 2), (8, 4), (4, 8), (16, 16), (2, 1024), (2, 2048), (2, 4096), (64, 256),
                                   (2, 4, 8), (8, 2, 32), (4, 16, 512), (256, 512)])
def test_2d_3d_blocks_equal_single_steps(shape, kind, nc, two):
    _compare(shape, kind, nc, two)


@pytest.mark.parametrize("kind,nc,two", KINDS + [("bragg", 2, False)])
@pytest.mark.parametrize("n", [2, 8, 16, 64, 1024, 2048, 4096])
def test_1d_blocks_equal_single_steps(n, kind, nc, two):
    _compare((n,), kind, nc, two)


def _compare(shape, kind, nc, two):
    from atus2_amd import hip
    d = len(shape)
    L = [20.0, 16.0, 18.0][:d]
    dx, dk = [l / n for l, n in zip(L, shape)], [2 * np.pi / l for l in L]
    rng = np.random.default_rng(11)
    psi = [rng.standard_normal(shape) + 1j * rng.standard_normal(shape) for _ in range(nc)]
    pot = rng.uniform(0, 5, shape)
    las = hip.laser(amp0=5.0, amp1=3.0, laser_k=1.1, laser_domh=0.6, chirp_rate0=0.2, phase0=0.3, beta0=0.05,
                    beta=(0.03, -0.02, 0.01), deltaL=(0.0, -0.7, 0.4, 0.3))
    las2 = hip.laser(amp0=3.0, laser_k=0.7, laser_domh=0.5, laser_dk=0.1, beta0=-0.04)
    dt, t0, dur = 1e-3, 0.1, (1.0, 0.1 + 2.5e-3)
    step = {"freeprop": hip.STEP_FREEPROP, "if": hip.STEP_FREEPROP_IF, "if2": hip.STEP_FREEPROP_IF,
            "ds": hip.STEP_BRAGG_AD, "bragg": hip.STEP_BRAGG_AD, "double": hip.STEP_DOUBLE_BRAGG,
            "num": hip.STEP_NUM_BRAGG, "raman": hip.STEP_RAMAN}[kind]
    species = kind in ("if2", "ds")
    out = []
    for block in (True, False):
        with hip.Context(shape, dx, dk, nc) as ctx:
            for c in range(nc):
                ctx.upload(c, psi[c])
            if kind == "freeprop":
                ctx.set_potential(nc - 1, pot)
            ctx.set_g(np.linspace(0.5, 2.0, nc * nc))
            ctx.set_alpha([0.5, 0.4, 0.3][:d])
            if two and nc % 2 == 0:
                ctx.set_alpha2([0.2, 0.3, 0.6][:d])
            t = t0
            if block:
                t = ctx.run_block_ds(step, dt, NK, t, las, las2, 0.0, dur) if species else \
                    ctx.run_block(step, dt, NK, t, las)
            else:
                ctx.kinetic(0.5, dt)
                t += 0.5 * dt
                for m in range(1, NK + 1):
                    if species:
                        ctx.v_step_ds(step, dt, t, las, las2, 0.0, dur)
                    else:
                        ctx.v_step(step, dt, t, las)
                    ctx.kinetic(1.0 if m < NK else 0.5, dt)
                    t += dt if m < NK else 0.5 * dt
            out.append((t, np.stack([ctx.download(c) for c in range(nc)])))
    assert out[0][0] == out[1][0]
    e = np.linalg.norm(out[0][1] - out[1][1]) / np.linalg.norm(out[1][1])
    assert e < (TOL_BRAGG if kind in ("ds", "bragg", "double") else TOL), e


@pytest.mark.parametrize("runs", [1, 3, 70])
@pytest.mark.parametrize("n", [16, 256, 2048])
def test_batched_1d_blocks_equal_single_runs(n, runs):
    from atus2_amd import hip
    rng = np.random.default_rng(5)
    dx, dk = [40.0 / n], [2 * np.pi / 40.0]
    psi = rng.standard_normal((2 * runs, n)) + 1j * rng.standard_normal((2 * runs, n))
    gs = rng.uniform(1, 3, (runs, 4))
    las = [hip.laser(amp0=float(rng.uniform(1, 5)), laser_k=1.0, laser_domh=0.5) for _ in range(runs)]
    F = rng.uniform(0.5, 1.0, (NK, runs))
    with hip.BatchContext((n,), dx, dk, runs) as B:
        for c in range(2 * runs):
            B.upload(c, psi[c])
        B.set_alpha([0.5])
        B.set_runs(gs, las)
        B.run_batch_block(hip.STEP_BRAGG_AD, 1e-3, NK, 0.0, F)
        got = np.stack([B.download(c) for c in range(2 * runs)])
    for r in {0, runs // 2, runs - 1}:
        it = iter(F[:, r])
        with hip.Context((n,), dx, dk, 2) as S:
            S.upload(0, psi[2 * r])
            S.upload(1, psi[2 * r + 1])
            S.set_g(gs[r])
            S.set_alpha([0.5])
            S.run_block(hip.STEP_BRAGG_AD, 1e-3, NK, 0.0, las[r], lambda t: next(it))
            ref = np.stack([S.download(0), S.download(1)])
        e = np.linalg.norm(got[2 * r:2 * r + 2] - ref) / np.linalg.norm(ref)
        assert e < TOL_BRAGG, (r, e)

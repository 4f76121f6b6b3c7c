"""1D blocks in one launch (k_block1d, atus_set_resident): the block of a
single run, of a batch and of a replayed graph agrees with the block run
with a launch per step, for every pencil length up to 4096, both
values-per-thread choices and the fused V kinds; blocks of changing length
reuse and regrow the step tables.  The arithmetic is the same, but the
compiler may fuse multiply-adds differently inside the step loop than across
separate launches, so the two paths agree to rounding, not bit for bit:
within 1e-13 relative L2 after a block, or 100 times the difference that
inputs changed in the last bits make.  The Bragg closed form (bragg.cpp
eigenvector normalisation) loses digits where the coupling nearly vanishes,
so it amplifies rounding differences injected at every step; a replayed graph of the resident
block equals the eager resident block exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from atus2_amd import hip as H
    H.load()
    return H


def _state(orc, g, ncomp, seed):
    x = orc.coords_x(g)[0]
    rng = np.random.default_rng(seed)
    base = np.exp(-0.5 * (x / 3.0) ** 2)
    out = []
    for c in range(ncomp):
        psi = base * (1.0 if c == 0 else 0.4) + 1e-3 * (rng.standard_normal(base.shape)
                                                         + 1j * rng.standard_normal(base.shape))
        out.append(psi.astype(np.complex128))
    return out


TOL = 1e-13


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _box(n):
    # dx >= 1/4: the kinetic phase of the highest mode stays below 0.1 per
    # step, so rounding differences are not amplified by unresolved modes
    return [max(24.0, 0.25 * n)]


def _amp(t):
    return float(np.exp(-0.5 * ((t - 0.03) / 0.02) ** 2))


KINDS = ["freeprop1", "freeprop2", "freeprop_if1", "freeprop_if2", "bragg_ad"]


def _ctx(hip, orc, g, kind, rm, resident, seed=3, perturb=False):
    n = int(g.n[0])
    ncomp = 1 if kind.endswith("1") else 2
    ctx = hip.Context.from_grid(g, ncomp)
    for c, p in enumerate(_state(orc, g, ncomp, seed)):
        if perturb:
            # inputs changed in the last bits: the noise floor of the dynamics
            p = p * (1 + 2e-16 * np.random.default_rng(99 + c).standard_normal(p.shape))
        ctx.upload(c, p)
    ctx.set_alpha([0.5])
    ctx.set_g([10.0] if ncomp == 1 else [100.0, 95.0, 95.0, 100.0])
    if kind.startswith("freeprop") and not kind.startswith("freeprop_if"):
        x = orc.coords_x(g)[0]
        for c in range(ncomp):
            ctx.set_potential(c, 0.5 * (1.0 + 0.1 * c) * x ** 2 * np.ones(n))
    ctx.tune("kin", rm)
    ctx.set_resident(resident)
    return ctx, ncomp


def _kind(hip, kind):
    if kind == "bragg_ad":
        return hip.STEP_BRAGG_AD
    return hip.STEP_FREEPROP_IF if kind.startswith("freeprop_if") else hip.STEP_FREEPROP


LAS = dict(amp0=5.0, laser_k=1.3, laser_domh=8.0, beta0=0.02, deltaL=(0.0, 0.3), chirp_rate0=0.1, phase0=0.2)


@pytest.mark.parametrize("n", [2, 16, 64, 256, 1024, 2048, 4096])
@pytest.mark.parametrize("rm", [8, 16])
@pytest.mark.parametrize("kind", KINDS)
def test_resident_block_equals_step_launches(hip, orc, n, rm, kind):
    g = orc.make_grid((n,), L=_box(n))
    las = hip.laser(**LAS)
    hk = _kind(hip, kind)
    amp = _amp if kind == "bragg_ad" else None
    a, nc = _ctx(hip, orc, g, kind, rm, True)
    b, _ = _ctx(hip, orc, g, kind, rm, False)
    p, _ = _ctx(hip, orc, g, kind, rm, False, perturb=True)
    try:
        ta = tb = tp = 0.0
        # block lengths that grow and shrink the step tables
        for Nk in (7, 40, 1, 3):
            ta = a.run_block(hk, 1e-3, Nk, ta, las, amp)
            tb = b.run_block(hk, 1e-3, Nk, tb, las, amp)
            tp = p.run_block(hk, 1e-3, Nk, tp, las, amp)
            assert ta == tb == tp
            for c in range(nc):
                d = rel(a.download(c), b.download(c))
                tol = max(TOL, 100 * rel(p.download(c), b.download(c)))
                assert d <= tol, (Nk, c, d, tol)
    finally:
        a.close()
        b.close()
        p.close()


def test_resident_block_matches_the_oracle(hip, orc):
    # the 1D rt_solver workload's step on a short block, against the oracle
    n, L, dt, Nk = 4096, 80.0, 1e-3, 50
    g = orc.make_grid((n,), L=L)
    x = orc.coords_x(g)[0]
    rng = np.random.default_rng(1)
    psi = (np.pi ** -0.25 * np.exp(-0.5 * x ** 2) + 1e-3 * (rng.standard_normal(n)
                                                           + 1j * rng.standard_normal(n))).astype(np.complex128)
    V = 0.5 * x ** 2
    S = orc.RTSolver(g, [psi], [10.0], [0.5], dt=dt, pots=[V])
    with hip.Context.from_grid(g, 1) as ctx:
        ctx.upload(0, psi)
        ctx.set_g([10.0])
        ctx.set_alpha([0.5])
        ctx.set_potential(0, V)
        t = 0.0
        for _ in range(2):
            S.block(orc.FREEPROP, Nk)
            t = ctx.run_block(hip.STEP_FREEPROP, dt, Nk, t)
            assert t == S.t
        out = ctx.download(0)
    err = np.linalg.norm(out - S.psis[0]) / np.linalg.norm(S.psis[0])
    assert err < 1e-12, err


@pytest.mark.parametrize("n,rm", [(64, 16), (1024, 8), (1024, 16), (4096, 16)])
@pytest.mark.parametrize("kind", ["bragg", "freeprop_if"])
def test_resident_batch_equals_step_launches(hip, orc, n, rm, kind):
    g = orc.make_grid((n,), L=_box(n))
    nb, dt, Nk = 5, 1e-3, 12
    rng = np.random.default_rng(4)
    gsl = [[gg, 0.95 * gg, 0.95 * gg, gg] for gg in rng.uniform(1, 200, nb)]
    lasers = [hip.laser(amp0=a, laser_k=1.3, laser_domh=d, deltaL=(0.0, 0.2 * r))
              for r, (a, d) in enumerate(zip(rng.uniform(1, 10, nb), rng.uniform(6, 10, nb)))]
    sig = rng.uniform(0.01, 0.03, nb)
    hk = hip.STEP_BRAGG_AD if kind == "bragg" else hip.STEP_FREEPROP_IF
    bs = []
    # resident, a launch per step, and a launch per step from inputs
    # changed in the last bits (the noise floor)
    for resident, perturb in ((True, False), (False, False), (False, True)):
        B = hip.BatchContext((n,), [g.dx[0]], [g.dk[0]], nb)
        for r in range(nb):
            p = _state(orc, g, 2, 20 + r)
            for c in range(2):
                q = p[c] * (1 + 2e-16 * np.random.default_rng(99 + c).standard_normal(n)) if perturb else p[c]
                B.upload(2 * r + c, q)
        B.set_alpha([0.5])
        B.set_runs(gsl, lasers)
        B.tune("kin", rm)
        B.set_resident(resident)
        bs.append(B)
    try:
        t = [0.0, 0.0, 0.0]
        for blk, nk in enumerate((Nk, 30, 2)):
            t1 = np.array(bs[0].step_times(t[0], dt, nk))[:, None]
            F = np.exp(-0.5 * ((t1 - 0.02) / sig[None, :]) ** 2)
            for i, B in enumerate(bs):
                t[i] = B.run_batch_block(hk, dt, nk, t[i], F)
            assert t[0] == t[1] == t[2]
            for c in range(2 * nb):
                d = rel(bs[0].download(c), bs[1].download(c))
                tol = max(TOL, 100 * rel(bs[2].download(c), bs[1].download(c)))
                assert d <= tol, (blk, c, d, tol)
    finally:
        for B in bs:
            B.close()


@pytest.mark.parametrize("n", [256, 4096])
def test_graph_of_a_resident_block(hip, orc, n):
    # replays equal the eager resident block exactly and agree with a
    # launch per step to rounding
    g = orc.make_grid((n,), L=_box(n))
    las = hip.laser(**LAS)
    dt, Nk = 1e-3, 15
    a, _ = _ctx(hip, orc, g, "bragg_ad", 16, True)
    b, _ = _ctx(hip, orc, g, "bragg_ad", 16, True)
    s, _ = _ctx(hip, orc, g, "bragg_ad", 16, False)
    p, _ = _ctx(hip, orc, g, "bragg_ad", 16, False, perturb=True)
    try:
        with hip.Graph(a, hip.STEP_BRAGG_AD, dt, Nk, las) as G:
            ta = tb = ts = tp = 0.01
            for blk in range(3):
                F = np.array([_amp(t1) for t1 in hip.BatchContext.step_times(ta, dt, Nk)])
                ta = G.launch(ta, F)
                tb = b.run_block(hip.STEP_BRAGG_AD, dt, Nk, tb, las, _amp)
                ts = s.run_block(hip.STEP_BRAGG_AD, dt, Nk, ts, las, _amp)
                tp = p.run_block(hip.STEP_BRAGG_AD, dt, Nk, tp, las, _amp)
                assert ta == tb == ts == tp
                for c in range(2):
                    assert np.array_equal(a.download(c), b.download(c)), (blk, c)
                    d = rel(a.download(c), s.download(c))
                    tol = max(TOL, 100 * rel(p.download(c), s.download(c)))
                    assert d <= tol, (blk, c, d, tol)
                # eager work between replays, on the resident path too
                ta = a.run_block(hip.STEP_BRAGG_AD, dt, 4, ta, las, _amp)
                tb = b.run_block(hip.STEP_BRAGG_AD, dt, 4, tb, las, _amp)
                ts = s.run_block(hip.STEP_BRAGG_AD, dt, 4, ts, las, _amp)
                tp = p.run_block(hip.STEP_BRAGG_AD, dt, 4, tp, las, _amp)
    finally:
        for x in (a, b, s, p):
            x.close()


def test_set_resident_rejects_other_values(hip):
    with hip.Context((64,), [0.5], [2 * np.pi / 32], 1) as ctx:
        with pytest.raises(hip.AtusError, match="resident"):
            hip._check(hip._lib.atus_set_resident(ctx._h, 2))


@pytest.mark.parametrize("n,ncomp", [(1024, 1), (4096, 1), (256, 2)])
def test_phases_beyond_a_million(n, ncomp):
    """Resident blocks whose potential turns the phase by more than 10^6 per
    step on part of the grid, where the V step's sine takes the library's
    routine: against the same steps in numpy."""
    from atus2_amd import hip
    L, dt, nk = 20.0, 2.0 ** -13, 4
    dx, dk = L / n, 2 * np.pi / L
    x = (np.arange(n) - n // 2) * dx
    k = ((np.arange(n) + n // 2) % n - n // 2) * dk
    # powers of two, so that dt V is exact: 2^21 and 2^19
    V = np.where(np.abs(x) > 5, 2.0 ** 34, 2.0 ** 32) * np.where(x > 0, 1.0, -1.0)
    psis = [np.exp(-(x - 1 - c) ** 2 / 30).astype(np.complex128) for c in range(ncomp)]
    out = [p.copy() for p in psis]
    kin = lambda p, s: np.fft.ifft(np.fft.fft(p) * np.exp(-0.5j * s * dt * k ** 2))
    out = [kin(p, 0.5) for p in out]
    for m in range(nk):
        out = [kin(p * np.exp(-1j * (dt * V)), 1.0 if m + 1 < nk else 0.5) for p in out]
    with hip.Context((n,), [dx], [dk], ncomp) as ctx:
        for c in range(ncomp):
            ctx.upload(c, psis[c])
            ctx.set_potential(c, V)
        ctx.set_g([0.0] * ncomp ** 2)
        ctx.set_alpha([0.5])
        ctx.run_block(hip.STEP_FREEPROP, dt, nk, 0.0)
        for c in range(ncomp):
            # transforms and sines to rounding, four steps
            assert np.linalg.norm(ctx.download(c) - out[c]) < 1e-13 * np.linalg.norm(out[c])

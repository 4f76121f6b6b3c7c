"""A run of a batch gives the same bits whatever runs share the batch: the
kernels that round differently are chosen by one run's size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _advance(hip, g, shape, psi, runs, k0, thr):
    d = len(shape)
    with hip.BatchContext(shape, [g.dx[a] for a in range(d)], [g.dk[a] for a in range(d)], len(runs)) as B:
        for r in range(len(runs)):
            B.upload(2 * r, psi)
            B.upload(2 * r + 1, 0.3 * psi)
        B.set_alpha([0.5] * d)
        B.set_runs([[a, 0.95 * a, 0.95 * a, a] for a, _ in runs],
                   [hip.laser(amp0=5.0, laser_k=4.0, laser_domh=w, laser_dk=0.05) for _, w in runs])
        B.run_batch_block(hip.STEP_BRAGG_AD, 1e-3, 3, 0.0)
        rabi = B.batch_rabi_integrals(0, k0, thr)
        last = 2 * (len(runs) - 1)
        return B.download(last), B.download(last + 1), np.array(rabi[-1])


# runs: under and over 80 MiB and 2^21 values of state for the whole batch
@pytest.mark.parametrize("shape,runs", [((512, 512), 16), ((256, 2048), 6), ((64, 64, 64), 12), ((16, 32, 16), 300),
                                        ((8192,), 150), ((2048,), 40)])
def test_same_bits_alone_and_in_company(orc, shape, runs):
    from atus2_amd import hip
    d = len(shape)
    g = orc.make_grid(shape, L=[24.0] * d)
    xs = orc.coords_x(g)
    rng = np.random.default_rng(4)
    psi = np.exp(-sum(x ** 2 for x in xs) / 18.0) * np.ones(shape) + 0.01 * rng.standard_normal(shape)
    psi = psi.astype(np.complex128)
    par = [(10.0 + r, 6.0 + 0.1 * r) for r in range(runs)]
    k0 = [(0.0,) * d, (8.0,) + (0.0,) * (d - 1)]
    a = _advance(hip, g, shape, psi, par[-1:], k0, 1.5)
    b = _advance(hip, g, shape, psi, par, k0, 1.5)
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    if d == 3:
        # the box's populations; those of 1D and 2D grids are sums over
        # segments whose number of partials follows the batch
        assert np.array_equal(a[2], b[2])
    else:
        # sums of at most 2^19 squares
        assert np.allclose(a[2], b[2], rtol=1e-13, atol=0)

"""Rabi integrals of 3D grids over index boxes of few columns, whose last
pass holds all of them in one workgroup (its sums need whole wavefronts)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("thr", [0.6, 1.3, 2.2])
@pytest.mark.parametrize("shape", [(32, 16, 16), (64, 32, 16), (16, 16, 64), (512, 16, 32)])
def test_small_boxes_match_oracle(orc, shape, thr):
    from atus2_amd import hip
    g = orc.make_grid(shape, L=[2 * np.pi] * 3)  # dk = 1
    rng = np.random.default_rng(7)
    psi = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    with hip.Context.from_grid(g, 1) as ctx:
        ctx.upload(0, psi)
        got = ctx.rabi_integrals(0, [(0.0, 0.0, 0.0)], thr)
    # every mode within thr of k = 0 (threshold and modes are apart by 0.1
    # and more, so rounding does not decide membership)
    f = np.fft.fftn(psi) * np.prod([g.dx[a] for a in range(3)]) / (2 * np.pi) ** 1.5
    k = [np.fft.fftfreq(n, 1 / n) for n in shape]
    r = np.sqrt(k[0][:, None, None] ** 2 + k[1][None, :, None] ** 2 + k[2][None, None, :] ** 2)
    ref = np.sum(np.abs(f[r < thr]) ** 2)
    # sums of at most 33 squares of transforms of at most 2^18 terms
    assert abs(got[0] / ref - 1) < 1e-12

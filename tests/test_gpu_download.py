"""Downloads through the library's pinned pool: the sizes around its limits
(shorter copies, single pieces, several pieces, copies by several threads),
an odd component of many, and several threads at once (the pool serves one,
the others copy by themselves)."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 4096, 32768, 65536, 131072, 262144, 524288, 1048576])
def test_downloads_return_what_was_uploaded(n):
    from atus2_amd import hip
    rng = np.random.default_rng(n)
    psi = rng.standard_normal((3, n)) + 1j * rng.standard_normal((3, n))
    with hip.Context((n,), [0.1], [0.1], 3) as ctx:
        for c in range(3):
            ctx.upload(c, psi[c])
        for c in (2, 0, 1, 1):
            assert np.array_equal(ctx.download(c), psi[c])


def test_downloads_follow_the_context_s_work():
    from atus2_amd import hip
    rng = np.random.default_rng(1)
    psi = rng.standard_normal((128, 64, 128)) + 1j * rng.standard_normal((128, 64, 128))
    with hip.Context(psi.shape, [0.1] * 3, [0.1] * 3, 1) as ctx:
        for k in range(3):
            ctx.upload(0, psi * (k + 1))
            ctx.snapshot_save(0)
            ctx.upload(0, psi * 0)
            ctx.snapshot_restore(0)
            assert np.array_equal(ctx.download(0), psi * (k + 1))


def test_several_threads_at_once():
    from atus2_amd import hip
    shapes = [(1048576,), (64, 128, 128), (65536,), (512, 512)]
    bad = []

    def work(i, shape):
        rng = np.random.default_rng(i)
        psi = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
        d = len(shape)
        with hip.Context(shape, [0.1] * d, [0.1] * d, 1) as ctx:
            ctx.upload(0, psi)
            for _ in range(10):
                if not np.array_equal(ctx.download(0), psi):
                    bad.append(i)

    th = [threading.Thread(target=work, args=(i, s)) for i, s in enumerate(shapes)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad

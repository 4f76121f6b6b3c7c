"""The warm-start network's products at the edges of their 64 x 64 x 32
tiles (single rows, remainders in every direction, widths that are not a
multiple of four, a product split along k) and its training loop over more
steps than are enqueued at once, against the CPU restatement in
float64."""
import numpy as np
import pytest

from oracle import mlp_oracle as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("terms", [1, 3])
@pytest.mark.parametrize("dims,batch", [((1, 1, 1, 1, 1), 1), ((4, 64, 32, 64, 128), 64), ((5, 33, 70, 17, 131), 65),
                                        ((3, 65, 31, 63, 129), 1), ((4, 16, 16, 17, 4100), 70),
                                        ((130, 66, 64, 20, 36), 257)])
def test_forward_and_gradients(dims, batch, terms):
    from atus2_amd import hip
    rng = np.random.default_rng(8)
    with hip.Net(dims, max_batch=batch, seed=3) as net:
        net.set_precision(terms)
        p = (net.get_params() + 0.05 * rng.standard_normal(net.nparams)).astype(np.float32)
        net.set_params(p)
        x = rng.uniform(-1, 1, (batch, dims[0])).astype(np.float32)
        t = rng.standard_normal((batch, dims[4])).astype(np.float32)
        y = net.forward(x)
        loss, g = net.gradients(x, t)
    # against float64 throughout.  Operands of one bf16 term are off by
    # 2^-9, of a pair by 2^-17 at most; a product of two by twice that, the
    # forward pass by four layers' worth, a gradient by eight products'.
    # The loss is a mean of squares.
    u = 2.0 ** -9 if terms == 1 else 2.0 ** -17
    ref = M.forward(p, dims, x, None)[4]
    assert np.linalg.norm(y - ref) < 4 * 2 * u * np.linalg.norm(ref)
    lref, gref = M.loss_and_gradients(p, dims, x, t, None)
    assert abs(loss / lref - 1) < 2 * 4 * 2 * u
    for wo, ws, bo, bn in M.layout(dims)[0]:
        for o, n in ((wo, ws[0] * ws[1]), (bo, bn)):
            e = np.linalg.norm(g[o:o + n] - gref[o:o + n])
            assert e < 8 * 2 * u * np.linalg.norm(gref[o:o + n]), (o, n, e)


@pytest.mark.parametrize("dims,max_batch,batches", [((4, 256, 256, 64, 32768), 256, (128, 191, 192)),
                                                    ((4, 256, 256, 64, 32768), 200, (101, 128, 192)),
                                                    ((4, 64, 256, 256, 32768), 65, (33, 64)),
                                                    ((4, 16, 16, 17, 4100), 300, (1, 64, 128, 193, 256)),
                                                    ((4, 65, 17, 64, 130), 2100, (511, 512, 1000, 2100))])
def test_batches_below_the_largest(dims, max_batch, batches):
    # fewer rows of tiles are split into more parts along k: the workspace
    # holds those of every batch, not of the largest alone.  Tolerances as in
    # test_forward_and_gradients.
    from atus2_amd import hip
    rng = np.random.default_rng(5)
    u = 2.0 ** -17
    with hip.Net(dims, max_batch=max_batch, seed=3) as net:
        p = net.get_params()
        for batch in batches:
            x = rng.uniform(-1, 1, (batch, dims[0])).astype(np.float32)
            t = rng.standard_normal((batch, dims[4])).astype(np.float32)
            net.set_params(p)
            loss, g = net.gradients(x, t)
            lref, gref = M.loss_and_gradients(p, dims, x, t, None)
            assert abs(loss / lref - 1) < 2 * 4 * 2 * u
            for wo, ws, bo, bn in M.layout(dims)[0]:
                for o, n in ((wo, ws[0] * ws[1]), (bo, bn)):
                    e = np.linalg.norm(g[o:o + n] - gref[o:o + n])
                    assert e < 8 * 2 * u * np.linalg.norm(gref[o:o + n]), (batch, o, n, e)
            net.set_data(x, t)
            assert abs(net.train(1, batch, 1e-3)[0] / lref - 1) < 2 * 4 * 2 * u


@pytest.mark.parametrize("dims", [(4, 16, 16, 16, 16), (3, 65, 17, 8, 33)])
def test_gradients_of_large_batches_add_in_parts(dims):
    # 65536 equal rows: the mean's scale is a power of two, so every addend of
    # a gradient is 2^-16 of the one row's, exactly, and the gradients differ
    # by what the sums round off.  A column sum adds 32 / 4 values of 8 slices
    # in a thread, 4 threads, at most 64 splits in a wavefront and 4
    # wavefronts; a weight 8 slices of 3 products of 32 terms, then the same.
    # One after another the columns' threads add 16384 values each, off by
    # 1e-4 and more.
    from atus2_amd import hip
    big = 65536
    rng = np.random.default_rng(6)
    x = rng.uniform(-1, 1, (1, dims[0])).astype(np.float32)
    t = rng.standard_normal((1, dims[4])).astype(np.float32)
    g = []
    with hip.Net(dims, max_batch=big, seed=3) as net:
        for rows in (1, big):
            g.append(net.gradients(np.repeat(x, rows, 0), np.repeat(t, rows, 0))[1].astype(np.float64))
    for wo, ws, bo, bn in M.layout(dims)[0]:
        w, b = slice(wo, wo + ws[0] * ws[1]), slice(bo, bo + bn)
        assert np.all(np.abs(g[1][b] - g[0][b]) <= (64 + 4 + 64 + 4) * 2.0 ** -24 * np.abs(g[0][b]))
        assert np.all(np.abs(g[1][w] - g[0][w]) <= (8 * 3 * 33 + 64 + 4) * 2.0 ** -24 * np.abs(g[0][w]) + 1e-38)


def test_training_in_chunks_equals_single_steps():
    # 300 steps run as two chunks; the same steps one call each give the
    # same losses (constant rate, the whole set as one batch)
    from atus2_amd import hip
    rng = np.random.default_rng(1)
    dims = (4, 16, 16, 8, 40)
    x = rng.uniform(-1, 1, (24, 4)).astype(np.float32)
    t = rng.standard_normal((24, 40)).astype(np.float32)
    out = []
    for single in (False, True):
        with hip.Net(dims, max_batch=24, seed=2) as net:
            net.set_data(x, t)
            if single:
                # every call reshuffles: a batch is a permutation of the set
                losses = np.concatenate([net.train(1, 24, 1e-3, 1e-3, seed=k) for k in range(300)])
            else:
                losses = net.train(300, 24, 1e-3, 1e-3, seed=1)
            out.append(losses)
    # the permutations only reorder fp32 sums; Adam carries the difference
    assert np.max(np.abs(out[0] / out[1] - 1)) < 1e-3


def test_a_loss_that_is_not_finite_stops_training():
    from atus2_amd import hip
    dims = (2, 8, 8, 8, 16)
    with hip.Net(dims, max_batch=4, seed=2) as net:
        p0 = net.get_params()
        net.set_data(np.zeros((4, 2), np.float32), np.full((4, 16), np.nan, np.float32))
        with pytest.raises(hip.AtusError, match="not finite"):
            net.train(5, 4, 1e-3)
        assert np.array_equal(net.get_params(), p0)
        # and the next run, on good data, trains
        net.set_data(np.zeros((4, 2), np.float32), np.ones((4, 16), np.float32))
        assert np.all(np.isfinite(net.train(5, 4, 1e-3)))
        assert not np.array_equal(net.get_params(), p0)

"""BatchNorm's results to the bit, in both directions.

Behind many Relu layers a last bit of one BatchNorm call decides on which side of zero single values fall, and a network's gradients
move by 1e-3: so which product of a sum is rounded by itself and which is fused, in which order, belongs to a call's results.  The digests
are those of the calls' results on an MI355X, recorded from the plain calls while the compiler still chose the fused products; every later
form of the kernels has to give the same."""
import zlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one-pass kernels of 16, 32 and 64 values a thread; ranges of 16-byte words, with read-ahead loops and remainders; ranges without words
SHAPES = [(2, 3, 5, 5), (16, 4, 14, 14), (32, 4, 15, 15), (32, 6, 17, 17), (16, 3, 32, 32), (8, 4, 112, 112), (16, 3, 71, 71)]
GOLDEN = {
    (2, 3, 5, 5): (1803107568, 3230562865, 1183227773, 1171934599),
    (16, 4, 14, 14): (3954799238, 3671639413, 239292508, 3001953959),
    (32, 4, 15, 15): (2466055982, 49538025, 2270622261, 3741949911),
    (32, 6, 17, 17): (204916229, 279849675, 1670038264, 1180378973),
    (16, 3, 32, 32): (2237242307, 4129929770, 1863065929, 1882697053),
    (8, 4, 112, 112): (613838288, 2268043695, 4016568529, 2412863682),
    (16, 3, 71, 71): (2639025669, 1539595629, 2947938412, 1927376946),
}


def digests(shape):
    """(forward, gradient from saved statistics, gradient without, the fused pair's gradient from saved statistics)"""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx = nd.gpu(0)
    rng = np.random.RandomState(sum(shape))
    c = shape[1]
    x, dy = [nd.array(rng.normal(size=shape).astype(np.float32), ctx) for _ in range(2)]
    gamma, beta = [nd.array(rng.normal(size=(1, c, 1, 1)).astype(np.float32), ctx) for _ in range(2)]
    y, dx = nd.empty(shape, ctx), nd.empty(shape, ctx)
    mean, istd, dg, db = [nd.empty((1, c, 1, 1), ctx) for _ in range(4)]

    def digest(*arrays):
        crc = 0
        for a in arrays:
            crc = zlib.crc32(np.ascontiguousarray(a.asnumpy()).tobytes(), crc)
        return crc
    L.CuDNN_Batch_Normalization(x, gamma, beta, y, mean, istd, 0.99, 0.01)
    out = [digest(y, mean, istd)]
    for saved in ((mean, istd), (None, None)):
        L.CuDNN_Batch_Normalization_gradient(dy, x, gamma, dx, dg, db, *saved, 0.01)
        out.append(digest(dx, dg, db))
    L.batch_norm_relu(x, gamma, beta, y, mean, istd, 0.01)
    L.batch_norm_relu_gradient(dy, x, gamma, beta, dx, dg, db, mean, istd, 0.01)
    return tuple(out + [digest(y, mean, istd, dx, dg, db)])


@pytest.mark.parametrize("shape", SHAPES)
def test_results_keep_their_bits(shape):
    assert digests(shape) == GOLDEN[shape]


# the same kernels, planes of whole words in memory order (56 x 56 and 112 x 112) and short planes in words (4 x 4)
@pytest.mark.parametrize("shape", SHAPES + [(1030, 3, 4, 4), (16, 3, 56, 56)])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_pair_passes_on_nan_as_the_two_calls_do(shape, bad):
    """A NaN or an infinity makes its channel's statistics NaN: the gradients of BatchNorm + Relu in one call, with saved doubles or with
    both layers' arrays, are NaN where those of the two calls are, beta's among them."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx = nd.gpu(0)
    rng = np.random.RandomState(sum(shape))
    c = shape[1]
    x = rng.normal(size=shape).astype(np.float32)
    x[1, 1, 1, 1] = bad
    gx, dy = nd.array(x, ctx), nd.array(rng.normal(size=shape).astype(np.float32), ctx)
    gamma, beta = [nd.array(rng.normal(size=(1, c, 1, 1)).astype(np.float32), ctx) for _ in range(2)]
    bn, y, dbn = [nd.empty(shape, ctx) for _ in range(3)]

    def gradients():
        return nd.empty(shape, ctx), nd.empty((1, c, 1, 1), ctx), nd.empty((1, c, 1, 1), ctx)
    two, one, both = gradients(), gradients(), gradients()
    L.CuDNN_Batch_Normalization(gx, gamma, beta, bn, None, None, 0.99, 0.01)
    L.relu(bn, y)
    L.relu_gradient(bn, dy, dbn)
    L.CuDNN_Batch_Normalization_gradient(dbn, gx, gamma, *two, None, None, 0.01)
    assert np.isnan(two[2].asnumpy()[0, 1]) and np.isfinite(two[2].asnumpy()[0, [0, 2]]).all()
    y1, mean, istd = nd.empty(shape, ctx), nd.empty((c, 2), ctx), nd.empty((c, 2), ctx)
    L.batch_norm_relu(gx, gamma, beta, y1, mean, istd, 0.01)
    L.batch_norm_relu_gradient(dy, gx, gamma, beta, *one, mean, istd, 0.01)
    pair, bn1, r1, dbn1 = nd.empty((c, 2), ctx), nd.empty(shape, ctx), nd.empty(shape, ctx), nd.empty(shape, ctx)
    L.batch_norm_then_relu(gx, gamma, beta, bn1, r1, pair, None, None, 0.01)
    L.batch_norm_then_relu_gradient(dy, gx, gamma, pair, dbn1, *both, None, None, 0.01)
    for got, want in [(y1, y), (bn1, bn), (r1, y), (dbn1, dbn)] + list(zip(one, two)) + list(zip(both, two)):
        np.testing.assert_array_equal(got.asnumpy(), want.asnumpy())


# planes in words and not, a channel in registers and not
@pytest.mark.parametrize("shape", [(16, 4, 14, 14), (8, 4, 112, 112), (16, 3, 71, 71)])
def test_a_tape_that_is_asked_to_fuse_takes_saved_floats_and_one_that_is_not_gives_the_bits_of_two_calls(shape):
    from tsplit_amd import gpu_links as L, graph, ndarray as nd
    ctx = nd.gpu(0)
    rng = np.random.RandomState(sum(shape))
    c = shape[1]
    x, dy = [nd.array(rng.normal(size=shape).astype(np.float32), ctx) for _ in range(2)]
    gamma, beta = [nd.array(rng.normal(size=(1, c, 1, 1)).astype(np.float32), ctx) for _ in range(2)]
    bn, y, dbn, dx = [nd.empty(shape, ctx) for _ in range(4)]
    mean, istd, dg, db = [nd.empty((1, c, 1, 1), ctx) for _ in range(4)]
    want = {}
    L.batch_norm_relu(x, gamma, beta, y, mean, istd, 0.01)
    L.batch_norm_relu_gradient(dy, x, gamma, beta, dx, dg, db, mean, istd, 0.01)
    want[True] = [a.asnumpy() for a in (y, dx, dg, db)]
    L.CuDNN_Batch_Normalization(x, gamma, beta, bn, None, None, 0.99, 0.01)
    L.relu(bn, y)
    L.relu_gradient(bn, dy, dbn)
    L.CuDNN_Batch_Normalization_gradient(dbn, x, gamma, dx, dg, db, None, None, 0.01)
    want[False] = [a.asnumpy() for a in (y, dx, dg, db)]
    for fuse in (True, False):
        t = graph.Tape(graph.GpuBackend(ctx))
        t.fuse_bn_relu = fuse
        leaves = [t.param(v, v.shape) for v in (x, gamma, beta)]
        out = t.bn_then_relu(*leaves)
        assert [n.out is out for n in t._nodes] == [True]
        t._nodes[0].back(dy)
        for a, b in zip([out.value] + [v.grad for v in leaves], want[fuse]):
            np.testing.assert_array_equal(a.asnumpy(), b)

"""The one-pass BatchNorm kernels by where a channel's values lie: arrays off 16 bytes, planes of whole words and of single values at every count
of rows a wave takes, and planes too far apart for 32-bit offsets, in every form, hold the same bits.

A channel's result depends on its own values alone, so what is asked for is always the result of the same channels as planes of one value
on 16 bytes, whose rows the tests of the kernels' edges hold to float64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
FORMS = ["alone", "saved", "fused", "exact", "both", "sum"]


def _run(form, x, dy, more, gamma, beta, like):
    """y, dx and, where the form writes them, Relu's array and the gradient behind it; `like` makes an array of x's shape."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, c = nd.gpu(0), x.shape[1]
    y, dx, dg, db = like(), like(), nd.empty((1, c, 1, 1), ctx), nd.empty((1, c, 1, 1), ctx)
    small, wide = ([nd.empty(s, ctx) for _ in range(2)] for s in ((1, c, 1, 1), (c, 2)))
    got = [y, dx, dg, db]
    if form in ("alone", "saved"):
        stats = small if form == "saved" else (None, None)
        L.CuDNN_Batch_Normalization(x, gamma, beta, y, *stats, 0.99, 0.01)
        L.CuDNN_Batch_Normalization_gradient(dy, x, gamma, dx, dg, db, *stats, 0.01)
    elif form == "both":
        r, behind, pair = like(), like(), wide[0]
        L.batch_norm_then_relu(x, gamma, beta, y, r, pair)
        L.batch_norm_then_relu_gradient(dy, x, gamma, pair, behind, dx, dg, db)
        got += [r, behind]
    else:
        stats = small if form == "fused" else wide
        if form == "sum":
            L.batch_norm_relu_add(x, gamma, beta, more, y, *stats, 0.01)
        else:
            L.batch_norm_relu(x, gamma, beta, y, *stats, 0.01)
        L.batch_norm_relu_gradient(dy, x, gamma, beta, dx, dg, db, *stats, 0.01)
    return got


def _parameters(c, tile=1):
    from tsplit_amd import ndarray as nd
    rng = np.random.RandomState(c)
    return [nd.array(np.tile(v, (1, tile, 1, 1)), nd.gpu(0)) for v in rng.normal(size=(2, 1, c, 1, 1)).astype(np.float32)]


# values a channel: one row, the edges of 4, 8, 16, 32, 40, 48, 56 and 64 rows; planes of words, and of 1, 2, 3, 7 x 7 and 17 x 17 values
SHAPES = [(1, 3, 1, 1), (85, 2, 3, 1), (256, 3, 2, 2), (1025, 2, 1, 1), (257, 3, 2, 2), (64, 2, 4, 8), (65, 2, 4, 8), (2049, 2, 1, 1), (64, 5, 7, 7), (2048, 2, 2, 1), (64, 3, 8, 8), (585, 2, 7, 1), (167, 2, 7, 7), (32, 3, 16, 16),
          (1171, 2, 7, 1), (33, 3, 16, 16), (208, 2, 7, 7), (40, 2, 16, 16), (209, 3, 7, 7), (48, 2, 16, 16), (250, 2, 7, 7), (251, 3, 7, 7), (49, 2, 16, 16),
          (292, 2, 7, 7), (293, 3, 7, 7), (56, 2, 17, 17)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("form", FORMS)
def test_arrays_on_and_off_16_bytes_and_planes_of_one_value(form, shape):
    from tsplit_amd import ndarray as nd
    ctx, (n, c, h, w), rng = nd.gpu(0), shape, np.random.RandomState(7)
    values = [rng.normal(size=shape).astype(np.float32) for _ in range(3)]

    def placed(off):
        wholes = []

        def like(v=None):
            """An array of the shape, `off` floats behind a 16-byte boundary, with 7 around it."""
            whole = np.full((off + n * c * h * w + 8, 1), 7, np.float32)
            if v is not None:
                whole[off:off + v.size, 0] = v.ravel()
            whole, a = nd.array(whole, ctx), nd.empty(shape, ctx)
            wholes.append((a, a.handle.contents.data, whole))
            a.handle.contents.data = whole.handle.contents.data + 4 * off
            return a
        try:
            got = _run(form, *(like(v) for v in values), *_parameters(c), like)
            out = [v.asnumpy() for v in got]
            for _, _, whole in wholes:
                flat = whole.asnumpy().ravel()
                assert (flat[:off] == 7).all() and (flat[off + n * c * h * w:] == 7).all()
            return out
        finally:                                  # the arrays have their own memory back before they are freed
            for a, own, _ in wholes:
                a.handle.contents.data = own
    on = placed(0)
    for off in (1, 2, 3):
        for one, other in zip(on, placed(off)):
            np.testing.assert_array_equal(one, other)
    apart = [v.transpose(0, 2, 3, 1).reshape(-1, c, 1, 1) for v in values]
    ones = _run(form, *(nd.array(np.ascontiguousarray(v), ctx) for v in apart), *_parameters(c), lambda: nd.empty(apart[0].shape, ctx))
    for one, other in zip(on, ones):
        other = other.asnumpy()
        if other.shape[0] > 1 or one.shape != other.shape:
            other = other.reshape(n, h, w, c).transpose(0, 3, 1, 2)
        np.testing.assert_array_equal(one, other)


@pytest.mark.parametrize("form", FORMS)
def test_planes_2_gib_apart(form):
    """258 images of 2.1 million planes of one value, 60 different channels again and again: a channel's first rows reach beyond 2 GiB."""
    from tsplit_amd import ndarray as nd
    ctx, n, few, times = nd.gpu(0), 258, 60, 34834
    values = np.random.RandomState(2).normal(size=(3, n, few, 1, 1)).astype(np.float32)
    near = [v.asnumpy() for v in _run(form, *(nd.array(v, ctx) for v in values), *_parameters(few), lambda: nd.empty((n, few, 1, 1), ctx))]
    shape = (n, few * times, 1, 1)
    far = _run(form, *(nd.array(np.tile(v, (1, times, 1, 1)), ctx) for v in (values if form == "sum" else values[:2])), *([None] if form != "sum" else []),
               *_parameters(few, times), lambda: nd.empty(shape, ctx))
    for one, other in zip(near, far):
        got = other.asnumpy().reshape(other.shape[0], times, few)
        for i in range(other.shape[0]):
            assert (got[i] == one.reshape(-1, few)[i]).all(), i

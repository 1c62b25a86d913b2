"""The one-pass BatchNorm kernels where their rows of 256 values end: one value, one off a row, every number of rows a wave takes, planes of
whole words and not, of one to three values, and planes too far apart for 32-bit offsets.

Bars: the mean is that of 256 float sums in the order of the rows, to the bit; y within 8 roundings of float64 at its magnitude (the mean's and
the deviation's rounding, the two coefficients', the fused multiply-add's, on float sums of up to 64 values); gradients likewise, with the sums'
own m * 2^-24 / sqrt(m) walk below that."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(2, 3, 1, 1), (255, 3, 1, 1), (256, 2, 1, 1), (257, 2, 1, 1), (85, 2, 1, 3), (129, 5, 1, 2), (64, 2, 8, 8), (33, 3, 11, 11), (65, 2, 8, 8),
          (32, 2, 16, 16), (29, 3, 17, 17), (40, 2, 16, 16), (41, 2, 16, 16), (56, 2, 16, 16), (57, 3, 16, 16), (64, 2, 16, 16), (56, 2, 17, 17)]


def _mean(x):
    v = x.transpose(1, 0, 2, 3).reshape(x.shape[1], -1)
    rows = -(-v.shape[1] // 256)
    s = np.zeros((v.shape[0], 256), np.float32)
    v = np.pad(v, ((0, 0), (0, rows * 256 - v.shape[1]))).reshape(v.shape[0], rows, 256)
    for r in range(rows):
        s += v[:, r]
    return (s.astype(np.float64).sum(1) / (x.size // x.shape[1])).astype(np.float32)


@pytest.mark.parametrize("shape", SHAPES)
def test_both_directions(shape, rng):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, c = nd.gpu(0), shape[1]
    x, dy = (rng.normal(size=shape).astype(np.float32) + np.float32(0.25) for _ in range(2))
    gamma, beta = (rng.normal(size=(1, c, 1, 1)).astype(np.float32) for _ in range(2))
    gx, gdy, gg, gb = (nd.array(v, ctx) for v in (x, dy, gamma, beta))
    y, dx = nd.array(np.full(shape, 7, np.float32), ctx), nd.array(np.full(shape, 7, np.float32), ctx)
    mean, istd, dg, db = (nd.empty((1, c, 1, 1), ctx) for _ in range(4))
    L.CuDNN_Batch_Normalization(gx, gg, gb, y, mean, istd, 0.99, 0.01)
    np.testing.assert_array_equal(mean.asnumpy().ravel(), _mean(x))
    ax, x64, dy64 = (0, 2, 3), x.astype(np.float64), dy.astype(np.float64)
    mu, inv = x64.mean(ax, keepdims=True), 1 / np.sqrt(x64.var(ax, keepdims=True) + 0.01)
    hat, eps = (x64 - mu) * inv, 2.0 ** -24
    assert (np.abs(y.asnumpy() - (gamma * hat + beta)) <= 8 * eps * (np.abs(gamma) * inv * (np.abs(x64) + np.abs(mu)) + np.abs(beta) + 1)).all()
    for saved in ((mean, istd), (None, None)):
        L.CuDNN_Batch_Normalization_gradient(gdy, gx, gg, dx, dg, db, *saved, 0.01)
        want_b, want_g = dy64.sum(ax, keepdims=True), (dy64 * hat).sum(ax, keepdims=True)
        m = x.size // c
        want = gamma * inv * (dy64 - want_b / m - hat * want_g / m)
        assert (np.abs(db.asnumpy() - want_b) <= 66 * eps * np.abs(dy64).sum(ax, keepdims=True)).all()
        assert (np.abs(dg.asnumpy() - want_g) <= 140 * eps * (np.abs(dy64) * (np.abs(x64) + np.abs(mu)) * inv).sum(ax, keepdims=True)).all()
        scale = np.abs(gamma) * inv * (np.abs(dy64) + np.abs(dy64).mean(ax, keepdims=True) + (np.abs(x64) + np.abs(mu)) * inv)
        assert (np.abs(dx.asnumpy() - want) <= 300 * eps * (scale + 1)).all()


def test_planes_2_gib_apart():
    """258 images of 2.1 million planes of one value: the planes of a channel's first row reach beyond 2 GiB."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, n, c = nd.gpu(0), 258, 2_090_000
    v = np.random.RandomState(1).randint(-8, 9, n).astype(np.float32)
    gx = nd.array((v[:, None] + (np.arange(c, dtype=np.float32) % 5)[None]).reshape(n, c, 1, 1), ctx)
    gy = nd.empty((n, c, 1, 1), ctx)
    L.CuDNN_Batch_Normalization(gx, nd.array(np.ones((1, c, 1, 1), np.float32), ctx), nd.array(np.zeros((1, c, 1, 1), np.float32), ctx), gy,
                                None, None, 0.99, 0.01)
    want = ((v - v.astype(np.float64).mean()) / np.sqrt(v.astype(np.float64).var() + 0.01)).astype(np.float32)
    y = gy.asnumpy().reshape(n, c)
    for i in range(n):
        assert np.abs(y[i] - want[i]).max() <= 1e-5, i

"""The tile kernel of the convolutions (csrc/conv_tile.h), forward and data gradient, at the edges of its tiles, of its blocks of 8
channels, its bit masks of 32 and 64 taps and its words: against float64.  The second argument of a case: the forward pass also
leaves the output's channel sums.

Bar: an output is a sum of K = channels x taps fp32 products, in whatever order: within K * 2^-24 of the sum of their magnitudes
(gamma_K to first order), one more 2^-24 for each of up to 32 ranges' results added by the fold.  A channel sum adds P output values,
at most 64 of them in fp32: their error and (64 + 1) * 2^-24 of the sum of the magnitudes."""
import numpy as np
import pytest

from oracle import ops as O

pytestmark = pytest.mark.gpu

# N, C, H, W, O, kh, kw, ph, pw, stride; sums
CASES = [
    ((1, 40, 1, 1, 1, 1, 1, 0, 0, 1), False),       # one value
    ((3, 64, 8, 8, 65, 1, 1, 0, 0, 1), True),       # one row past a tile; a dense operand in words
    ((2, 130, 7, 9, 64, 1, 1, 0, 0, 1), True),      # planes that are not whole words
    ((2, 36, 9, 7, 130, 1, 1, 0, 0, 2), False),     # one tap, stride 2: odd planes, dx written in twos
    ((3, 33, 8, 16, 34, 1, 1, 0, 0, 2), False),     # the same in words of two columns
    ((2, 40, 8, 8, 20, 1, 1, 1, 1, 1), False),      # one tap with padding
    ((2, 5, 11, 13, 9, 5, 5, 2, 2, 1), False),      # few channels: depth in the filter's order, 25 taps
    ((2, 17, 9, 10, 12, 3, 3, 1, 1, 1), True),      # 24 = 17 + 7 padded channels
    ((2, 41, 10, 9, 33, 7, 7, 3, 3, 2), True),      # 49 taps, stride 2
    ((2, 9, 12, 11, 16, 8, 8, 4, 3, 3), False),     # 64 taps, stride 3: nine phases in three launches
    ((1, 96, 5, 4, 40, 1, 7, 0, 3, 2), False),      # filter rows that reach no odd row
    ((4, 64, 23, 29, 192, 3, 3, 0, 0, 2), True),    # whole tiles and a ragged last one, depth in ranges
    ((40, 160, 20, 20, 96, 3, 1, 1, 0, 1), True),   # every range and round of blocks
]


def _bound(values, ranges_and_terms):
    return ranges_and_terms * 2.0 ** -24 * values + 1e-30


@pytest.mark.parametrize("case,sums", CASES)
def test_convolutions_at_the_edges(case, sums, rng, monkeypatch):
    from tsplit_amd import gpu_links as L, ndarray as nd
    monkeypatch.setenv("TSPLIT_CONV_WINOGRAD", "0")
    ctx, (N, C, H, W, Oc, kh, kw, ph, pw, s) = nd.gpu(0), case
    x = rng.normal(size=(N, C, H, W)).astype(np.float32)
    w = rng.normal(size=(Oc, C, kh, kw)).astype(np.float32)
    ref, mag = O.conv2d(x, w, ph, pw, s), O.conv2d(np.abs(x), np.abs(w), ph, pw, s)
    dy = rng.normal(size=ref.shape).astype(np.float32)
    gx, gw, y, dx = nd.array(x, ctx), nd.array(w, ctx), nd.array(np.full(ref.shape, 7, np.float32), ctx), nd.array(np.full(x.shape, 7, np.float32), ctx)
    K = C * kh * kw
    if sums:
        stats = nd.empty((4 * Oc,), ctx)
        L.conv2d_batch_norm_stats(gx, gw, y, stats, 0, ph, pw, s)
        got = stats.asnumpy().view(np.float64).reshape(Oc, 2)
        out = y.asnumpy().astype(np.float64)
        assert (np.abs(got[:, 0] - out.sum((0, 2, 3))) <= _bound(np.abs(out).sum((0, 2, 3)), 65)).all()
        assert (np.abs(got[:, 1] - (out ** 2).sum((0, 2, 3))) <= _bound((out ** 2).sum((0, 2, 3)), 66)).all()
    else:
        L.CuDNN_conv2d(gx, gw, y, ph, pw, s)
    assert (np.abs(y.asnumpy() - ref) <= _bound(mag, K + 32)).all(), case
    L.CuDNN_conv2d_gradient_of_data(gw, nd.array(dy, ctx), dx, ph, pw, s)
    want, size = O.conv2d_grad_data(w, dy, x.shape, ph, pw, s), O.conv2d_grad_data(np.abs(w), np.abs(dy), x.shape, ph, pw, s)
    assert (np.abs(dx.asnumpy() - want) <= _bound(size, Oc * kh * kw + 32)).all(), case


@pytest.mark.parametrize("case", [
    (3, 34, 8, 8, 35, 1, 1, 0, 0, 1),      # words
    (3, 33, 7, 7, 35, 1, 1, 0, 0, 1),      # planes that are not whole words
    (3, 33, 9, 7, 35, 1, 1, 0, 0, 2),
    (3, 17, 9, 10, 19, 3, 3, 1, 1, 1),     # 24 = 17 + 7 padded channels, 24 = 19 + 5
    (3, 17, 9, 10, 19, 3, 3, 1, 1, 2),     # pairs of phases
    (3, 5, 11, 13, 9, 5, 5, 2, 2, 1),      # depth in the filter's order
    (3, 9, 12, 11, 16, 8, 8, 4, 3, 3),     # single phases
])
def test_infinities_stay_in_their_images_and_channels(case, rng, monkeypatch):
    """The channels that pad the depth are the next image's or the next filter's first values: they must not reach a sum, not even
    times zero, in either pass."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    monkeypatch.setenv("TSPLIT_CONV_WINOGRAD", "0")
    ctx, (N, C, H, W, Oc, kh, kw, ph, pw, s) = nd.gpu(0), case
    ys = (N, Oc, (H + 2 * ph - kh) // s + 1, (W + 2 * pw - kw) // s + 1)
    x, w, dy = (rng.normal(size=shape).astype(np.float32) for shape in ((N, C, H, W), (Oc, C, kh, kw), ys))
    x[1] = dy[1] = np.inf
    y, dx = nd.empty(ys, ctx), nd.empty(x.shape, ctx)

    def run():
        L.CuDNN_conv2d(nd.array(x, ctx), nd.array(w, ctx), y, ph, pw, s)
        L.CuDNN_conv2d_gradient_of_data(nd.array(w, ctx), nd.array(dy, ctx), dx, ph, pw, s)
        return np.isfinite(y.asnumpy()), np.isfinite(dx.asnumpy())
    for finite in run():
        assert finite[[0, 2]].all() and not finite[1].all()
    w[3, 4] = np.nan                             # one channel of one filter: the output's channel 3, the gradient's channel 4
    fy, fdx = run()
    assert np.delete(fy, 3, 1)[[0, 2]].all() and not fy[0, 3].any(), "forward"
    assert np.delete(fdx, 4, 1)[[0, 2]].all() and not fdx[0, 4].all(), "data gradient"


def test_channels_past_the_last_beyond_32_bit_offsets(rng):
    """Eight output channels in a tile of 64 rows or more, planes so large that the missing ones lie past 32-bit offsets: nothing
    is stored for them anywhere."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, C, Oc, H = nd.gpu(0), 17, 8, 5400
    x = np.resize(rng.normal(size=1009).astype(np.float32), (1, C, H, H))
    w = rng.normal(size=(Oc, C, 3, 3)).astype(np.float32)
    y = nd.empty((1, Oc, H, H), ctx)
    L.CuDNN_conv2d(nd.array(x, ctx), nd.array(w, ctx), y, 1, 1, 1)
    got = y.asnumpy()
    for row in (0, 1, 2, 2699, 5398, 5399):
        rows = np.zeros((1, C, 3, H), np.float32)
        lo, hi = max(0, row - 1), min(H, row + 2)
        rows[:, :, lo - row + 1:hi - row + 1] = x[:, :, lo:hi]
        ref, mag = O.conv2d(rows, w, 0, 1, 1), O.conv2d(np.abs(rows), np.abs(w), 0, 1, 1)
        assert (np.abs(got[:, :, row:row + 1] - ref) <= _bound(mag, C * 9 + 32)).all(), row


def test_infinities_behind_the_channels_past_the_last(rng):
    """A layer of one tap on large planes, 33 channels in two steps of 32: the offsets of the missing ones leave 32 bits, and folded
    back they would lie inside the image.  Infinities there stay in their own columns."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, C, Oc, H = nd.gpu(0), 33, 8, 3900
    x = np.resize(rng.normal(size=1009).astype(np.float32), (1, C, H, H))
    at = [k * H * H - (1 << 29) for k in range(C, 64) if 0 <= k * H * H - (1 << 29) < x.size]   # 2^31 + 4 k H H - 2^32 bytes
    for a in at:
        x.reshape(-1)[a:a + 4] = np.inf
    y = nd.empty((1, Oc, H, H), ctx)
    L.CuDNN_conv2d(nd.array(x, ctx), nd.array(rng.normal(size=(Oc, C, 1, 1)).astype(np.float32), ctx), y, 0, 0, 1)
    own = np.zeros(H * H, bool)
    for a in at:
        own[np.arange(a, a + 4) % (H * H)] = True
    finite = np.isfinite(y.asnumpy()).reshape(Oc, -1)
    assert len(at) > 9 and finite[:, ~own].all() and not finite[:, own].any()

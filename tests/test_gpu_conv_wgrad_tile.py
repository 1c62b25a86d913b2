"""The filter gradient's tile kernel (csrc/conv_wgrad_tile.h) at the edges of its tiles, of its groups of 16, 4 and 2 channels, of its 16-byte
words and of the images its depth runs over: against float64.

Bar: an output is a sum of K = images x positions fp32 products, in whatever order: within K * 2^-24 of the sum of their
magnitudes (gamma_K to first order), one more 2^-24 for each range's result added by the fold (at most K / 32 of them)."""
import numpy as np
import pytest

from oracle import ops as O

pytestmark = pytest.mark.gpu

CASES = [
    (1, 40, 1, 1, 1, 1, 1, 0, 0, 1),       # one position: a word of four holds one value
    (7, 33, 1, 1, 5, 1, 1, 0, 0, 1),       # several images in a step
    (3, 64, 8, 8, 65, 1, 1, 0, 0, 1),      # one row past a tile; whole words
    (5, 130, 7, 7, 64, 1, 1, 0, 0, 1),     # 49 positions: every image's last word is cut, in both operands
    (2, 47, 6, 5, 129, 1, 1, 0, 0, 1),     # 30 positions, cut by two; channels past the last block
    (2, 36, 9, 7, 130, 1, 1, 0, 0, 2),     # one tap, stride 2
    (3, 40, 8, 8, 20, 1, 1, 1, 1, 1),      # one tap with padding
    (2, 17, 9, 10, 12, 3, 3, 1, 1, 1),     # 32 = 17 + 15 padded channels
    (9, 48, 2, 2, 70, 3, 3, 1, 1, 1),      # images of one word
    (2, 41, 10, 9, 33, 7, 7, 3, 3, 2),     # 49 taps, stride 2
    (2, 9, 12, 11, 16, 8, 8, 4, 3, 3),     # 64 taps, stride 3
    (2, 96, 5, 17, 40, 1, 7, 0, 3, 1),     # a row of taps
    (4, 64, 23, 29, 192, 3, 3, 0, 0, 2),   # whole tiles and a ragged last one
    (40, 160, 20, 20, 96, 3, 1, 1, 0, 1),  # many ranges
    (3, 3, 17, 19, 70, 7, 7, 3, 3, 2),     # groups of 4 channels, one of them padding: four taps a block of 16 columns
    (2, 20, 9, 9, 33, 3, 3, 1, 1, 1),      # groups of 4 without padding; the last block of columns is not full
    (2, 5, 11, 13, 129, 5, 5, 2, 2, 2),    # groups of 2, one channel padding
    (3, 18, 8, 7, 40, 1, 3, 0, 1, 1),      # groups of 2 without padding
    (5, 6, 30, 30, 353, 3, 3, 1, 1, 1),    # groups of 2 on wide tiles
]


def _gradients(case, rng):
    N, C, H, W, Oc, kh, kw, ph, pw, s = case
    x = rng.normal(size=(N, C, H, W)).astype(np.float32)
    dy = rng.normal(size=(N, Oc, (H + 2 * ph - kh) // s + 1, (W + 2 * pw - kw) // s + 1)).astype(np.float32)
    return x, dy, (Oc, C, kh, kw)


def _check(case, x, dy, shape):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (ph, pw, s) = nd.gpu(0), case[7:]
    dw = nd.array(np.full(shape, 7, np.float32), ctx)
    L.CuDNN_conv2d_gradient_of_filter(nd.array(x, ctx), nd.array(dy, ctx), dw, ph, pw, s)
    want, size = O.conv2d_grad_filter(x, dy, shape, ph, pw, s), O.conv2d_grad_filter(np.abs(x), np.abs(dy), shape, ph, pw, s)
    K = dy.size // dy.shape[1]
    assert (np.abs(dw.asnumpy() - want) <= (K + K / 32 + 1) * 2.0 ** -24 * size + 1e-30).all(), case


@pytest.mark.parametrize("case", CASES)
def test_filter_gradients_at_the_edges(case, rng, monkeypatch):
    monkeypatch.setenv("TSPLIT_CONV_WINOGRAD", "0")
    _check(case, *_gradients(case, rng))


def test_ranges_shortened_to_what_a_block_reaches(rng, monkeypatch):
    monkeypatch.setenv("TSPLIT_CONV_WINOGRAD", "0")
    case = (12, 48, 9, 9, 34, 3, 3, 1, 1, 1)
    monkeypatch.setenv("TSPLIT_CONV_REACH_BYTES", str(4 * 4 * (48 + 128) * 81))   # four images
    _check(case, *_gradients(case, rng))


@pytest.mark.parametrize("case", [(3, 40, 7, 7, 20, 1, 1, 0, 0, 1), (3, 40, 7, 7, 20, 3, 3, 1, 1, 1), (3, 12, 7, 7, 20, 3, 3, 1, 1, 1),
                                  (3, 9, 7, 7, 20, 3, 3, 1, 1, 1)])
def test_infinities_stay_in_their_rows(case, rng, monkeypatch):
    """A cut word holds the next channel's first values: they must not reach this channel's sums, not even times zero."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    monkeypatch.setenv("TSPLIT_CONV_WINOGRAD", "0")
    ctx, (ph, pw, s) = nd.gpu(0), case[7:]
    x, dy, shape = _gradients(case, rng)
    dy[:, 11, 0, 0] = np.inf
    x[:, 5, 0, 0] = np.nan
    dw = nd.empty(shape, ctx)
    L.CuDNN_conv2d_gradient_of_filter(nd.array(x, ctx), nd.array(dy, ctx), dw, ph, pw, s)
    finite = np.isfinite(dw.asnumpy()).all((2, 3))
    rest = np.ones(shape[:2], bool)
    rest[11, :] = rest[:, 5] = False
    assert finite[rest].all() and not finite[11, 5]


def test_steps_that_span_more_images_than_a_block_reaches(rng):
    """2 x 2 positions of images of 300 MB: a 32-deep step covers all eight images, 32-bit offsets four of them."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    N, C, H, Oc, s = 8, 300, 512, 16, 256
    x = np.resize(rng.normal(size=1000003).astype(np.float32), (N, C, H, H))
    dy = rng.normal(size=(N, Oc, 2, 2)).astype(np.float32)
    dw = nd.array(np.full((Oc, C, 3, 3), 7, np.float32), nd.gpu(0))
    L.CuDNN_conv2d_gradient_of_filter(nd.array(x, nd.gpu(0)), nd.array(dy, nd.gpu(0)), dw, 1, 1, s)
    got = dw.asnumpy()
    for u in range(3):
        for v in range(3):
            rows, cols = [r for r in range(2) if r * s + u >= 1], [c for c in range(2) if c * s + v >= 1]
            a = dy[:, :, rows][:, :, :, cols].transpose(1, 0, 2, 3).reshape(Oc, -1).astype(np.float64)
            b = np.stack([x[:, :, r * s - 1 + u, c * s - 1 + v] for r in rows for c in cols], 2).transpose(0, 2, 1).reshape(-1, C).astype(np.float64)
            assert (np.abs(got[:, :, u, v] - a @ b) <= 36 * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + 1e-30).all(), (u, v)

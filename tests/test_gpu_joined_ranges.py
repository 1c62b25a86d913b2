"""Ranges of the depth added up by the launch that computes them: every count of ranges the planner takes on the four tiles, whole and
part tiles, the same bits at every call (the counts of the tiles are 0 again behind each), on two streams at once and in a recorded step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# m, n, k: two ranges and more, one tile and many, rows and columns past the last tile
PRODUCTS = [(64, 64, 2048), (65, 67, 1031), (200, 130, 3000), (100, 4096, 4096), (1000, 500, 2050), (128, 1000, 2048), (512, 512, 4096), (700, 900, 777),
            (1500, 1200, 1600), (10, 10, 8192), (384, 2048, 512)]
# n, c, h, w, o, kernel, pad, stride
LAYERS = [(5, 96, 35, 33, 200, 3, 0, 2), (5, 96, 35, 33, 200, 3, 0, 1), (8, 512, 4, 4, 512, 3, 1, 1), (3, 300, 7, 7, 130, 1, 0, 1), (2, 700, 9, 9, 70, 1, 0, 2),
          (4, 256, 17, 17, 192, 5, 2, 1), (1, 1024, 14, 14, 300, 1, 0, 1)]


def _close(got, want, depth, scale):
    """Sums of `depth` products of normal values: rounding errors of a chain within 8 of their walk."""
    assert np.abs(got - want).max() <= 8 * 2.0 ** -24 * np.sqrt(depth) * scale * 6, np.abs(got - want).max()


@pytest.mark.parametrize("m,n,k", PRODUCTS)
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_products(m, n, k, ta, tb):
    from tsplit_amd import gpu_links as L, ndarray as nd
    from tsplit_amd.stream import create_stream_handle
    rng, ctx = np.random.default_rng(m + n + k), nd.gpu(0)
    a, b, bias, more = (rng.standard_normal(s, dtype=np.float32) for s in ((m, k), (k, n), (n,), (m, n)))
    ga, gb, gbias, gmore = (nd.array(np.ascontiguousarray(v), ctx) for v in (a.T if ta else a, b.T if tb else b, bias, more))
    want = a.astype(np.float64) @ b.astype(np.float64)
    streams = [None, create_stream_handle(ctx)]
    outs = [[nd.empty((m, n), ctx) for _ in range(6)] for _ in streams]
    fused = [nd.empty((m, n), ctx) for _ in streams]
    relus = [nd.empty((m, n), ctx) for _ in streams]
    nd.empty((1,), ctx).asnumpy()
    for i in range(6):
        for s, o in zip(streams, outs):
            L.matrix_multiply(ga, ta, gb, tb, o[i], s)
    for s, o, r in zip(streams, fused, relus):
        L.matrix_multiply_add(ga, ta, gb, tb, o, gbias, gmore, r, s)
    streams[1].sync()
    first = outs[0][0].asnumpy()
    _close(first, want, k, np.sqrt(k) / 4 + 1)
    for o in outs[0] + outs[1]:
        np.testing.assert_array_equal(o.asnumpy(), first)
    whole = (first + bias) + more
    for o, r in zip(fused, relus):
        np.testing.assert_array_equal(o.asnumpy(), whole)
        np.testing.assert_array_equal(r.asnumpy(), np.maximum(whole, 0))


@pytest.mark.parametrize("n,c,h,w,o,k,pad,s", LAYERS)
def test_convolutions(n, c, h, w, o, k, pad, s):
    import torch
    from tsplit_amd import gpu_links as L, ndarray as nd
    rng, ctx = np.random.default_rng(n + c + h + o + k), nd.gpu(0)
    oh, ow = (h + 2 * pad - k) // s + 1, (w + 2 * pad - k) // s + 1
    x, f, g = (rng.standard_normal(v, dtype=np.float32) for v in ((n, c, h, w), (o, c, k, k), (n, o, oh, ow)))
    xt, ft = (torch.from_numpy(v).double().requires_grad_() for v in (x, f))
    y = torch.nn.functional.conv2d(xt, ft, stride=s, padding=pad)
    y.backward(torch.from_numpy(g).double())
    gx, gf, gg = (nd.array(v, ctx) for v in (x, f, g))
    got = []
    for _ in range(5):
        out, dx, dw = nd.array(np.full(g.shape, 7, np.float32), ctx), nd.array(np.full(x.shape, 7, np.float32), ctx), nd.array(np.full(f.shape, 7, np.float32), ctx)
        L.CuDNN_conv2d(gx, gf, out, pad, pad, s)
        L.CuDNN_conv2d_gradient_of_data(gf, gg, dx, pad, pad, s)
        L.CuDNN_conv2d_gradient_of_filter(gx, gg, dw, pad, pad, s)
        got.append([v.asnumpy() for v in (out, dx, dw)])
    for v, want, depth in zip(got[0], (y.detach(), xt.grad, ft.grad), (c * k * k, o * k * k, n * oh * ow)):
        _close(v, want.numpy(), depth, np.sqrt(depth) / 4 + 1)
    for later in got[1:]:
        for v, w0 in zip(later, got[0]):
            np.testing.assert_array_equal(v, w0)

"""Convolutions of several taps whose depth is one, two, three and more steps of 32, whole and cut, in one range and many: the first and the last step
of a range are forms of their own.  Each pass within rounding of float64, and with the same bits every time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# n, c, h, w, o, kernel (rows, columns), pad (rows, columns), stride: none that the Winograd routine takes, whose errors are others (3x3 with padding,
# from 16 K positions on)
LAYERS = [(1, 8, 4, 9, 16, (1, 2), (0, 0), 1), (1, 8, 4, 8, 8, (1, 3), (0, 1), 1), (2, 8, 4, 4, 24, (5, 1), (2, 0), 1), (1, 8, 8, 12, 130, (1, 7), (0, 3), 1),
          (2, 24, 9, 9, 40, (3, 3), (1, 1), 1), (1, 7, 3, 3, 9, (3, 3), (1, 1), 1), (3, 33, 7, 9, 70, (3, 3), (0, 0), 2), (5, 96, 35, 33, 200, (3, 3), (0, 0), 2),
          (8, 512, 4, 4, 512, (3, 3), (1, 1), 1), (4, 256, 17, 17, 192, (5, 5), (2, 2), 1), (2, 64, 21, 20, 64, (7, 7), (3, 3), 1), (32, 128, 17, 17, 256, (7, 1), (3, 0), 1),
          (18, 64, 35, 35, 96, (3, 3), (0, 0), 1), (2, 6, 11, 10, 20, (3, 3), (1, 1), 2), (1, 16, 5, 5, 300, (4, 4), (3, 3), 2)]


@pytest.mark.parametrize("n,c,h,w,o,k,pad,s", LAYERS)
def test_all_three_passes(n, c, h, w, o, k, pad, s):
    import torch
    from tsplit_amd import gpu_links as L, ndarray as nd
    rng, ctx = np.random.default_rng(n + c + h + o + k[0]), nd.gpu(0)
    oh, ow = (h + 2 * pad[0] - k[0]) // s + 1, (w + 2 * pad[1] - k[1]) // s + 1
    x, f, g = (rng.standard_normal(v, dtype=np.float32) for v in ((n, c, h, w), (o, c) + k, (n, o, oh, ow)))

    def passes(x, f, g):
        xt, ft = (torch.from_numpy(v).double().requires_grad_() for v in (x, f))
        y = torch.nn.functional.conv2d(xt, ft, stride=s, padding=pad)
        y.backward(torch.from_numpy(g).double())
        return y.detach().numpy(), xt.grad.numpy(), ft.grad.numpy()
    wants, sizes, depths = passes(x, f, g), passes(abs(x), abs(f), abs(g)), (c * k[0] * k[1], o * k[0] * k[1], n * oh * ow)
    gx, gf, gg = (nd.array(v, ctx) for v in (x, f, g))
    first = None
    for _ in range(3):
        out, dx, dw = (nd.array(np.full(v.shape, 7, np.float32), ctx) for v in (g, x, f))
        L.CuDNN_conv2d(gx, gf, out, pad[0], pad[1], s)
        L.CuDNN_conv2d_gradient_of_data(gf, gg, dx, pad[0], pad[1], s)
        L.CuDNN_conv2d_gradient_of_filter(gx, gg, dw, pad[0], pad[1], s)
        got = [v.asnumpy() for v in (out, dx, dw)]
        first = first or got
        for v, again in zip(got, first):
            np.testing.assert_array_equal(v, again)
    # a chain of `depth` roundings walks sqrt(depth) of them, as a share of the sum of the products' magnitudes
    for v, want, size, depth in zip(first, wants, sizes, depths):
        assert (np.abs(v - want) <= 2.0 ** -24 * (8 + np.sqrt(depth)) * size + 1e-30).all()

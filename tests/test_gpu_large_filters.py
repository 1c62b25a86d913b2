"""Layers whose filters are re-laid, and whose filter gradients are folded, in tiles through LDS (from a million values on): channels that
fill no tile on either side, filters of one row, planes of a few positions.  Bound: a result is a sum of m products, rounded m times at
most on any path through its ranges; random signs leave about the square root, so m 2^-24 of the root mean square of its terms times
sqrt(m) is held with room: 4 sqrt(m) 2^-24 of the largest magnitude of the plane."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (ranges: into how many the depth of the filter gradient is cut, which the fold adds up in fours)
@pytest.mark.parametrize("n,c,h,w,o,kh,kw,ph,pw,s,ranges", [(2, 500, 4, 3, 261, 3, 3, 1, 1, 1, 1), (1, 520, 5, 4, 700, 1, 3, 0, 1, 1, 1),
                                                            (3, 263, 6, 7, 170, 5, 5, 2, 2, 2, 1), (2, 513, 3, 3, 259, 3, 3, 0, 0, 1, 1),
                                                            (64, 500, 4, 4, 261, 3, 3, 1, 1, 1, 2), (33, 263, 9, 7, 170, 5, 5, 2, 2, 2, 3),
                                                            (64, 512, 4, 4, 512, 3, 3, 1, 1, 1, 4), (16, 500, 8, 8, 700, 1, 3, 0, 1, 1, 5)])
def test_large_filters(n, c, h, w, o, kh, kw, ph, pw, s, ranges, rng):
    from tsplit_amd import gpu_links as L, ndarray as nd, profiler
    ctx = nd.gpu(0)
    oh, ow = (h + 2 * ph - kh) // s + 1, (w + 2 * pw - kw) // s + 1
    assert c * o * kh * kw >= 1 << 20
    x, f, g = [rng.normal(size=sh).astype(np.float32) for sh in ((n, c, h, w), (o, c, kh, kw), (n, o, oh, ow))]
    gx, gf, gg = [nd.array(a, ctx) for a in (x, f, g)]
    y, dx, dw = nd.empty(g.shape, ctx), nd.empty(x.shape, ctx), nd.empty(f.shape, ctx)
    L.CuDNN_conv2d(gx, gf, y, ph, pw, s)
    L.CuDNN_conv2d_gradient_of_data(gf, gg, dx, ph, pw, s)
    p = profiler.CreateProfiler()
    L.CuDNN_conv2d_gradient_of_filter(gx, gg, dw, ph, pw, s, None, p)
    assert abs(p.workspace_memory * 2 ** 18 / f.size - ranges) < 1e-3
    # the sums in float64: patches of the padded input, [n, oh * ow, c * kh * kw]
    xp = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (ph, ph), (pw, pw)))
    patches = np.stack([xp[:, :, u:u + s * (oh - 1) + 1:s, v:v + s * (ow - 1) + 1:s] for u in range(kh) for v in range(kw)], axis=2)
    patches = patches.reshape(n, c * kh * kw, oh * ow)
    f2, g2 = f.astype(np.float64).reshape(o, -1), g.astype(np.float64).reshape(n, o, oh * ow)
    want_dw = np.einsum("nop,nkp->ok", g2, patches).reshape(f.shape)
    back = np.einsum("ok,nop->nkp", f2, g2).reshape(n, c, kh, kw, oh, ow)
    want_dx = np.zeros(xp.shape)
    for u in range(kh):
        for v in range(kw):
            want_dx[:, :, u:u + s * (oh - 1) + 1:s, v:v + s * (ow - 1) + 1:s] += back[:, :, u, v]
    want_dx = want_dx[:, :, ph:ph + h, pw:pw + w]
    for got, want, m in ((y, np.einsum("ok,nkp->nop", f2, patches).reshape(g.shape), c * kh * kw), (dx, want_dx, o * kh * kw), (dw, want_dw, n * oh * ow)):
        assert np.abs(got.asnumpy() - want).max() <= 4 * np.sqrt(m) * 2.0 ** -24 * np.abs(want).max()

"""Products, convolutions and filter gradients at ragged sizes and for values that have no split into three bf16 numbers - infinities, NaN, numbers
above bf16's largest and numbers so small that bf16 does not hold their parts: with the split-bf16 switch off, as here, the fp32 instruction
multiplies them like any other.

Bar for ordinary values: within (K + 64) 2^-24 of the sum of the products' magnitudes; and, as the mean over many results,
no further from 64 bits than fp32 sums in any order usually are (2^-24 sqrt(K) of the root of the squares' sum)."""
import numpy as np
import pytest

from oracle import ops as O

pytestmark = pytest.mark.gpu

# M, N, K: rows or columns the fewer, ragged in every direction, depths that a step cuts
SHAPES = [(2048, 512, 512), (515, 2047, 1031), (2050, 516, 1001), (100, 4096, 4096), (4096, 100, 4093), (4099, 257, 130), (4098, 4100, 65)]


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("shape", SHAPES)
def test_products(shape, ta, tb, rng):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K) = nd.gpu(0), shape
    a = rng.normal(size=(K, M) if ta else (M, K)).astype(np.float32)
    b = rng.normal(size=(N, K) if tb else (K, N)).astype(np.float32)
    a64, b64 = (a.T if ta else a).astype(np.float64), (b.T if tb else b).astype(np.float64)
    c = nd.array(np.full((M, N), 7, np.float32), ctx)
    L.matrix_multiply(nd.array(a, ctx), ta, nd.array(b, ctx), tb, c)
    off = np.abs(c.asnumpy() - a64 @ b64)
    assert (off <= (K + 64) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))).all()
    assert np.sqrt(np.mean(off ** 2)) <= 2.0 ** -24 * K      # sqrt(K) for the sum's length, sqrt(K) for the results' size


FLT_MAX = np.float32(3.4028235e38)


def _special(a, rng, kind, where):
    """Plants values of a kind into every 9973rd element or, "rows", makes some whole rows of them."""
    at = np.zeros(a.shape, bool)
    if where == "rows":
        at[::37] = True
    else:
        at.reshape(-1)[5::9973] = True
    v = {"inf": np.float32(np.inf), "nan": np.float32(np.nan), "huge": FLT_MAX * np.float32(0.9999)}.get(kind)
    if v is not None:
        a[at] = v * np.where(rng.random_sample(int(at.sum())) < 0.5, np.float32(-1), np.float32(1))
    elif kind == "small":
        a[at] *= np.float32(1e-36)
    else:   # subnormal
        a[at] = (a[at] * np.float32(1e-30)) * np.float32(1e-11)
    return a


def _compare(got, want, tol):
    """Infinities and NaN where 64 bits have them, everything else to `tol` of the sum of its products' magnitudes."""
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    np.testing.assert_array_equal(got[inf], want[inf].astype(np.float32))
    ok = np.isfinite(want)
    assert (np.abs(got[ok] - want[ok]) <= tol[ok]).all()


@pytest.mark.parametrize("prepared", [True, False])
@pytest.mark.parametrize("kind,where", [("inf", "some"), ("nan", "some"), ("huge", "some"), ("small", "rows"), ("subnormal", "rows")])
def test_products_of_values_without_a_split(kind, where, prepared, rng):
    """In the operand with fewer rows (`prepared`) and in the other one."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K) = nd.gpu(0), (500, 2048, 520)
    a, b = rng.normal(size=(M, K)).astype(np.float32), rng.normal(size=(N, K)).astype(np.float32)
    if kind == "huge":
        a, b = a * np.float32(1e-3), b * np.float32(1e-3)
    if kind in ("small", "subnormal"):   # against values that bring the results back into range
        (b if prepared else a)[:] *= np.float32(1e20)
    _special(a if prepared else b, rng, kind, where)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    with np.errstate(invalid="ignore", over="ignore"):
        want, size = a64 @ b64.T, np.abs(a64) @ np.abs(b64.T)
    c = nd.empty((M, N), ctx)
    L.matrix_multiply(nd.array(a, ctx), False, nd.array(b, ctx), True, c)
    _compare(c.asnumpy(), want, (K + 64) * 2.0 ** -24 * size + 1e-37)


# N, C, H, W, O, kh, kw, ph, pw, s: blocks of channels and the filter's own order, 1 x 1, stride 2 in pairs of phases, few channels
LAYERS = [(3, 40, 13, 11, 72, 3, 3, 1, 1, 1), (4, 3, 21, 19, 33, 5, 5, 2, 2, 1), (2, 24, 17, 15, 130, 3, 3, 0, 0, 2), (16, 512, 28, 28, 128, 1, 1, 0, 0, 1),
          (3, 40, 20, 21, 48, 1, 7, 0, 3, 1), (6, 10, 50, 50, 375, 5, 5, 2, 2, 1)]   # the second and the last: few channels


@pytest.mark.parametrize("kind,where", [("inf", "some"), ("nan", "some"), ("huge", "some"), ("small", "rows"), ("subnormal", "rows")])
@pytest.mark.parametrize("layer", LAYERS)
def test_convolutions_of_values_without_a_split(layer, kind, where, rng, monkeypatch):
    """All three passes, the values once in the first operand and once in the second."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    monkeypatch.setenv("TSPLIT_CONV_WINOGRAD", "0")
    ctx, (n, c, h, w, o, kh, kw, ph, pw, s) = nd.gpu(0), layer
    oh, ow = (h + 2 * ph - kh) // s + 1, (w + 2 * pw - kw) // s + 1
    scale = np.float32(1e-3 if kind == "huge" else 1e20 if kind in ("small", "subnormal") else 1)
    draw = lambda *shape: rng.normal(size=shape).astype(np.float32)   # noqa: E731
    passes = [
        ("forward", (n, c, h, w), (o, c, kh, kw), (n, o, oh, ow), lambda x, f: O.conv2d(x, f, ph, pw, s), lambda x, f, y: L.CuDNN_conv2d(x, f, y, ph, pw, s)),
        ("data gradient", (n, o, oh, ow), (o, c, kh, kw), (n, c, h, w), lambda dy, f: O.conv2d_grad_data(f, dy, (n, c, h, w), ph, pw, s),
         lambda dy, f, dx: L.CuDNN_conv2d_gradient_of_data(f, dy, dx, ph, pw, s)),
        ("filter gradient", (n, c, h, w), (n, o, oh, ow), (o, c, kh, kw), lambda x, dy: O.conv2d_grad_filter(x, dy, (o, c, kh, kw), ph, pw, s),
         lambda x, dy, dw: L.CuDNN_conv2d_gradient_of_filter(x, dy, dw, ph, pw, s)),
    ]
    for name, sa, sb, so, ref, run in passes:
        for first in (True, False):
            a, b = draw(*sa), draw(*sb)
            if kind == "huge":
                a, b = a * scale, b * scale
            elif kind in ("small", "subnormal"):
                (b if first else a)[:] *= scale
            _special(a if first else b, rng, kind, where)
            depth = np.prod(sb[1:]) if name == "forward" else o * kh * kw if name == "data gradient" else n * oh * ow
            out = nd.empty(so, ctx)
            run(nd.array(a, ctx), nd.array(b, ctx), out)
            got = out.asnumpy()
            finite = lambda v: np.where(np.isfinite(v), v, 0)   # noqa: E731
            size = ref(np.abs(finite(a)), np.abs(finite(b)))
            if kind in ("inf", "nan"):
                # which results an infinity or NaN reaches, from the same convolution of where they are; one that meets the padding
                # makes NaN of its product with that zero or not
                bad_a, bad_b = (~np.isfinite(a)).astype(np.float32), (~np.isfinite(b)).astype(np.float32)
                touched = ref(bad_a, np.ones_like(b)) + ref(np.ones_like(a), bad_b) > 0.5
                assert not np.isfinite(got[touched]).any(), (name, first)
                ok = ~touched
                if not first:   # every result of a row of the filter, or of dy's channel, that holds one
                    rows = bad_b.any(axis=(0, 2, 3)) if name != "forward" else bad_b.any(axis=(1, 2, 3))
                    ok &= ~(rows[None, :, None, None] if name != "filter gradient" else rows[:, None, None, None])
            else:
                ok = np.ones(so, bool)
            want = ref(finite(a), finite(b))
            assert (np.abs(got[ok] - want[ok]) <= (depth + 64) * 2.0 ** -24 * size[ok] + 1e-37).all(), (name, first, kind)


@pytest.mark.parametrize("scales", [(1.0, 1.0), (1e-36, 1e20), (1e20, 1e-36), (1e-41, 1e30), (1e35, 1e-3)])
@pytest.mark.parametrize("layer", [(2, 144, 14, 18, 200), (3, 272, 7, 9, 130)])
def test_winograd_gemms_hold_every_scale(layer, scales, rng, monkeypatch):
    """Forward and filter gradient of layers with more than 64 channels on both sides (their data gradients, whose summed channels are no
    multiple of 16, take the direct kernels), with operands that have no split."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    monkeypatch.setenv("TSPLIT_CONV_WINOGRAD", "1")
    ctx, (n, c, h, w, o) = nd.gpu(0), layer
    x, f, dy = [rng.normal(size=s) for s in ((n, c, h, w), (o, c, 3, 3), (n, o, h, w))]
    x32, f32, dy32 = (x * scales[0]).astype(np.float32), (f * scales[1]).astype(np.float32), (dy * scales[1]).astype(np.float32)
    y, dx, dw = nd.empty((n, o, h, w), ctx), nd.empty((n, c, h, w), ctx), nd.empty((o, c, 3, 3), ctx)
    L.CuDNN_conv2d(nd.array(x32, ctx), nd.array(f32, ctx), y, 1, 1, 1)
    L.CuDNN_conv2d_gradient_of_filter(nd.array(x32, ctx), nd.array(dy32, ctx), dw, 1, 1, 1)
    L.CuDNN_conv2d_gradient_of_data(nd.array(f32, ctx), nd.array((dy * scales[0]).astype(np.float32), ctx), dx, 1, 1, 1)
    size = scales[0] * scales[1]
    # the transforms' own share is 2e-5; subnormal operands come with fewer bits of their own
    tol = 1e-4 if min(scales) > 1e-38 else 1e-2
    for got, want in ((y, O.conv2d(x32, f32, 1, 1, 1)), (dw, O.conv2d_grad_filter(x32, dy32, f.shape, 1, 1, 1)),
                      (dx, O.conv2d_grad_data(f32, (dy * scales[0]).astype(np.float32), x.shape, 1, 1, 1))):
        want = want / size
        assert np.abs(got.asnumpy().astype(np.float64) / size - want).max() <= tol * np.abs(want).max()

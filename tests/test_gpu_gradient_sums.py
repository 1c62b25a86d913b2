"""A data gradient added to what is there in the launch that makes it: the bits of the gradient and the sum by themselves."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# n, c, h, w, o, kernel, pad, stride: whole words and single values, ranges of the depth, part tiles, both rows of a strided plane
# with and without a last one of its own, and the forms that stay two launches
SHAPES = [(2, 64, 28, 28, 96, 1, 0, 1), (3, 70, 17, 17, 130, 1, 0, 1), (1, 33, 5, 7, 1500, 1, 0, 1), (1, 32, 8, 8, 2048, 1, 0, 1), (20, 256, 28, 28, 64, 1, 0, 1),
          (2, 1, 1, 1, 1, 1, 0, 1), (2, 64, 28, 28, 128, 1, 0, 2), (3, 40, 15, 13, 70, 1, 0, 2), (2, 24, 14, 9, 1300, 1, 0, 2), (2, 20, 9, 10, 24, 1, 0, 3),
          (2, 24, 12, 11, 40, 1, 1, 1), (2, 64, 16, 16, 64, 3, 1, 1), (2, 24, 13, 12, 30, 3, 0, 2), (0, 8, 4, 4, 8, 1, 0, 1)]


@pytest.mark.parametrize("n,c,h,w,o,k,pad,s", SHAPES)
def test_bits_of_the_two_calls(n, c, h, w, o, k, pad, s):
    from tsplit_amd import gpu_links as L, ndarray as nd
    rng, ctx = np.random.default_rng(n + c + h + o + k + s), nd.gpu(0)
    oh, ow = (h + 2 * pad - k) // s + 1, (w + 2 * pad - k) // s + 1
    f = nd.array(rng.standard_normal((o, c, k, k), dtype=np.float32), ctx)
    dy = nd.array(rng.standard_normal((n, o, oh, ow), dtype=np.float32), ctx)
    a = rng.standard_normal((n, c, h, w), dtype=np.float32)
    a.reshape(-1)[::97] = np.inf
    alone, whole, apart, there = (nd.empty((n, c, h, w), ctx) for _ in range(4))
    addend = nd.array(a, ctx)
    L.CuDNN_conv2d_gradient_of_data(f, dy, alone, pad, pad, s)
    L.matrix_elementwise_add(addend, alone, whole)
    L.conv2d_gradient_of_data_add(f, dy, addend, apart, pad, pad, s)
    nd.array(a, ctx).copyto(there)
    L.conv2d_gradient_of_data_add(f, dy, there, there, pad, pad, s)
    np.testing.assert_array_equal(apart.asnumpy(), whole.asnumpy())
    np.testing.assert_array_equal(there.asnumpy(), whole.asnumpy())
    np.testing.assert_array_equal(addend.asnumpy(), a)


def test_an_addend_of_another_size_is_refused():
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx = nd.gpu(0)
    with pytest.raises(RuntimeError):
        L.conv2d_gradient_of_data_add(nd.empty((8, 4, 1, 1), ctx), nd.empty((2, 8, 4, 4), ctx), nd.empty((2, 4, 4, 3), ctx), nd.empty((2, 4, 4, 4), ctx))


@pytest.mark.parametrize("stride,hw", [(1, 9), (2, 8)])
def test_branches_of_a_tape(stride, hw):
    """Three readers of one value, whose gradient begins as a shared array: as a tape that adds one by one has it."""
    from tsplit_amd import graph, ndarray as nd
    rng = np.random.default_rng(hw)
    x, u, v = (rng.standard_normal(s, dtype=np.float32) for s in ((3, 12, hw, hw), (12, 12, 1, 1), (20, 12, 1, 1)))

    def gradients(fused):
        b = graph.GpuBackend(nd.gpu(0))
        t = graph.Tape(b)
        t._adds_data_gradient = t._adds_data_gradient if fused else lambda *a: False
        p = [t.param(b.from_numpy(a), a.shape) for a in (x, u, v)]
        h = t.relu(p[0])
        y = t.relu(t.conv2d(h, p[2], 0, 0, stride))
        z = t.add(t.relu(t.add(t.conv2d(h, p[1], 0, 0, 1), h)), h)
        flat = t.matmul(t.reshape(z, (3, -1)), t.const(b.from_numpy(np.ones((z.shape[1] * hw * hw, 4), np.float32)), (z.shape[1] * hw * hw, 4)))
        other = t.matmul(t.reshape(y, (3, -1)), t.const(b.from_numpy(np.ones((int(np.prod(y.shape[1:])), 4), np.float32)), (int(np.prod(y.shape[1:])), 4)))
        loss = t.softmax_ce(t.add(flat, other), t.const(b.from_numpy(np.eye(4, dtype=np.float32)[:3]), (3, 4)))
        t.backward(loss)
        return [q.grad.asnumpy() for q in p]
    for one, two in zip(gradients(True), gradients(False)):
        np.testing.assert_array_equal(one, two)


# positions that no tap reaches, in whole words and value by value, with the depth in one range and in several
@pytest.mark.parametrize("n,c,h,w,o,s", [(2, 64, 28, 28, 32, 2), (3, 40, 15, 13, 30, 2), (2, 24, 14, 9, 32, 2), (2, 64, 28, 28, 128, 2), (2, 24, 14, 9, 1300, 2),
                                         (2, 64, 28, 28, 32, 1), (1, 33, 5, 7, 1500, 1)])
def test_zeros_have_the_sign_that_the_two_calls_give_them(n, c, h, w, o, s):
    from tsplit_amd import gpu_links as L, ndarray as nd
    rng, ctx = np.random.default_rng(n + c + h + o + s), nd.gpu(0)
    f, dy = rng.standard_normal((o, c, 1, 1), dtype=np.float32), rng.standard_normal((n, o, (h - 1) // s + 1, (w - 1) // s + 1), dtype=np.float32)
    f[:, ::3], dy[0] = 0, 0
    a = np.where(rng.random((n, c, h, w)) < 0.5, np.float32(-0.0), np.float32(0.0))
    f, dy, addend = (nd.array(v, ctx) for v in (f, dy, a))
    alone, whole, apart = (nd.empty((n, c, h, w), ctx) for _ in range(3))
    L.CuDNN_conv2d_gradient_of_data(f, dy, alone, 0, 0, s)
    L.matrix_elementwise_add(addend, alone, whole)
    L.conv2d_gradient_of_data_add(f, dy, addend, apart, 0, 0, s)
    L.conv2d_gradient_of_data_add(f, dy, addend, addend, 0, 0, s)
    for got in (apart, addend):
        np.testing.assert_array_equal(got.asnumpy().view(np.uint32), whole.asnumpy().view(np.uint32))


# images in runs of 3, 3 and 1, of 2, and one by one; not even one in reach: two calls
@pytest.mark.parametrize("reach", [160_000, 110_000, 60_000, 20_000])
@pytest.mark.parametrize("s", [1, 2])
def test_runs_of_images(s, reach, monkeypatch):
    from tsplit_amd import gpu_links as L, ndarray as nd
    rng, ctx, (n, c, h, o) = np.random.default_rng(s), nd.gpu(0), (7, 16, 20 * s, 32)
    f, dy, a = (nd.array(rng.standard_normal(v, dtype=np.float32), ctx) for v in ((o, c, 1, 1), (n, o, 20, 20), (n, c, h, h)))
    alone, whole, apart = (nd.empty((n, c, h, h), ctx) for _ in range(3))
    monkeypatch.setenv("TSPLIT_CONV_REACH_BYTES", str(reach))
    L.CuDNN_conv2d_gradient_of_data(f, dy, alone, 0, 0, s)
    L.matrix_elementwise_add(a, alone, whole)
    L.conv2d_gradient_of_data_add(f, dy, a, apart, 0, 0, s)
    L.conv2d_gradient_of_data_add(f, dy, a, a, 0, 0, s)
    for got in (apart, a):
        np.testing.assert_array_equal(got.asnumpy(), whole.asnumpy())

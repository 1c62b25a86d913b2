"""BatchNorm over planes that are not of whole 16-byte words: the kernels in the order of memory give the bits of the kernels that
take an array off 16 bytes value by value."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# more than 16384 values a channel; odd planes of one to many words, one channel, arrays that end inside a word, planes of three
SHAPES = [(101, 3, 13, 13), (3301, 3, 5, 1), (2801, 3, 3, 2), (17001, 1, 7, 1), (1, 1, 129, 129), (1, 5, 131, 129), (5501, 5, 3, 1), (15, 33, 35, 35)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("form", ["alone", "saved", "exact", "fused", "both"])
def test_bits_on_and_off_16_bytes(shape, form, rng):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (n, c, h, w) = nd.gpu(0), shape
    x, dy = (rng.normal(size=shape).astype(np.float32) for _ in range(2))
    x.reshape(-1)[-1], x.reshape(-1)[h * w % x.size] = 3e4, -3e4
    gamma, beta = (nd.array(rng.normal(size=(1, c, 1, 1)).astype(np.float32), ctx) for _ in range(2))

    def both_ways(off):
        def like(v=None):
            """An array of the shape that begins on 16 bytes, or off them."""
            whole = nd.array(np.full((2 * n, c, h, w), 7, np.float32), ctx)
            a = nd.slice_for_micro_tensor(whole, 1 if off else 0, 2)
            assert bool(a.data_ptr % 16) == off
            if v is not None:
                nd.array(v, ctx).copyto(a)
            return a
        gx, gdy, y, r, dx, dg = like(x), like(dy), like(), like(), like(), like()
        a, b, pair = (nd.array(np.zeros((c, 2) if form == "exact" or i == 2 else (1, c, 1, 1), np.float32), ctx) for i in range(3))
        da, db = (nd.empty((1, c, 1, 1), ctx) for _ in range(2))
        if form in ("alone", "saved"):
            saved = (a, b) if form == "saved" else (None, None)
            L.CuDNN_Batch_Normalization(gx, gamma, beta, y, *saved, 0.99, 0.01)
            L.CuDNN_Batch_Normalization_gradient(gdy, gx, gamma, dx, da, db, *saved, 0.01)
        elif form == "both":
            L.batch_norm_then_relu(gx, gamma, beta, y, r, pair)
            L.batch_norm_then_relu_gradient(gdy, gx, gamma, pair, dg, dx, da, db)
        else:
            L.batch_norm_relu(gx, gamma, beta, y, a, b, 0.01)
            L.batch_norm_relu_gradient(gdy, gx, gamma, beta, dx, da, db, a, b, 0.01)
        return [v.asnumpy() for v in (y, r, dx, dg, da, db)]
    for one, other in zip(both_ways(False), both_ways(True)):
        np.testing.assert_array_equal(one, other)

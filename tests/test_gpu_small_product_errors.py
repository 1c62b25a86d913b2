"""Small products (csrc/gemm_waves.h) have the bits of the tile kernel and its fold, and are no further from float64 than its order of adding is:
fused multiply-adds in fp32 along each of its ranges of the depth, the ranges' results added one by one.  That order is followed here value by
value on the host.

Bar of the latter: 1.15 times its rms error.  The matrix instruction may add the four products of a step in another order, which moves a single value's
error and not the rms of thousands; a chain twice as long has 1.4 times the error."""
import numpy as np
import pytest

from product_plan import plan


def _chain(a, b):
    """The running fp32 sums of a[..., k] * b[..., k] along k, a fused multiply-add each (the product is exact in float64)."""
    s = np.zeros(np.broadcast_shapes(a.shape[:-1], b.shape[:-1]), np.float32)
    for k in range(a.shape[-1]):
        s = (s.astype(np.float64) + a[..., k].astype(np.float64) * b[..., k]).astype(np.float32)
    return s


def _in_ranges(a, b, step):
    s = None
    for k in range(0, a.shape[1], step):
        part = _chain(a[:, None, k:k + step], b.T[None, :, k:k + step])
        s = part if s is None else s + part
    return s


def _rms(v):
    return float(np.sqrt(np.mean(v * v)))


# linear layers of the networks that train here: forward, and the gradients whose depth is the batch or the classes
SHAPES = [(128, 256, 784), (128, 256, 256), (64, 512, 512), (385, 256, 1024), (32, 1000, 1536), (64, 1000, 2048), (96, 130, 1100),
          (33, 65, 159), (60, 900, 1800), (256, 256, 128), (197, 1189, 271)]


def test_ranges_are_the_tile_kernels_and_of_batches_shorter():
    rng = np.random.RandomState(5)
    drawn = [tuple(int(round(np.exp(rng.uniform(0, np.log(top))))) for top in (2048, 5003, 5003, 64)) for _ in range(3000)]
    seen = 0
    for M, N, K, batch in [s + (1,) for s in SHAPES] + drawn:
        p = plan(M, N, K, batch)
        if p.waves:
            seen += 1
            assert p.range == p.tile_range if batch == 1 else p.range <= p.tile_range and -(-K // p.range) <= 4, (M, N, K, batch, p)
            lds = -(-K // p.range) * (p.tile[0] + 1) * p.tile[1] * 4
            assert p.range % 32 == 0 and 2 <= p.waves <= 4 and lds <= 80 * 1024, (M, N, K, batch, p)
    assert seen > 500


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("shape", SHAPES)
def test_bits_of_the_tile_kernel_and_its_fold(shape, ta, tb):
    """The tile kernel makes each range's product by itself where the rows are the first of many."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K), rng = nd.gpu(0), shape, np.random.RandomState(4)
    p = plan(M, N, K)
    assert p.waves
    rows = next(m for m in (4096, 16384) if m > M and not plan(m, N, p.range).waves and plan(m, N, p.range).range >= min(K, p.range))
    a, b = rng.normal(size=(M, K)).astype(np.float32), rng.normal(size=(K, N)).astype(np.float32)

    def product(x, y):
        c = nd.empty((x.shape[0], N), ctx)
        x, y = (np.ascontiguousarray(v.T) if t else np.ascontiguousarray(v) for v, t in ((x, ta), (y, tb)))
        L.matrix_multiply(nd.array(x, ctx), ta, nd.array(y, ctx), tb, c)
        return c.asnumpy()
    want = None
    for k in range(0, K, p.range):
        many = np.zeros((rows, min(K, k + p.range) - k), np.float32)
        many[:M] = a[:, k:k + p.range]
        assert not plan(rows, N, many.shape[1]).waves
        part = product(many, b[k:k + p.range])[:M]
        want = part if want is None else want + part
    np.testing.assert_array_equal(product(a, b), want)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_no_further_from_float64_than_the_tile_kernels_order(shape):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K), rng = nd.gpu(0), shape, np.random.RandomState(11)
    p = plan(M, N, K)
    assert p.waves
    a, b = rng.normal(size=(M, K)).astype(np.float32), rng.normal(size=(K, N)).astype(np.float32)
    want = a.astype(np.float64) @ b.astype(np.float64)
    order = _rms(_in_ranges(a, b, p.tile_range) - want)
    for ta in (False, True):
        for tb in (False, True):
            c = nd.empty((M, N), ctx)
            L.matrix_multiply(nd.array(np.ascontiguousarray(a.T) if ta else a, ctx), ta, nd.array(np.ascontiguousarray(b.T) if tb else b, ctx), tb, c)
            assert _rms(c.asnumpy() - want) <= 1.15 * order, (ta, tb, _rms(c.asnumpy() - want) / order)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(64, 256, 1100), (64, 1000, 2048), (250, 256, 1024), (33, 70, 1003)])
def test_column_sums_have_the_tile_kernels_bits(shape):
    """Its order: of 16 rows a lane group adds its four as a tree, those of 256 rows one by one, and these; then the four groups, then the ranges."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K), rng = nd.gpu(0), shape, np.random.RandomState(3)
    p = plan(M, N, K)
    assert p.waves and p.range == p.tile_range
    b = rng.normal(size=(K, N)).astype(np.float32) + np.float32(0.5)
    c, s = nd.empty((M, N), ctx), nd.empty((N,), ctx)
    L.matrix_multiply_sums(nd.array(rng.normal(size=(K, M)).astype(np.float32), ctx), nd.array(b, ctx), c, s)
    total = np.zeros(N, np.float32)
    for k in range(0, K, p.range):
        rows = b[k:k + p.range]
        padded = np.zeros((-(-len(rows) // 256) * 256, N), np.float32)
        padded[:len(rows)] = rows
        four = padded.reshape(-1, 16, 4, 4, N)                      # [256 rows][16 rows][lane group][its rows]
        four = (four[:, :, :, 0] + four[:, :, :, 1]) + (four[:, :, :, 2] + four[:, :, :, 3])
        col = np.zeros((4, N), np.float32)
        for long in four:
            some = np.zeros((4, N), np.float32)
            for sixteen in long:
                some = some + sixteen
            col = col + some
        total = total + ((col[0] + col[1]) + (col[2] + col[3]))
    np.testing.assert_array_equal(s.asnumpy(), total)

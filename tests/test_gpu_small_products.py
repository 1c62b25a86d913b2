"""Products small enough that the waves of a block share the depth of one 16- or 32-wide tile (csrc/gemm_waves.h): edges of the tiles, of a
wave's 32 values and of the last 16-byte word; operands on 4-byte boundaries, plain, with more behind them, with column sums and over heads.

Bar: a sum of K fp32 products in any order is within K * 2^-24 of the sum of their magnitudes; what follows rounds once each (four more)."""
import numpy as np
import pytest

from test_gpu_product_tiles import _device

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def _operands(rng, M, N, K, ta, tb, lead=()):
    a = rng.normal(size=lead + ((K, M) if ta else (M, K))).astype(np.float32)
    b = rng.normal(size=lead + ((N, K) if tb else (K, N))).astype(np.float32)
    a64, b64 = (np.swapaxes(v, -1, -2) if t else v for v, t in ((a.astype(np.float64), ta), (b.astype(np.float64), tb)))
    return a, b, a64 @ b64, K * EPS * (np.abs(a64) @ np.abs(b64)) + 1e-30


# no depth at all, one share of it and a part, more shares than waves; rows and columns one off the tiles; a CU's worth of tiles and more
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("shape", [(3, 5, 0), (16, 16, 32), (17, 31, 33), (1, 48, 129), (33, 1, 31), (100, 250, 1027), (31, 97, 4098), (530, 270, 70)])
def test_products(shape, ta, tb, rng):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K) = nd.gpu(0), shape
    a, b, want, bound = _operands(rng, M, N, max(K, 1), ta, tb)
    if not K:
        a, b, want, bound = a[:, :0] if not ta else a[:0], b[:0] if not tb else b[:, :0], np.zeros((M, N)), np.zeros((M, N))
    bias, add, x = rng.normal(size=N).astype(np.float32), rng.normal(size=(M, N)).astype(np.float32), rng.normal(size=(M, N)).astype(np.float32)
    for shift in (0, 1) if K else (0,):
        ga, gb = _device(nd, ctx, a, shift), _device(nd, ctx, b, 3 * shift)
        c, r = (nd.array(np.full((M, N), 7, np.float32), ctx) for _ in range(2))
        L.matrix_multiply(ga, ta, gb, tb, c)
        plain = c.asnumpy()
        L.matrix_multiply_add(ga, ta, gb, tb, c, nd.array(bias, ctx), nd.array(add, ctx), r, gate=nd.array(x, ctx))
        more, gated = c.asnumpy(), r.asnumpy()
        for v in (ga, gb):
            if v._owner:
                v.handle.contents.data = v._owner[1]
        assert (np.abs(plain - want) <= bound).all(), (shape, ta, tb, shift)
        np.testing.assert_array_equal(more, plain + bias + add)
        np.testing.assert_array_equal(gated, np.where(x > 0, more, 0))


@pytest.mark.parametrize("shape", [(1, 1, 1), (16, 33, 31), (33, 31, 100), (300, 130, 1003), (20, 17, 4099)])
def test_column_sums(shape, rng):
    """Sums: each value passes at most K / 64 + 12 roundings (four of a group of 16 as a tree, a wave's groups one by one, lanes, waves)."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K) = nd.gpu(0), shape
    a, b, want, bound = _operands(rng, M, N, K, True, False)
    c, s = nd.array(np.full((M, N), 7, np.float32), ctx), nd.array(np.full(N, 7, np.float32), ctx)
    L.matrix_multiply_sums(nd.array(a, ctx), nd.array(b, ctx), c, s)
    assert (np.abs(c.asnumpy() - want) <= bound).all()
    b64 = b.astype(np.float64)
    assert (np.abs(s.asnumpy() - b64.sum(0)) <= (K / 64 + 12) * EPS * np.abs(b64).sum(0)).all()


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (3, 17, 33, 70), (6, 40, 50, 64), (2, 31, 5, 300)])
def test_batches(shape, ta, tb, rng):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (B, M, N, K) = nd.gpu(0), shape
    a, b, want, bound = _operands(rng, M, N, K, ta, tb, (B,))
    c = nd.array(np.full((B, M, N), 7, np.float32), ctx)
    L.batch_matrix_multiply(nd.array(a, ctx), ta, nd.array(b, ctx), tb, c)
    assert (np.abs(c.asnumpy() - want) <= bound).all()

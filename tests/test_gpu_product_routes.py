"""Both kernels of the matrix products at ragged sizes, on every tile, with the depth in one range and in several: each case says which
kernel and tile it is for, and the plan (csrc/tile_plan.h, compiled for the host) is asked whether it goes there.  csrc/gemm_waves.h: rows and
columns off its four tiles, depths off its 32 and its 16-byte words.  csrc/gemm_tile.h likewise, and over heads.

Bars: a sum of K fp32 products in any order is within K * 2^-24 of the sum of their magnitudes, one 2^-24 more for each range that is added
and for each operation behind it; what follows a product in its launch has the bits of the operators by themselves; sums of columns pass at
most K / 64 + 24 roundings (four of a group of 16 as a tree, groups in turn, lanes, ranges)."""
import numpy as np
import pytest

from product_plan import plan
from test_gpu_product_tiles import _device

EPS = 2.0 ** -24
WAVES, TILE = "waves", "tile"
# M, N, K, batch, kernel, its tile, ranges of the depth
ONE = [(17, 31, 11, 1, WAVES, (16, 16), 1), (17, 31, 133, 1, WAVES, (16, 16), 1), (113, 127, 159, 1, WAVES, (16, 16), 1), (147, 823, 229, 1, WAVES, (16, 16), 4),
       (33, 67, 163, 1, WAVES, (16, 16), 6), (1, 1102, 2019, 1, WAVES, (16, 16), 64),
       (449, 145, 33, 1, WAVES, (16, 32), 1), (197, 1189, 271, 1, WAVES, (16, 32), 3), (51, 1053, 183, 1, WAVES, (16, 32), 6),
       (597, 193, 61, 1, WAVES, (32, 16), 1), (755, 331, 333, 1, WAVES, (32, 16), 3), (1027, 97, 271, 1, WAVES, (32, 16), 5),
       (393, 483, 263, 1, WAVES, (32, 32), 3), (139, 919, 263, 1, WAVES, (32, 32), 5),
       (363, 1089, 1, 1, TILE, (64, 64), 1), (895, 441, 47, 1, TILE, (64, 64), 1), (515, 2047, 70, 1, TILE, (64, 64), 1),
       (1, 1, 1545, 1, TILE, (64, 64), 25), (31, 97, 4098, 1, TILE, (64, 64), 43), (129, 66, 2047, 1, TILE, (64, 64), 32), (1, 3000, 16387, 1, TILE, (64, 64), 16),
       (839, 1189, 907, 1, TILE, (64, 128), 5)]
MANY = [(13, 29, 37, 6, WAVES, (16, 16), 2), (1, 273, 11, 57, WAVES, (16, 32), 1), (1, 41, 143, 88, WAVES, (16, 32), 3), (287, 1, 53, 109, WAVES, (32, 16), 2),
        (21, 1, 227, 138, WAVES, (32, 16), 4), (1025, 19, 265, 6, WAVES, (32, 32), 3), (55, 17, 337, 100, WAVES, (32, 32), 4),
        (300, 200, 5, 100, TILE, (64, 64), 1), (257, 255, 64, 256, TILE, (64, 64), 1), (257, 255, 67, 40, TILE, (64, 128), 1), (1, 557, 43, 90, TILE, (64, 128), 1),
        (665, 1, 39, 124, TILE, (128, 64), 1), (1043, 1091, 37, 6, TILE, (128, 128), 1), (256, 256, 64, 256, TILE, (128, 128), 1)]
BOTH_WAYS = [(False, False), (False, True), (True, False), (True, True)]
_name = lambda case: "%dx%dx%d of %d" % (case[:3] + case[3:4])


@pytest.mark.parametrize("case", ONE + MANY, ids=_name)
def test_cases_go_where_they_say(case):
    M, N, K, batch, kernel, tile, ranges = case
    p = plan(M, N, K, batch)
    assert (WAVES if p.waves else TILE, p.tile, -(-K // p.range)) == (kernel, tile, ranges)


def _operands(rng, M, N, K, ta, tb, lead=()):
    a, b = rng.normal(size=lead + (M, K)).astype(np.float32), rng.normal(size=lead + (K, N)).astype(np.float32)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    a, b = (np.ascontiguousarray(np.swapaxes(v, -1, -2)) if t else v for v, t in ((a, ta), (b, tb)))
    return a, b, a64 @ b64, EPS * (np.abs(a64) @ np.abs(b64))


class _Shifted:
    """Arrays on the device, some floats behind a 16-byte boundary; they have their own memory back at the end."""

    def __init__(self, nd, ctx, *pairs):
        self.arrays = [_device(nd, ctx, v, shift) for v, shift in pairs]

    def __enter__(self):
        return self.arrays

    def __exit__(self, *_):
        for v in self.arrays:
            if v._owner:
                v.handle.contents.data = v._owner[1]


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", BOTH_WAYS)
@pytest.mark.parametrize("case", ONE, ids=_name)
def test_products(case, ta, tb, rng):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K, _, _, _, ranges) = nd.gpu(0), case
    a, b, want, size = _operands(rng, M, N, K, ta, tb)
    bias, add, x = rng.normal(size=N).astype(np.float32), rng.normal(size=(M, N)).astype(np.float32), rng.normal(size=(M, N)).astype(np.float32)
    for shift in (0, 1):
        c, r, h, s = (nd.array(np.full(z, 7, np.float32), ctx) for z in ((M, N), (M, N), (M, N), (N,)))
        with _Shifted(nd, ctx, (a, shift), (b, 3 * shift), (bias, shift), (add, shift), (x, 2 * shift)) as (ga, gb, gbias, gadd, gx):
            L.matrix_multiply(ga, ta, gb, tb, c)
            plain = c.asnumpy()
            L.matrix_multiply_add(ga, ta, gb, tb, c, gbias, gadd, r, gate=gx)
            L.matrix_multiply_add(ga, ta, gb, tb, h, gbias, None, None)
            more, gated, biased = c.asnumpy(), r.asnumpy(), h.asnumpy()
            if ta and not tb:
                L.matrix_multiply_sums(ga, gb, h, s)
                np.testing.assert_array_equal(h.asnumpy(), plain)
                b64 = b.astype(np.float64)
                assert (np.abs(s.asnumpy() - b64.sum(0)) <= (K / 64 + 24 + ranges) * EPS * np.abs(b64).sum(0)).all()
        assert (np.abs(plain - want) <= (K + ranges) * size).all(), shift
        np.testing.assert_array_equal(biased, plain + bias)
        np.testing.assert_array_equal(more, plain + bias + add)
        np.testing.assert_array_equal(gated, np.where(x > 0, more, 0))


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", BOTH_WAYS)
@pytest.mark.parametrize("case", MANY, ids=_name)
def test_batches(case, ta, tb, rng):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K, batch, _, _, ranges) = nd.gpu(0), case
    a, b, want, size = _operands(rng, M, N, K, ta, tb, (batch,))
    c = nd.array(np.full((batch, M, N), 7, np.float32), ctx)
    with _Shifted(nd, ctx, (a, 1), (b, 3)) as (ga, gb):
        L.batch_matrix_multiply(ga, ta, gb, tb, c)
        assert (np.abs(c.asnumpy() - want) <= (K + ranges) * size).all()


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("case", MANY, ids=_name)
def test_products_over_heads(case, ta, tb, rng):
    """A product with a scale, a mask, the causal fill and an addend, from heads side by side in a row; and one from heads one by one."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K, batch, _, _, ranges) = nd.gpu(0), case
    heads = next(h for h in (8, 4, 3, 2, 1) if batch % h == 0)
    n = batch // heads
    a, b, want, size = _operands(rng, M, N, K, ta, tb, (n, heads))
    side = lambda v: np.ascontiguousarray(v.transpose(0, 2, 1, 3).reshape(n, v.shape[2], -1))
    mask, add = rng.randint(0, 3, size=(n, N)).astype(np.float32), rng.normal(size=(n, heads, M, N)).astype(np.float32)
    alpha, value, fill = np.float32(0.3), -2.0, 5.0
    want, size = alpha * want, alpha * size
    c = nd.array(np.full((n, M, heads * N), 7, np.float32), ctx)
    L.heads_matrix_multiply(nd.array(side(a), ctx), ta, nd.array(side(b), ctx), tb, c, heads, alpha, nd.array(mask, ctx), value, True, fill, nd.array(side(add), ctx))
    more = want + np.where(mask != 0, 0, value)[:, None, None, :]
    more = np.where(np.triu(np.ones((M, N), bool), 1), fill, more) + add
    got = c.asnumpy().reshape(n, M, heads, N).transpose(0, 2, 1, 3)
    assert (np.abs(got - more) <= (K + ranges + 1) * size + 4 * EPS * (np.abs(want) + abs(value) + fill + np.abs(add))).all()
    c = nd.array(np.full((n, heads, M, N), 7, np.float32), ctx)
    L.heads_matrix_multiply(nd.array(a, ctx), ta, nd.array(b, ctx), tb, c, heads, alpha)
    assert (np.abs(c.asnumpy() - want) <= (K + ranges + 2) * size).all()


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", BOTH_WAYS)
@pytest.mark.parametrize("case", [c for c in ONE + MANY if min(c[:2]) > 8 and c[2] > 1 and c[0] * c[1] * c[3] < 4e6], ids=_name)
def test_infinities_stay_in_their_rows_and_columns(case, ta, tb, rng):
    """A word that the end of K cuts holds the next row's first values, and behind a batch's last row lies the next batch."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K, batch, _, _, _) = nd.gpu(0), case
    a, b = rng.normal(size=(batch, M, K)).astype(np.float32), rng.normal(size=(batch, K, N)).astype(np.float32)
    a[0, 7, 0], b[0, 0, 5] = np.inf, np.nan
    if batch > 1:
        a[1, 0, :], b[1, :, 0] = np.inf, np.nan
    ga, gb = (nd.array(np.ascontiguousarray(v.transpose(0, 2, 1)) if t else v, ctx) for v, t in ((a, ta), (b, tb)))
    c = nd.array(np.full((batch, M, N), 7, np.float32), ctx)
    if batch > 1:
        L.batch_matrix_multiply(ga, ta, gb, tb, c)
    else:
        L.matrix_multiply(nd.view(ga, ga.shape[1:]), ta, nd.view(gb, gb.shape[1:]), tb, nd.view(c, (M, N)))
    bad = np.zeros((batch, M, N), bool)
    bad[0, 7, :] = bad[0, :, 5] = True
    if batch > 1:
        bad[1, 0, :] = bad[1, :, 0] = True
    np.testing.assert_array_equal(~np.isfinite(c.asnumpy()), bad)

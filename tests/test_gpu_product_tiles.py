"""The tile kernel of the matrix products (csrc/gemm_tile.h) at the edges of its tiles, its 32-deep steps and its 16-byte
words, plain and batched, from operands on 4-byte boundaries: against float64 products.

Bar: a sum of K fp32 products, however it is ordered, is within K * 2^-24 of the sum of their magnitudes (Higham's
gamma_K to first order); one more 2^-24 for each of up to 64 ranges' results added by the fold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# M, N, K: one value; one past a word, a step and a tile; whole tiles; ranges of K that the last one does not fill
SHAPES = [(1, 1, 1), (1, 5, 7), (65, 129, 33), (128, 128, 32), (129, 63, 31), (64, 130, 66), (127, 4, 1030), (10, 256, 785), (300, 132, 1002),
          (1024, 640, 96)]


def _bound(a64, b64):
    return (a64.shape[-1] + 64) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64)) + 1e-30


def _device(nd, ctx, a, shift):
    """a on the device, `shift` floats behind a 16-byte boundary."""
    whole = nd.array(np.concatenate([np.zeros(shift, np.float32), a.reshape(-1)]).reshape(-1, 1), ctx)
    if not shift:
        return nd.array(a, ctx)
    view = nd.empty(a.shape, ctx)
    own = view.handle.contents.data
    view.handle.contents.data = whole.handle.contents.data + 4 * shift
    view._owner = (whole, own)
    return view


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("shape", SHAPES)
def test_products_at_the_edges(shape, ta, tb, rng):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K) = nd.gpu(0), shape
    a = rng.normal(size=(K, M) if ta else (M, K)).astype(np.float32)
    b = rng.normal(size=(N, K) if tb else (K, N)).astype(np.float32)
    a64, b64 = (a.T if ta else a).astype(np.float64), (b.T if tb else b).astype(np.float64)
    for shift in (0, 1):
        ga, gb, c = _device(nd, ctx, a, shift), _device(nd, ctx, b, 3 * shift), nd.array(np.full((M, N), 7, np.float32), ctx)
        L.matrix_multiply(ga, ta, gb, tb, c)
        got = c.asnumpy()
        for v in (ga, gb):          # give the arrays their own memory back before they are freed
            if v._owner:
                v.handle.contents.data = v._owner[1]
        assert (np.abs(got - a64 @ b64) <= _bound(a64, b64)).all(), (shape, ta, tb, shift)


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("shape", [(3, 1, 1, 1), (5, 77, 50, 64), (40, 129, 65, 33), (20, 64, 128, 77)])
def test_batched_products_at_the_edges(shape, ta, tb, rng):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (B, M, N, K) = nd.gpu(0), shape
    a = rng.normal(size=(B, K, M) if ta else (B, M, K)).astype(np.float32)
    b = rng.normal(size=(B, N, K) if tb else (B, K, N)).astype(np.float32)
    a64, b64 = (a.transpose(0, 2, 1) if ta else a).astype(np.float64), (b.transpose(0, 2, 1) if tb else b).astype(np.float64)
    c = nd.array(np.full((B, M, N), 7, np.float32), ctx)
    L.batch_matrix_multiply(nd.array(a, ctx), ta, nd.array(b, ctx), tb, c)
    assert (np.abs(c.asnumpy() - a64 @ b64) <= _bound(a64, b64)).all(), (shape, ta, tb)


@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("shape", [(70, 45, 5), (40, 130, 33), (65, 66, 1030)])
def test_infinities_stay_in_their_rows_and_columns(shape, ta, tb, rng):
    """A word that the end of K cuts holds the next row's first values, and behind a batch's last row lies the next batch: neither may
    reach another row's sums, not even times zero."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (M, N, K) = nd.gpu(0), shape
    a, b = rng.normal(size=(2, M, K)).astype(np.float32), rng.normal(size=(2, K, N)).astype(np.float32)
    a[0, 7, 0], b[0, 0, 5] = np.inf, np.nan
    a[1, 0, :], b[1, :, 0] = np.inf, np.nan      # behind the first batch
    ga, gb = (np.ascontiguousarray(v.transpose(0, 2, 1)) if t else v for v, t in ((a, ta), (b, tb)))
    c, batched = nd.empty((M, N), ctx), nd.empty((2, M, N), ctx)
    L.matrix_multiply(nd.array(ga[0], ctx), ta, nd.array(gb[0], ctx), tb, c)
    L.batch_matrix_multiply(nd.array(ga, ctx), ta, nd.array(gb, ctx), tb, batched)
    for got, row, col in ((c.asnumpy(), 7, 5), (batched.asnumpy()[0], 7, 5), (batched.asnumpy()[1], 0, 0)):
        own = np.zeros((M, N), bool)
        own[row, :] = own[:, col] = True
        finite = np.isfinite(got)
        assert finite[~own].all() and not finite[own].any()


def test_rows_of_the_result_beyond_32_bit_offsets(rng):
    """64 rows of the result span more than 2 GiB: every row whole, nothing past the last."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, M, N, K = nd.gpu(0), 66, (1 << 23) + 5, 2
    a, b = rng.normal(size=(M, K)).astype(np.float32), np.resize(rng.normal(size=(K, 1009)).astype(np.float32), (K, N))
    c = nd.array(np.full((M, N), 7, np.float32), ctx)
    L.matrix_multiply(nd.array(a, ctx), False, nd.array(b, ctx), False, c)
    got, b64 = c.asnumpy(), b.astype(np.float64)
    for row in range(M):
        a64 = a[row:row + 1].astype(np.float64)
        assert (np.abs(got[row] - (a64 @ b64)[0]) <= _bound(a64, b64)[0]).all(), row


@pytest.mark.parametrize("M,N,ta,batched", [(48, 512, False, False), (130, 512, True, False), (40, 512, True, True), (512, 40, False, True), (130, 512, True, True)])
def test_operands_beyond_32_bit_offsets(M, N, ta, batched, rng):
    """An operand of more than 2 GiB, K far longer than the result is wide.  Whole numbers of at most 1, so that every sum is exact in
    fp32 in whatever order; a plain product is cut into ranges of K (they leave a workspace)."""
    from tsplit_amd import gpu_links as L, ndarray as nd
    from tsplit_amd.profiler import Profiler
    ctx, K = nd.gpu(0), (1 << 29) // max(M, N) + 4321
    wide = rng.randint(-1, 2, size=(K, max(M, N))).astype(np.float32)
    slim = rng.randint(-1, 2, size=(K, min(M, N))).astype(np.float32)
    want = np.zeros((min(M, N), max(M, N)), np.float32)
    for at in range(0, K, 1 << 16):
        want += slim[at:at + (1 << 16)].T @ wide[at:at + (1 << 16)]
    a, b, want = (slim, wide, want) if M < N else (wide, slim, want.T)
    a = a if ta else np.ascontiguousarray(a.T)
    if batched:
        c = nd.empty((1, M, N), ctx)
        L.batch_matrix_multiply(nd.array(a[None], ctx), ta, nd.array(b[None], ctx), False, c)
        np.testing.assert_array_equal(c.asnumpy()[0], want)
    else:
        c, p = nd.empty((M, N), ctx), Profiler()
        L.matrix_multiply(nd.array(a, ctx), ta, nd.array(b, ctx), False, c, profiler=p)
        np.testing.assert_array_equal(c.asnumpy(), want)
        assert p.workspace_memory > 0

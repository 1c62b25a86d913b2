"""Calls that run the operators behind a product in its launch, class indices as labels, token look-up with positions.

Bars: a product with a bias, an addend and Relu behind it gives the bits of the product, broadcast, addition and Relu one by one; products over
heads and the loss are within K (or the columns') roundings of float64; a whole Transformer is held to the oracle by test_gpu_graphs.py."""
import numpy as np
import pytest

from oracle import ops as O

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def _dev(*arrays):
    from tsplit_amd import ndarray as nd
    return [nd.array(a, nd.gpu(0)) for a in arrays]


def _full(shape):
    return _dev(np.full(shape, 7, np.float32))[0]


# edges of the tiles; K in ranges (few tiles, deep); columns that are no multiple of a word; one row
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("shape", [(1, 5, 3), (64, 64, 32), (65, 130, 33), (129, 66, 2047), (100, 1024, 4096), (515, 2047, 70)])
def test_product_with_bias_addend_and_relu(shape, ta, tb, rng):
    from tsplit_amd import gpu_links as L
    M, N, K = shape
    a, b = rng.normal(size=(K, M) if ta else (M, K)).astype(np.float32), rng.normal(size=(N, K) if tb else (K, N)).astype(np.float32)
    bias, add = rng.normal(size=N).astype(np.float32), rng.normal(size=(M, N)).astype(np.float32)
    ga, gb, gbias, gadd = _dev(a, b, bias, add)
    plain = _full((M, N))
    L.matrix_multiply(ga, ta, gb, tb, plain)
    product = plain.asnumpy()
    for with_bias, with_add, with_relu in ((True, True, True), (True, False, False), (False, True, False), (False, False, True)):
        c, r = _full((M, N)), _full((M, N))
        L.matrix_multiply_add(ga, ta, gb, tb, c, gbias if with_bias else None, gadd if with_add else None, r if with_relu else None)
        want = product + bias if with_bias else product
        want = want + add if with_add else want
        np.testing.assert_array_equal(c.asnumpy(), want)
        if with_relu:
            np.testing.assert_array_equal(r.asnumpy(), np.maximum(want, 0))
    x = rng.normal(size=(M, N)).astype(np.float32)        # a Relu's input: zeros of both signs and NaN among it
    x.ravel()[::5], x.ravel()[1::7], x.ravel()[2::11] = 0.0, -0.0, np.nan
    gx, c, r, grad = _dev(x)[0], _full((M, N)), _full((M, N)), _full((M, N))
    L.matrix_multiply_add(ga, ta, gb, tb, c, addend=gadd, relu=r, gate=gx)
    L.relu_gradient(gx, c, grad)
    np.testing.assert_array_equal(c.asnumpy(), product + add)
    np.testing.assert_array_equal(r.asnumpy(), grad.asnumpy())
    L.matrix_multiply_add(ga, ta, gb, tb, c, addend=gadd, gate=gx)
    np.testing.assert_array_equal(c.asnumpy(), grad.asnumpy())
    with pytest.raises(RuntimeError):
        L.matrix_multiply_add(ga, ta, gb, tb, c, gate=c)
    acc = _dev(add)[0]                                    # added to in place
    L.matrix_multiply_add(ga, ta, gb, tb, acc, addend=acc)
    np.testing.assert_array_equal(acc.asnumpy(), product + add)


# tiles' edges, one range and many, depths off the steps, columns that are no words, one column; operands of three axes; split-bf16
@pytest.mark.parametrize("shape", [(1, 1, 1), (64, 64, 32), (65, 130, 33), (33, 35, 5000), (512, 512, 8192), (256, 1024, 250), (130, 66, 2047), (784, 10, 100)])
def test_product_with_column_sums(shape, rng):
    """Bar of the sums: every value passes at most 40 roundings of partial sums (pairs in a step, eight steps, 64 groups of steps as a tree
    of ranges), each below 2^-24 of the sum of magnitudes."""
    from tsplit_amd import gpu_links as L
    M, N, K = shape
    a, b = rng.normal(size=(K, M)).astype(np.float32), (rng.normal(size=(K, N)) + 0.5).astype(np.float32)
    ga, gb = _dev(a, b)
    plain = _full((M, N))
    L.matrix_multiply(ga, True, gb, False, plain)
    for split in (False, True):
        c, sums = _full((M, N)), _full((N,))
        was = L.split_bf16(split)
        try:
            L.matrix_multiply_sums(ga, gb, c, sums)
        finally:
            L.split_bf16(was)
        if not split:
            np.testing.assert_array_equal(c.asnumpy(), plain.asnumpy())
        assert np.all(np.abs(sums.asnumpy() - b.astype(np.float64).sum(0)) <= 40 * EPS * np.abs(b.astype(np.float64)).sum(0))
    if K % 2 == 0:
        from tsplit_amd import ndarray as nd
        c, sums = _full((M, N)), _full((N,))
        L.matrix_multiply_sums(nd.view(ga, (2, K // 2, M)), nd.view(gb, (2, K // 2, N)), c, sums)
        np.testing.assert_array_equal(c.asnumpy(), plain.asnumpy())
    with pytest.raises(RuntimeError):
        L.matrix_multiply_sums(ga, gb, plain, _full((N + 1,)))


def test_column_sums_of_ranges_deeper_than_16384_rows_are_the_reductions_own(rng):
    """(1344 x 1472 fill the chip, so 16640 rows stay one range)"""
    from tsplit_amd import gpu_links as L
    M, N, K = 1344, 1472, 16640
    draw = np.random.default_rng(rng.randint(1 << 30))
    ga, gb = _dev(draw.standard_normal((K, M), np.float32), draw.standard_normal((K, N), np.float32))
    plain, c, want, sums = _full((M, N)), _full((M, N)), _full((N,)), _full((N,))
    L.matrix_multiply(ga, True, gb, False, plain)
    L.reduce_sum_axis_zero(gb, want)
    L.matrix_multiply_sums(ga, gb, c, sums)
    np.testing.assert_array_equal(c.asnumpy(), plain.asnumpy())
    np.testing.assert_array_equal(sums.asnumpy(), want.asnumpy())


def test_product_with_more_split_bf16_and_arrays_of_more_axes(rng):
    from tsplit_amd import gpu_links as L
    x, w, add = rng.normal(size=(3, 7, 40)).astype(np.float32), rng.normal(size=(40, 36)).astype(np.float32), rng.normal(size=(3, 7, 36)).astype(np.float32)
    gx, gw, acc = _dev(x, w, add)
    c = _full((3, 7, 36))
    L.matrix_multiply_add(gx, False, gw, False, c, addend=acc)
    want = x.astype(np.float64) @ w + add
    np.testing.assert_allclose(c.asnumpy(), want, rtol=0, atol=42 * EPS * 40)
    was = L.split_bf16(True)
    try:
        L.matrix_multiply_add(gx, False, gw, False, acc, addend=acc)      # the product of another kernel, the sum behind it
    finally:
        L.split_bf16(was)
    np.testing.assert_allclose(acc.asnumpy(), want, rtol=0, atol=42 * EPS * 40)
    with pytest.raises(RuntimeError):
        L.matrix_multiply_add(gx, False, gw, False, c, bias=_full((35,)))
    with pytest.raises(RuntimeError):
        L.matrix_multiply_add(gx, False, gw, True, c)


# one row, one column, more rows than columns and fewer, columns beyond one pass of a block
@pytest.mark.parametrize("shape", [(3, 1), (1, 4), (2, 3, 7, 5), (2, 2, 5, 9), (2, 70, 600), (0, 4)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("in_place", [False, True])
def test_scale_and_causal_selection(shape, causal, in_place, rng):
    from tsplit_amd import gpu_links as L
    x = rng.normal(size=shape).astype(np.float32)
    x.ravel()[::5] = np.inf
    gx = _dev(x)[0]
    out = gx if in_place else _full(shape)
    L.heads_scale(gx, -0.3, causal, out)
    want = (np.where(np.tril(np.ones(shape[-2:], bool)), x, np.float32(0)) if causal else x) * np.float32(-0.3)
    np.testing.assert_array_equal(out.asnumpy().view(np.uint32), want.view(np.uint32))
    with pytest.raises(RuntimeError):
        L.heads_scale(gx, 1.0, causal, _full((3, 2, 2)))


# heads' widths that are a word, none, larger than a tile; lengths off the tiles, few and many columns, wide results in words or not
@pytest.mark.parametrize("n,heads,tq,tk,dh", [(2, 3, 5, 7, 4), (3, 2, 65, 33, 33), (1, 4, 128, 64, 64), (2, 1, 70, 130, 66), (5, 4, 50, 77, 64)])
@pytest.mark.parametrize("causal", [False, True])
def test_products_over_heads(n, heads, tq, tk, dh, causal, rng):
    from tsplit_amd import gpu_links as L
    d = heads * dh
    q, k, v = (rng.normal(size=(n, t, d)).astype(np.float32) for t in (tq, tk, tk))
    mask = rng.randint(0, 3, size=(n, tk)).astype(np.float32)
    add = rng.normal(size=(n, tq, d)).astype(np.float32)
    gq, gk, gv, gmask, gadd = _dev(q, k, v, mask, add)
    apart = lambda x: x.astype(np.float64).reshape(n, -1, heads, dh).transpose(0, 2, 1, 3)
    together = lambda x: x.transpose(0, 2, 1, 3).reshape(n, -1, d)
    alpha, value = 0.3, -2.0
    scores = _full((n, heads, tq, tk))
    L.heads_matrix_multiply(gq, False, gk, True, scores, heads, alpha, gmask, value, causal, 5.0)
    want = alpha * (apart(q) @ apart(k).transpose(0, 1, 3, 2)) + np.where(mask != 0, 0, value)[:, None, None, :]
    size = alpha * (np.abs(apart(q)) @ np.abs(apart(k)).transpose(0, 1, 3, 2)) + 2
    if causal:
        future = np.triu(np.ones((tq, tk), bool), 1)
        want[:, :, future] = 5.0
    got = scores.asnumpy()
    assert (np.abs(got - want) <= (dh + 3) * EPS * size).all()
    context = _full((n, tq, d))
    L.heads_matrix_multiply(scores, False, gv, False, context, heads, addend=gadd)
    want = together(got.astype(np.float64) @ apart(v)) + add
    size = together(np.abs(got).astype(np.float64) @ np.abs(apart(v))) + np.abs(add)
    assert (np.abs(context.asnumpy() - want) <= (tk + 2) * EPS * size).all()
    dv = _full((n, tk, d))                                # scores' times rows of the context
    L.heads_matrix_multiply(scores, True, gq, False, dv, heads)
    want = together(got.astype(np.float64).transpose(0, 1, 3, 2) @ apart(q))
    size = together(np.abs(got).astype(np.float64).transpose(0, 1, 3, 2) @ np.abs(apart(q)))
    assert (np.abs(dv.asnumpy() - want) <= (tq + 2) * EPS * size).all()
    with pytest.raises(RuntimeError):
        L.heads_matrix_multiply(gq, False, gk, True, _full((n, heads, tq, tk + 1)), heads)


# columns: a wave's 4 and 16 words, 512 threads' 4, 16 and 64, past what registers hold; in words of four or not
@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 256), (5, 257), (7, 1024), (2, 1025), (3, 1028), (4, 8192), (3, 8193), (2, 8196), (2, 32768), (3, 32769),
                                       (2, 32772), (2, 40001)])
def test_cross_entropy_with_class_indices_and_with_label_arrays(rows, cols, rng):
    from tsplit_amd import gpu_links as L
    y = (3 * rng.normal(size=(rows, cols))).astype(np.float32)
    ids = rng.randint(0, cols, size=rows).astype(np.float32)
    ids[-1] = cols if rows > 1 else ids[-1]               # a class that does not exist: no hot value
    on, off = 0.9, 0.1 / cols
    lab = (on * (np.arange(cols) == ids[:, None]) + off)
    gy, gids, glab, gone = _dev(y, ids, lab.astype(np.float32), np.float32([0.5]))
    y64 = y.astype(np.float64)
    m = y64.max(1, keepdims=True)
    e = np.exp(y64 - m)
    s = e.sum(1, keepdims=True)
    per = lab * (np.log(s) - (y64 - m))
    want = per.sum(1).mean()
    grad = (e / s - lab) * 0.5 / rows
    for ids_form in (True, False):
        loss, g = _full((1,)), _full((rows, cols))
        if ids_form:
            L.softmax_cross_entropy_ids(gy, gids, on, off, loss)
            L.softmax_cross_entropy_ids_gradient(gy, gids, on, off, gone, g)
        else:
            L.softmax_cross_entropy(gy, glab, loss)
            L.softmax_cross_entropy_gradient(gy, glab, gone, g)
        # a thread's and the block's sums: fewer than 100 roundings each, exp and log within 4
        assert abs(loss.asnumpy()[0] - want) <= 100 * EPS * (np.abs(per).sum(1).mean() + 1)
        assert (np.abs(g.asnumpy() - grad) <= 100 * EPS * (e / s + lab) * 0.5 / rows).all()


# a wave's row, a block's in words and not, rows that registers do not hold; a loss without smoothing and with
@pytest.mark.parametrize("cols", [200, 1000, 5000, 5003, 40000, 40001])
@pytest.mark.parametrize("smoothing", [0.0, 0.1])
def test_cross_entropy_of_logits_masked_with_the_lowest_value(cols, smoothing, rng):
    from tsplit_amd import gpu_links as L
    y = rng.normal(size=(3, cols)).astype(np.float32)
    masked = rng.rand(3, cols) < 0.5
    masked[:, :2] = False
    y[masked] = np.finfo(np.float32).min
    ids = np.float32([0, 1, 1])
    on, off = 1.0 - smoothing, smoothing / cols
    lab = on * (np.arange(cols) == ids[:, None]) + off
    gy, gids, glab, loss, other = _dev(y, ids, lab.astype(np.float32)) + [_full((1,)), _full((1,))]
    L.softmax_cross_entropy_ids(gy, gids, on, off, loss)
    L.softmax_cross_entropy(gy, glab, other)
    y64 = y.astype(np.float64)
    m = y64.max(1, keepdims=True)
    per = lab * (np.log(np.exp(y64 - m).sum(1, keepdims=True)) - (y64 - m))
    for got in (loss, other):
        assert abs(got.asnumpy()[0] - per.sum(1).mean()) <= 100 * EPS * (np.abs(per).sum(1).mean() + 1)


@pytest.mark.parametrize("width", [64, 37])
def test_look_up_with_positions(width, rng):
    from tsplit_amd import gpu_links as L
    table, pos = rng.normal(size=(11, width)).astype(np.float32), rng.normal(size=(3, 5, width)).astype(np.float32)
    ids = rng.randint(0, 12, size=(3, 5)).astype(np.float32)      # 11 lies outside the table
    ids[0, :2] = 0
    dy, old = rng.normal(size=pos.shape).astype(np.float32), rng.normal(size=table.shape).astype(np.float32)
    gt, gi, gp, gdy, gold = _dev(table, ids, pos, dy, old)
    out, dt = _full(pos.shape), _full(table.shape)
    L.embedding_add(gt, gi, 0.25, gp, out)
    inside = ids < 11
    rows = O.embedding_lookup(table, np.where(inside, ids, 0)) * inside[..., None]
    want = 0.25 * rows.astype(np.float64) + np.where(ids[..., None] != 0, pos, 0)
    np.testing.assert_allclose(out.asnumpy(), want, rtol=0, atol=2 * EPS * 8)
    L.embedding_add_gradient(gdy, gi, 0.25, dt)
    want = O.embedding_lookup_grad(0.25 * dy * inside[..., None], np.where(inside, ids, 0), table.shape)
    np.testing.assert_allclose(dt.asnumpy(), want, rtol=0, atol=16 * EPS * 16)
    L.embedding_add_gradient(gdy, gi, 0.25, gold, add_to=True)
    np.testing.assert_allclose(gold.asnumpy(), want + old, rtol=0, atol=16 * EPS * 16)


def test_views_keep_their_array_and_leaves_are_copied(rng):
    """An operator's output reshaped on the tape is a view of it; an input is copied, so writing it again changes nothing behind."""
    from tsplit_amd import graph, ndarray as nd
    x = rng.normal(size=(6, 4)).astype(np.float32)
    t = graph.Tape(graph.GpuBackend())
    v = t.const(t.b.from_numpy(x), x.shape)
    copied = t.reshape(v, (4, 6))
    y = t.scale(v, 2.0)
    seen = t.reshape(y, (3, 8))
    assert seen.value.data_ptr == y.value.data_ptr and copied.value.data_ptr != v.value.data_ptr
    v.value[:] = np.zeros_like(x)
    y.value = None
    np.testing.assert_array_equal(copied.value.asnumpy(), x.reshape(4, 6))
    np.testing.assert_array_equal(seen.value.asnumpy(), (2 * x).reshape(3, 8))
    with pytest.raises(RuntimeError):
        nd.view(seen.value, (5, 5))


def test_scores_read_twice_and_leaf_gradients_over_two_sweeps(rng):
    """Scores that another operator reads too take their scale and selection in an operator of its own; a leaf's gradient array is the
    caller's once a sweep has ended: a second sweep adds into another one."""
    from oracle_backend import OracleBackend
    from tsplit_amd import graph
    qs, ks, vs = (rng.normal(size=(2, t, 8)).astype(np.float32) for t in (5, 6, 6))
    lab = np.full((2 * 5, 8), 0.125, np.float32)
    got = {}
    for tag, backend in (("gpu", graph.GpuBackend()), ("oracle", OracleBackend())):
        t = graph.Tape(backend)
        leaves = [t.param(backend.from_numpy(a), a.shape) for a in (qs, ks, vs)]
        grads = []
        for _ in range(2):
            q, k, v = leaves
            scores = t.head_scores(q, k, 2, 0.5, None, -1.0, True)
            out = t.head_context(scores, v, 2, q)
            more = t.head_context(scores, v, 2)
            loss = t.softmax_ce(t.reshape(t.add(out, more), (10, 8)), t.const(backend.from_numpy(lab), lab.shape))
            t.backward(loss)
            grads.append([p.grad for p in leaves])
        first, second = ([np.array(backend.to_numpy(g)) for g in gs] for gs in grads)
        for a, b in zip(first, second):
            np.testing.assert_allclose(b, 2 * a, rtol=1e-4, atol=1e-6)
        got[tag] = first
    for a, b in zip(got["gpu"], got["oracle"]):
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-5 * np.abs(b).max())

"""BatchNorm + Relu + a sum in one call: the bits of the two calls, values and saved statistics, on every forward kernel; and a tape's
node with the sum in it against the nodes one by one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# a channel in one block, of words and of values; planes of words, with edges, of three values (value by value), and an array off 16 bytes
SHAPES = [((2, 3, 1, 1), False), ((33, 3, 11, 11), False), ((64, 2, 16, 16), False), ((65, 3, 16, 16), False), ((101, 3, 13, 13), False),
          ((5501, 5, 3, 1), False), ((101, 3, 13, 13), True), ((1, 1, 132, 128), False)]


@pytest.mark.parametrize("shape,off", SHAPES)
@pytest.mark.parametrize("exact", [False, True])
def test_bits_of_the_two_calls(shape, off, exact, rng):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx, (n, c, h, w) = nd.gpu(0), shape
    x, more = (rng.normal(size=shape).astype(np.float32) for _ in range(2))
    more.reshape(-1)[::61] = np.nan
    gamma, beta = (nd.array(rng.normal(size=(1, c, 1, 1)).astype(np.float32), ctx) for _ in range(2))
    gm = nd.array(more, ctx)
    gx = nd.slice_for_micro_tensor(nd.array(np.concatenate([x, x]), ctx), 1, 2) if off else nd.array(x, ctx)
    stats = (c, 2) if exact else (1, c, 1, 1)
    a, b, a2, b2 = (nd.empty(stats, ctx) for _ in range(4))
    r, two, one = (nd.array(np.full(shape, 7, np.float32), ctx) for _ in range(3))
    L.batch_norm_relu(gx, gamma, beta, r, a, b, 0.01)
    L.matrix_elementwise_add(r, gm, two)
    L.batch_norm_relu_add(gx, gamma, beta, gm, one, a2, b2, 0.01)
    for p, q in ((one, two), (a, a2), (b, b2)):
        np.testing.assert_array_equal(p.asnumpy(), q.asnumpy())
    with pytest.raises(RuntimeError):
        L.batch_norm_relu_add(gx, gamma, beta, one, one, a2, b2, 0.01)


@pytest.mark.parametrize("fuse", [False, True])
def test_a_tapes_residual_block(fuse):
    from tsplit_amd import graph, ndarray as nd, workloads
    rng = np.random.default_rng(3)
    x, y = rng.standard_normal((3, 3, 64, 64), dtype=np.float32), np.eye(10, dtype=np.float32)[:3]

    def step(one_node):
        b = graph.GpuBackend(nd.gpu(0))
        t = graph.Tape(b)
        t.fuse_bn_relu = fuse
        if not one_node:
            t.bn_relu_then_add = lambda x, gamma, beta, residual, eps: t.add(t.bn_then_relu(x, gamma, beta, eps), residual)
        binder = workloads.Binder(t, workloads.ParamStore(5))
        loss, logits = workloads.resnet(t, binder, binder.input(x), binder.input(y), blocks=(2, 1, 1, 2), base=8, classes=10)
        t.backward(loss)
        return [logits.value.asnumpy()] + [v.grad.asnumpy() for v in binder.vars.values() if v.needs_grad]
    for one, two in zip(step(True), step(False)):
        np.testing.assert_array_equal(one, two)

"""Values that outlive the tape that made them: carried into another tape, or used again on their own after its reverse sweep, they are
leaves there, with their own gradient, whatever other call has the number they once had.  On the oracle backend, alone and with the
primitives that a device backend has for products with something behind them."""
import numpy as np
import pytest

from oracle_backend import OracleBackend, WithMore
from tsplit_amd import graph


BACKENDS = [OracleBackend, WithMore]


def _arrays(*shapes):
    rng = np.random.RandomState(3)
    return [rng.normal(size=s).astype(np.float32) for s in shapes]


def _carried(tape, value, calls):
    """A value that `tape` made as its operator call number `calls`."""
    v = tape.param(value, value.shape)
    for _ in range(calls + 1):
        v = tape.scale(v, 1.0)
    assert v.node == calls
    return v


def _loss(t, logits):
    n, c = logits.shape
    return t.softmax_ce(logits, t.const(np.eye(c, dtype=np.float32)[np.arange(n) % c], (n, c)))


@pytest.mark.parametrize("backend", BACKENDS)
@pytest.mark.parametrize("again", [False, True])
def test_a_value_is_used_on_another_tape_or_after_its_own_sweep(backend, again):
    x, w0, w1 = _arrays((5, 6), (6, 7), (7, 4))
    first = graph.Tape(backend())
    h = first.relu(first.matmul(first.const(x, x.shape), first.param(w0, w0.shape)))
    if again:
        first.backward(_loss(first, first.matmul(h, first.param(w1, w1.shape))))
    t = first if again else graph.Tape(backend())
    w = t.param(w1, w1.shape)
    grads = []
    for carried in (h, graph.Tape(backend()).param(np.array(h.value), h.shape)):
        carried.grad = w.grad = None
        t.backward(_loss(t, t.matmul(t.relu(carried), w)))
        grads.append((np.array(carried.grad), np.array(w.grad)))
    for a, b in zip(*grads):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("backend", BACKENDS)
def test_a_carried_value_takes_no_other_calls_relu_gradient(backend):
    x, w0, v, w1 = _arrays((5, 6), (6, 7), (5, 7), (7, 4))
    grads = []
    for number in (1, None):
        t = graph.Tape(backend())
        carried = _carried(graph.Tape(backend()), v, number) if number is not None else t.param(v, v.shape)
        t.relu(t.matmul(t.const(x, x.shape), t.param(w0, w0.shape)))      # calls 0 and 1, which nothing reads
        w = t.param(w1, w1.shape)
        t.backward(_loss(t, t.matmul(carried, w)))
        grads.append((np.array(carried.grad), np.array(w.grad)))
    for a, b in zip(*grads):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("backend", BACKENDS)
def test_a_carried_value_takes_no_other_calls_relu(backend):
    x, w0, b0, v = _arrays((5, 6), (6, 7), (7,), (5, 7))
    t = graph.Tape(backend())
    t.dense(t.const(x, x.shape), t.param(w0, w0.shape), t.param(b0, b0.shape), relu_follows=True)      # call 0
    carried = _carried(graph.Tape(backend()), v, 0)
    np.testing.assert_array_equal(t.relu(carried).value, np.maximum(v, 0))


@pytest.mark.parametrize("backend", BACKENDS)
def test_carried_scores_take_no_other_calls_scale(backend):
    q, s, v, w = _arrays((2, 3, 4), (2, 2, 3, 3), (2, 3, 4), (4, 5))
    grads = []
    for number in (0, None):
        t = graph.Tape(backend())
        k = t.param(q, q.shape)
        scores = _carried(graph.Tape(backend()), s, number) if number is not None else t.param(s, s.shape)
        t.head_scores(k, k, 2, 0.5, None, 0.0, True)      # call 0, which nothing reads
        val = t.param(v, v.shape)
        t.backward(_loss(t, t.matmul(t.reshape(t.head_context(scores, val, 2), (-1, 4)), t.param(w, w.shape))))
        grads.append([np.array(u.grad) for u in (scores, val)])
    for a, b in zip(*grads):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("backend", BACKENDS)
def test_a_carried_values_gradient_is_the_callers_after_the_sweep(backend):
    v, w0 = _arrays((5, 7), (7, 4))
    carried = _carried(graph.Tape(backend()), v, 0)
    t = graph.Tape(backend())
    t.backward(_loss(t, t.matmul(carried, t.param(w0, w0.shape))))
    kept, before = carried.grad, np.array(carried.grad)
    t.backward(_loss(t, t.matmul(carried, t.param(w0, w0.shape))))
    np.testing.assert_array_equal(kept, before)
    np.testing.assert_array_equal(carried.grad, before + before)

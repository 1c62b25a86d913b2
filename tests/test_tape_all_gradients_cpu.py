"""Operators that stand for several nodes give every input the gradient that the nodes give it, or refuse it."""
import numpy as np
import pytest

from oracle_backend import OracleBackend, WithMore
from tsplit_amd import graph


@pytest.mark.parametrize("backend", [OracleBackend, WithMore])
@pytest.mark.parametrize("learned", [(True, True), (False, True), (True, False)])
def test_embedding_and_positions_both_get_their_gradients(backend, learned):
    rng = np.random.RandomState(5)
    ids = np.array([[0, 2, 1], [4, 0, 2]], np.float32)
    table, positions, w = [rng.normal(size=s).astype(np.float32) for s in ((5, 4), (2, 3, 4), (4, 3))]
    grads = []
    for nodes in (False, True):
        t = graph.Tape(backend())
        tab, pos = [(t.param if yes else t.const)(a, a.shape) for a, yes in zip((table, positions), learned)]
        i = t.const(ids, ids.shape)
        if nodes:
            cond = t.broadcast_like(t.reshape(i, (2, 3, 1)), (2, 3, 4))
            y = t.add(t.scale(t.embedding(tab, i), 3.0), t.where(cond, pos, t.const(np.zeros((2, 3, 4), np.float32), (2, 3, 4))))
        else:
            y = t.embedding_add(tab, i, 3.0, pos)
        logits = t.matmul(t.reshape(y, (-1, 4)), t.param(w, w.shape))
        t.backward(t.softmax_ce(logits, t.const(np.eye(3, dtype=np.float32)[[0, 1, 2, 0, 1, 2]], (6, 3))))
        grads.append([None if v.grad is None else np.array(v.grad) for v in (tab, pos)])
    for got, want, yes in zip(*grads, learned):
        assert (got is not None) == (want is not None) == yes
        if yes:
            np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("learned", ["x", "initial"])
def test_lstm_cells_refuse_what_they_give_no_gradient(learned):
    class WithCells(WithMore):
        def lstm(self, x, params, initial, steps):
            return np.zeros((x.shape[0], 3), np.float32), None

    t = graph.Tape(WithCells())
    x, initial = [(t.param if name == learned else t.const)(np.zeros(s, np.float32), s) for name, s in (("x", (2, 8)), ("initial", (1,)))]
    params = [t.param(np.zeros(s, np.float32), s) for _ in range(4) for s in ((2, 3), (3, 3), (3,))]
    assert not t.takes_cells(x, initial, 4, 3)
    with pytest.raises(ValueError, match="gradient"):
        t.lstm_cells(x, params, initial, 4)

"""What the gradient of attention scores holds where its scale and its causal selection have not been applied by the product that made it
(scores read by something else than one head_context, or by a stretch run per micro-tensor): the planner's peak has to cover it, and its
values are those of the operators one by one."""
import numpy as np
import pytest

from oracle_backend import OracleBackend, WithMore
from tsplit_amd import graph, tape_budget as tb, workloads


def _transformer(batch):
    cfg = workloads.TransformerConfig(batch, 96, 96, 16, 4, 16, 1, 20, mask_value=-1.0)
    return lambda t, b, c: workloads.transformer(t, b, cfg, c["xs"], c["yi"], c["yo"])


def _another_reader(t, b, c):
    """Causal scores that a product reads: their gradient arrives as a view of the product's."""
    q, k = (t.reshape(t.add(c["x"], b.get(name, c["x"].shape, "one")), (4, 96, 16)) for name in ("q", "k"))
    scores = t.head_scores(q, k, 4, 0.5, None, 0.0, True)
    logits = t.matmul(t.reshape(scores, (4 * 4 * 96, 96)), b.get("w", (96, 2), "one"))
    return t.softmax_ce(logits, c["y"]), logits


def _held(build, shapes, ops, plan, calls=None):
    """Bytes the budgeted executor's own sweeps hold at their worst, on a backend that counts."""
    backend = tb.CountingBackend()
    t = tb.BudgetedTape(backend, plan, ops, None, piece_calls=calls)
    b = workloads.ShapeBinder(t, tb._Zeros())
    loss, _ = build(t, b, {k: t.const(backend.empty(s), s) for k, s in shapes.items()})
    t.backward(loss)
    return backend.counter.peak


ARRAYS = 200 * 256      # every array is counted in whole 256 bytes


def test_the_plan_covers_a_stretch_that_starts_between_causal_scores_and_their_reader():
    batch, pieces = 4, 4
    shapes = {"xs": (batch, 96), "yi": (batch, 96), "yo": (batch, 96)}
    build = _transformer(batch)
    ops, leaves = tb.record(build, shapes)
    calls = tb.trace_pieces(_transformer(batch // pieces), {k: (batch // pieces,) + s[1:] for k, s in shapes.items()})
    start = [i for i, op in enumerate(ops) if op.name == "head_context"][1]
    assert ops[start - 1].name == "head_scores"
    plan, cut = tb.plan_split(ops, leaves, 1 << 30, build, shapes, calls, pieces, split_from=start)
    assert plan.split_from == start and not plan.away and not plan.redo
    assert _held(build, shapes, cut, plan, calls) <= plan.peak_bytes + ARRAYS


def test_the_plan_covers_causal_scores_that_another_operator_reads():
    shapes = {"x": (4 * 96, 16), "y": (4 * 4 * 96, 2)}
    ops, leaves = tb.record(_another_reader, shapes)
    plan = tb.plan(ops, leaves, None)
    assert _held(_another_reader, shapes, ops, plan) <= plan.peak_bytes + ARRAYS


class _InOnePass(WithMore):
    def heads_scale(self, x, scale, causal, shape, out=None):
        y = np.where(np.tril(np.ones(shape[2:], bool)), x, np.float32(0)) if causal else x
        y = np.float32(scale) * y
        if out is None:
            return y
        out[...] = y
        return out


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("own", [False, True])
def test_scores_gradient_in_one_pass_is_that_of_the_operators(causal, own, rng):
    q, k, v = (rng.normal(size=(2, 6, 8)).astype(np.float32) for _ in range(3))
    w = rng.normal(size=(6, 3)).astype(np.float32)
    got = []
    for backend in (OracleBackend(), _InOnePass()):
        t = graph.Tape(backend)
        pq, pk = t.param(q.copy(), q.shape), t.param(k.copy(), k.shape)
        scores = t.head_scores(pq, pk, 2, 0.5, None, 0.0, causal)
        z = t.add(scores, scores) if own else scores      # (a sum of two of its own: an array that may be written)
        logits = t.matmul(t.reshape(z, (24, 6)), t.const(w, w.shape))
        t.backward(t.softmax_ce(logits, t.const(np.eye(3, dtype=np.float32)[np.arange(24) % 3], (24, 3))))
        got.append((pq.grad, pk.grad))
    for a, b in zip(*got):
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-6 * np.abs(a).max())

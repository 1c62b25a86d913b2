"""The sequence of LSTM cells in one call (TSplit_Lstm, TSplit_LstmGradient) against the cells operator by operator in float64:
sizes around the 16 x 16 tiles and the 64 and 128 units whose weights stay in registers, one step, one unit, frames of one value.  Bound: a gradient is a sum of n * steps terms, each
behind at most `steps` cells whose gates are sums of h + d + 1 products; every sum of m terms in fp32 is within
m 2^-24 of its terms' magnitudes, and random signs leave about its square root: 2e-6 of the largest value leaves a factor of four
over the largest seen."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _oracle(x, params, initial, steps, dlast):
    n, d = x.shape[0], x.shape[1] // steps
    W, U, B = params[0::3], params[1::3], params[2::3]
    h = np.full((n, U[0].shape[0]), initial)
    c = h.copy()
    tape = []
    sigmoid = lambda v: 1 / (1 + np.exp(-v))
    for t in range(steps):
        f = x[:, t * d:(t + 1) * d]
        z = [h @ U[g] + f @ W[g] + B[g] for g in range(4)]
        a = [sigmoid(z[0]), sigmoid(z[1]), sigmoid(z[2]), np.tanh(z[3])]
        c2 = c * a[0] + a[1] * a[3]
        tape.append((f, h, c, a, c2))
        h, c = np.tanh(c2) * a[2], c2
    grads = [np.zeros_like(p) for p in params]
    dh, dc = dlast, np.zeros_like(c)
    for f, hb, cb, a, c2 in reversed(tape):
        th = np.tanh(c2)
        dc = dc + dh * a[2] * (1 - th * th)
        dz = [dc * cb * a[0] * (1 - a[0]), dc * a[3] * a[1] * (1 - a[1]), dh * th * a[2] * (1 - a[2]), dc * a[1] * (1 - a[3] ** 2)]
        for g in range(4):
            grads[3 * g] += f.T @ dz[g]
            grads[3 * g + 1] += hb.T @ dz[g]
            grads[3 * g + 2] += dz[g].sum(0)
        dh, dc = sum(dz[g] @ U[g].T for g in range(4)), dc * a[0]
    return h, grads


@pytest.mark.parametrize("n,steps,d,units", [(1, 1, 1, 1), (16, 3, 15, 16), (17, 4, 7, 33), (3, 28, 28, 128), (33, 5, 64, 257), (130, 6, 3, 100), (5, 2, 9, 64), (20, 3, 5, 129)])
def test_cells_against_float64(n, steps, d, units):
    from tsplit_amd import graph, ndarray
    rng = np.random.default_rng(n * 1000 + units)
    x = rng.random((n, steps * d), dtype=np.float32)
    params = [rng.standard_normal(s, dtype=np.float32) * np.float32(0.1 if len(s) == 2 else 0.5) for _ in range(4) for s in ((d, units), (units, units), (units,))]
    initial, dlast = np.float32([0.25]), rng.standard_normal((n, units), dtype=np.float32)
    backend = graph.GpuBackend(ndarray.gpu(0))
    dev = [backend.from_numpy(p) for p in params]
    gx, gi = backend.from_numpy(x), backend.from_numpy(initial)
    last, saved = backend.lstm(gx, dev, gi, steps)
    grads = backend.lstm_grad(backend.from_numpy(dlast), gx, dev, gi, steps, saved)
    ref_last, ref = _oracle(x.astype(np.float64), [p.astype(np.float64) for p in params], 0.25, steps, dlast.astype(np.float64))
    for got, want in [(last, ref_last)] + list(zip(grads, ref)):
        err = np.abs(got.asnumpy() - want).max()
        assert err <= 2e-6 * max(np.abs(want).max(), 1e-3), (got.shape, err, np.abs(want).max())


def test_wrong_sizes_are_refused():
    from tsplit_amd import graph, ndarray
    backend = graph.GpuBackend(ndarray.gpu(0))
    z = lambda *s: backend.from_numpy(np.zeros(s, np.float32))
    params = [z(*s) for _ in range(4) for s in ((3, 8), (8, 8), (8,))]
    backend.lstm(z(2, 6), params, z(1), 2)
    for x, p, steps in ((z(2, 7), params, 2), (z(2, 8), params, 2), (z(2, 6), [params[1]] + params[1:], 2)):
        with pytest.raises(RuntimeError):
            backend.lstm(x, p, z(1), steps)

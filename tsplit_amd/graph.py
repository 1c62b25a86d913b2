"""A small reverse-mode tape over the operator library, for graphs with branches.

The reference builds such graphs with `ad.<op>_op` nodes and differentiates them with
`ad.gradients` (python/athena/gpu_ops/executor.py:160-196); each node's `compute` calls one
`gpu_links` function and its `gradient` names the nodes of the backward pass.  This tape does
the same work eagerly: every method below runs one forward operator and records the calls of
the backward operators the reference's `gradient` would schedule (cited per method).  It
exists so that the residual, multi-branch and attention graphs of the reference's examples
can be run through the C ABI; `trainer.py` remains the harness of the sequential nets.

The arithmetic comes from a backend object.  `GpuBackend` (below) maps every primitive onto
`gpu_links`; the tests plug in a numpy backend with the same methods to check whole graphs.
"""
import numpy as np

from . import gpu_links as L
from . import ndarray


class Var(object):
    """A value on the tape: backend array, shape, accumulated gradient; `node` is the index of the
    operator call that produced it on its tape (-1 for parameters, inputs and constants)."""
    __slots__ = ["value", "shape", "grad", "needs_grad", "name", "node", "home", "own"]

    def __init__(self, value, shape, needs_grad, name=None):
        self.value, self.shape, self.grad, self.needs_grad, self.name = value, tuple(shape), None, needs_grad, name
        self.node = -1
        self.home = None     # the sweep of the tape that `node` counts in
        self.own = False     # during a reverse sweep: `grad` is an array of this value alone, so more may be added in place


class Node(object):
    """One operator call: its output, the closure of its backward operators (None when no input
    needs a gradient), the Vars it read and the Vars its backward closure reads again."""
    __slots__ = ["out", "back", "inputs", "saved", "index", "redo"]

    def __init__(self, out, back, inputs, saved, index, redo=None):
        self.out, self.back, self.inputs, self.saved, self.index = out, back, tuple(inputs), tuple(saved), index
        # for operators that are cheap to run again (one to three passes over HBM): a closure that
        # computes the output once more from the inputs' current values, with the same bits
        self.redo = redo


class _Shape(object):
    """Stands for a value on a backend that computes nothing: the operand's shape."""

    def __init__(self, shape):
        self.shape = shape


def _shaped(value, shape):
    return _Shape(shape) if value is None else value


SELF = object()      # in a `saved` list: the operator's own output


def _prod(shape):
    n = 1
    for s in shape:
        n *= int(s)
    return n


def conv_out(size, k, pad, stride):
    return (size + 2 * pad - k) // stride + 1


class GpuBackend(object):
    """Primitives on device arrays, one `gpu_links` call each (plus the output allocation)."""

    fuses_pairs = True   # bn_relu has an exact form
    L = L        # the links module; a subclass that only counts memory puts a stand-in here

    def __init__(self, ctx=None, stream=None):
        self.ctx = ctx or ndarray.gpu(0)
        self.stream = stream

    # ---- batch micro-tensors
    def piece(self, x, pieces, index):
        """Rows [index * n / pieces, (index + 1) * n / pieces) of x as a zero-copy view
        (DLArraySliceForMicroTensor along the batch)."""
        return ndarray.slice_for_micro_tensor(x, index, pieces)

    def assign(self, dst, src):
        """dst <- src on the compute stream (dst is usually a micro-tensor view)."""
        src.copyto(dst, self.stream)

    # ---- storage
    def from_numpy(self, a):
        return ndarray.array(np.ascontiguousarray(a, dtype=np.float32), self.ctx)

    def to_numpy(self, x):
        return x.asnumpy()

    def empty(self, shape):
        return ndarray.empty(shape, self.ctx)

    def reshape(self, x, shape):
        out = self.empty(shape)
        self.L.array_reshape(x, out, self.stream)
        return out

    def view(self, x, shape):
        """x under another shape, without a copy."""
        return ndarray.view(x, shape)

    # ---- contractions
    def conv2d(self, x, w, xs, ws, ph, pw, s):
        y = self.empty((xs[0], ws[0], conv_out(xs[2], ws[2], ph, s), conv_out(xs[3], ws[3], pw, s)))
        L.CuDNN_conv2d(x, w, y, ph, pw, s, self.stream)
        return y

    def conv2d_grad_data(self, w, dy, xs, ph, pw, s):
        dx = self.empty(xs)
        L.CuDNN_conv2d_gradient_of_data(w, dy, dx, ph, pw, s, self.stream)
        return dx

    def conv2d_grad_data_add(self, w, dy, xs, ph, pw, s, addend, out=None):
        """conv2d_grad_data + addend, into `out` (it may be the addend) or a new array."""
        dx = self.empty(xs) if out is None else out
        L.conv2d_gradient_of_data_add(w, dy, addend, dx, ph, pw, s, self.stream)
        return dx

    def conv2d_grad_filter(self, x, dy, ws, ph, pw, s):
        dw = self.empty(ws)
        L.CuDNN_conv2d_gradient_of_filter(x, dy, dw, ph, pw, s, self.stream)
        return dw

    def matmul(self, a, ta, b, tb, out_shape):
        c = self.empty(out_shape)
        self.L.matrix_multiply(a, ta, b, tb, c, self.stream)
        return c

    def batch_matmul(self, a, ta, b, tb, out_shape):
        c = self.empty(out_shape)
        self.L.batch_matrix_multiply(a, ta, b, tb, c, self.stream)
        return c

    def matmul_add(self, a, ta, b, tb, out_shape, bias=None, addend=None, relu=False, out=None, gate=None):
        """-> (op(a) op(b) + bias + addend, its Relu or None) in one call; arrays of more axes are matrices of the last one's columns.
        out: the array to write (it may be the addend), or None for a new one.  gate: the input of a Relu that the result, its
        gradient, is taken through."""
        c = self.empty(out_shape) if out is None else out
        r = self.empty(out_shape) if relu else None
        self.L.matrix_multiply_add(a, ta, b, tb, c, bias, addend, r, self.stream, gate)
        return c, r

    def matmul_sums(self, a, b, out_shape, sums_shape):
        """-> (a' b, the sums of b's columns); arrays of more axes are matrices of the last one's columns."""
        c, sums = self.empty(out_shape), self.empty(sums_shape)
        self.L.matrix_multiply_sums(a, b, c, sums, self.stream)
        return c, sums

    def heads_matmul(self, a, ta, b, tb, out_shape, heads, alpha=1.0, mask=None, mask_value=0.0, causal=False, fill=0.0, addend=None):
        """Products per sample and head (gpu_links.heads_matrix_multiply)."""
        c = self.empty(out_shape)
        self.L.heads_matrix_multiply(a, ta, b, tb, c, heads, alpha, mask, mask_value, causal, fill, addend, self.stream)
        return c

    def heads_scale(self, x, scale, causal, shape, out=None):
        """scale * x, 0 right of the diagonals with `causal`.  out: the array to write (it may be x), or None for a new one."""
        out = self.empty(shape) if out is None else out
        self.L.heads_scale(x, scale, causal, out, self.stream)
        return out

    # ---- normalisation, activations, pooling
    def bn(self, x, gamma, beta, xs, eps):
        y = self.empty(xs)
        self.L.CuDNN_Batch_Normalization(x, gamma, beta, y, None, None, 0.99, eps, self.stream)
        return y

    def bn_grad(self, dy, x, gamma, xs, eps):
        dx, dg, db = self.empty(xs), self.empty((1, xs[1], 1, 1)), self.empty((1, xs[1], 1, 1))
        self.L.CuDNN_Batch_Normalization_gradient(dy, x, gamma, dx, dg, db, None, None, eps, self.stream)
        return dx, dg, db

    def bn_relu(self, x, gamma, beta, xs, eps, exact=False):
        """-> (relu(bn(x)), saved mean, saved inverse deviation): one call, the BatchNorm output is never written.  exact: the statistics
        are saved as doubles, and the pair has the bits of bn and relu."""
        saved = (xs[1], 2) if exact else (1, xs[1], 1, 1)
        y, mean, istd = self.empty(xs), self.empty(saved), self.empty(saved)
        self.L.batch_norm_relu(x, gamma, beta, y, mean, istd, eps, stream=self.stream)
        return y, mean, istd

    def bn_relu_add(self, x, gamma, beta, addend, xs, eps, exact=False):
        """bn_relu with relu(bn(x)) + addend in the place of relu(bn(x))."""
        saved = (xs[1], 2) if exact else (1, xs[1], 1, 1)
        y, mean, istd = self.empty(xs), self.empty(saved), self.empty(saved)
        self.L.batch_norm_relu_add(x, gamma, beta, addend, y, mean, istd, eps, stream=self.stream)
        return y, mean, istd

    def bn_relu_grad(self, dy, x, gamma, beta, mean, istd, xs, eps):
        dx, dg, db = self.empty(xs), self.empty((1, xs[1], 1, 1)), self.empty((1, xs[1], 1, 1))
        self.L.batch_norm_relu_gradient(dy, x, gamma, beta, dx, dg, db, mean, istd, eps, stream=self.stream)
        return dx, dg, db

    def relu(self, x, shape):
        y = self.empty(shape)
        self.L.relu(x, y, self.stream)
        return y

    def relu_grad(self, x, dy, shape):
        dx = self.empty(shape)
        self.L.relu_gradient(x, dy, dx, self.stream)
        return dx

    def max_pool(self, x, xs, k, pad, s):
        y = self.empty((xs[0], xs[1], conv_out(xs[2], k, pad, s), conv_out(xs[3], k, pad, s)))
        L.CuDNN_max_pooling2d(x, k, k, y, pad, s, self.stream)
        return y

    def max_pool_grad(self, x, y, dy, xs, k, pad, s):
        dx = self.empty(xs)
        L.CuDNN_max_pooling2d_gradient(y, dy, x, k, k, dx, pad, s, self.stream)
        return dx

    def avg_pool(self, x, xs, k, pad, s):
        y = self.empty((xs[0], xs[1], conv_out(xs[2], k, pad, s), conv_out(xs[3], k, pad, s)))
        L.CuDNN_average_pooling2d(x, k, k, y, pad, s, self.stream)
        return y

    def avg_pool_grad(self, x, y, dy, xs, k, pad, s):
        dx = self.empty(xs)
        L.CuDNN_average_pooling2d_gradient(y, dy, x, k, k, dx, pad, s, self.stream)
        return dx

    # ---- elementwise, broadcast, reduce, layout
    def add(self, a, b, shape):
        c = self.empty(shape)
        self.L.matrix_elementwise_add(a, b, c, self.stream)
        return c

    def add_to(self, a, b):
        """a += b."""
        self.L.matrix_elementwise_add(a, b, a, self.stream)

    def mul_const(self, a, c, shape):
        out = self.empty(shape)
        self.L.matrix_elementwise_multiply_by_const(a, c, out, self.stream)
        return out

    def add_const(self, a, c, shape):
        out = self.empty(shape)
        self.L.matrix_elementwise_add_by_const(a, c, out, self.stream)
        return out

    def mul(self, a, b, shape):
        out = self.empty(shape)
        self.L.matrix_elementwise_multiply(a, b, out, self.stream)
        return out

    def sigmoid(self, x, shape):
        out = self.empty(shape)
        self.L.sigmoid(x, out, self.stream)
        return out

    def tanh(self, x, shape):
        out = self.empty(shape)
        self.L.tanh(x, out, self.stream)
        return out

    def slice(self, x, begin, out_shape):
        out = self.empty(out_shape)
        self.L.matrix_slice(x, out, begin, self.stream)
        return out

    def slice_grad(self, dy, begin, in_shape):
        out = self.empty(in_shape)
        self.L.matrix_slice_gradient(dy, out, begin, self.stream)
        return out

    def broadcast_shape(self, x, out_shape):
        out = self.empty(out_shape)
        self.L.broadcast_shape(x, out, None, self.stream)
        return out

    def reduce_sum(self, x, axes, out_shape):
        out = self.empty(out_shape)
        self.L.reduce_sum(x, out, axes, self.stream)
        return out

    def broadcast_to(self, x, out_shape):
        out = self.empty(out_shape)
        self.L.broadcast_to(x, out, self.stream)
        return out

    def reduce_sum_axis_zero(self, x, out_shape):
        out = self.empty(out_shape)
        self.L.reduce_sum_axis_zero(x, out, self.stream)
        return out

    def concat(self, a, b, out_shape, axis):
        out = self.empty(out_shape)
        self.L.concat(a, b, out, axis, self.stream)
        return out

    def concat_grad(self, dout, in_shape, axis, idx):
        g = self.empty(in_shape)
        self.L.concat_gradient(dout, g, axis, idx, self.stream)
        return g

    def join(self, parts, out_shape, axis):
        out = self.empty(out_shape)
        self.L.join(parts, out, axis, self.stream)
        return out

    def part(self, whole, shapes, axis):
        out = [self.empty(s) for s in shapes]
        self.L.part(whole, out, axis, self.stream)
        return out

    def transpose(self, x, perm, out_shape):
        out = self.empty(out_shape)
        self.L.matrix_transpose(x, out, perm, self.stream)
        return out

    def where(self, cond, a, b, shape):
        out = self.empty(shape)
        self.L.where(cond, a, b, out, self.stream)
        return out

    def one_hot(self, ids, out_shape):
        out = self.empty(out_shape)
        self.L.one_hot(ids, out, self.stream)
        return out

    def embedding(self, table, ids, out_shape):
        out = self.empty(out_shape)
        self.L.embedding_lookup(table, ids, out, self.stream)
        return out

    def embedding_grad(self, dy, ids, table_shape):
        g = self.empty(table_shape)
        self.L.embedding_lookup_gradient(dy, ids, g, self.stream)
        return g

    def embedding_add(self, table, ids, scale, positions, out_shape):
        out = self.empty(out_shape)
        self.L.embedding_add(table, ids, scale, positions, out, self.stream)
        return out

    def embedding_add_grad(self, dy, ids, scale, table_shape, add_to=None):
        """The gradient of the table, or that added to the array `add_to`."""
        g = self.empty(table_shape) if add_to is None else add_to
        self.L.embedding_add_gradient(dy, ids, scale, g, add_to is not None, self.stream)
        return g

    def lstm(self, x, params, initial, steps):
        """-> (last state [n, units], what lstm_grad reads again)."""
        n, units = x.shape[0], params[1].shape[0]
        depth, padded = self.L.lstm_sizes(x.shape[1] // steps, units)
        saved = [self.empty(s) for s in ((n, steps, depth), (4 * padded * (depth + padded),), (n, steps, 4, padded), (n, steps, units))]
        last = self.empty((n, units))
        self.L.lstm(x, params, initial, steps, *saved, last, self.stream)
        return last, saved

    def lstm_grad(self, dlast, x, params, initial, steps, saved):
        """-> the gradients of `params`."""
        grads = [self.empty(p.shape) for p in params]
        self.L.lstm_gradient(dlast, x, params, initial, steps, *saved, self.empty(saved[2].shape), grads, self.stream)
        return grads

    def zeros(self, shape):
        out = self.empty(shape)
        self.L.array_set(out, 0.0, self.stream)
        return out

    # ---- loss, update
    def softmax_ce(self, logits, labels):
        loss = self.empty((1,))
        self.L.softmax_cross_entropy(logits, labels, loss, self.stream)
        return loss

    def softmax_ce_grad(self, logits, labels, shape, seed=1.0):
        one = self.empty((1,))
        self.L.array_set(one, float(seed), self.stream)
        g = self.empty(shape)
        self.L.softmax_cross_entropy_gradient(logits, labels, one, g, self.stream)
        return g

    def softmax_ce_ids(self, logits, ids, on, off):
        loss = self.empty((1,))
        self.L.softmax_cross_entropy_ids(logits, ids, on, off, loss, self.stream)
        return loss

    def softmax_ce_ids_grad(self, logits, ids, on, off, shape, seed=1.0):
        one = self.empty((1,))
        self.L.array_set(one, float(seed), self.stream)
        g = self.empty(shape)
        self.L.softmax_cross_entropy_ids_gradient(logits, ids, on, off, one, g, self.stream)
        return g

    def sgd(self, p, g, lr):
        self.L.sgd_update(p, g, lr, self.stream)

    def sync(self):
        if self.stream:
            self.stream.sync()
        else:
            ndarray.empty((1,), self.ctx).asnumpy()


def _op(fn):
    """Marks an operator method of Tape: every call goes through Tape._call, so that a tape may log the
    calls of a builder (trace) or put them off and run them per batch micro-tensor (MicroTape)."""
    def call(self, *args, **kwargs):
        return self._call(fn, args, kwargs)
    call.__name__, call.__doc__ = fn.__name__, fn.__doc__
    return call


class Tape(object):
    # the builders' BatchNorm + Relu pairs as one node each (bn_then_relu); off: the reference's two nodes
    fuse_bn_relu = False

    def __init__(self, backend):
        self.b = backend
        self._nodes = []     # every operator call, in order (Node)
        self._sweep = object()   # stands for these calls; the next sweep's are another's
        self._readers = []   # per operator call: how many inputs of later calls its output is
        self._ready = {}     # operator call -> the Relu of its output, where its launch has left that too
        self._leaves = []    # leaves whose gradient arrays are this sweep's
        self._scores = {}    # head_scores call -> (scale, causal)
        self._scaled = set() # head_scores calls whose gradient has arrived with scale and selection applied
        self._gates = {}     # relu call -> its input
        self._gated = set()  # relu calls whose gradient has arrived taken through them
        self._log = None     # with a list here, every operator call is appended as (name, args, kwargs)

    def _call(self, fn, args, kwargs):
        if self._log is not None:
            self._log.append((fn.__name__, args, kwargs))
        return fn(self, *args, **kwargs)

    # ---- leaves
    def param(self, value, shape, name=None):
        return Var(value, shape, True, name)

    def const(self, value, shape, name=None):
        return Var(value, shape, False, name)

    def _out(self, value, shape, inputs, backward, saved=None, redo=None):
        """Registers an operator call.  `saved`: the Vars the backward closure reads (SELF for the
        output itself); by default the inputs.  A closure must read them as `var.value` when it
        runs, so that an executor may move a value off the device in between.  `redo`: see Node."""
        v = Var(value, shape, any(i.needs_grad for i in inputs))
        saved = inputs if saved is None else [v if s is SELF else s for s in saved]
        node = Node(v, backward if v.needs_grad else None, inputs, saved if v.needs_grad else (), len(self._nodes), redo)
        v.node, v.home = node.index, self._sweep
        self._nodes.append(node)
        self._readers.append(0)
        for i in inputs:
            if i.home is v.home:
                self._readers[i.node] += 1
        self._after_forward(node)
        return v

    def _call_of(self, var):
        """The index of the operator call on this tape that produced var; -1 for a leaf, and for a value that was carried here from
        another tape or from before a reverse sweep, whose `node` counts other calls."""
        return var.node if var.home is self._sweep else -1

    # hooks of executors that manage memory (tsplit_amd.tape_budget)
    def _after_forward(self, node):
        pass

    def _before_backward(self, node):
        pass

    def _after_backward(self, node):
        pass

    def _acc(self, var, g, fresh=False):
        """Adds g to var's gradient.  fresh: g is an array that nothing else holds."""
        if not var.needs_grad:
            return
        if var.grad is None:
            var.grad = g
            self._owns(var, fresh)
        elif var.own:
            self.b.add_to(var.grad, g)
        else:
            var.grad = self.b.add(var.grad, g, var.shape)
            self._owns(var, True)

    def _owns(self, var, fresh):
        var.own = fresh and self._can("add_to")
        if var.own and var.home is not self._sweep:
            self._leaves.append(var)      # a leaf's gradient is the caller's once the sweep ends

    # ---- products with something behind them: one call where the backend has it, else the operators one by one
    def _can(self, name):
        return hasattr(type(self.b), name)

    def _seen_as(self, value, shape):
        """An operator's output (or a gradient) under another shape: a view where the backend has views."""
        return (self.b.view if self._can("view") else self.b.reshape)(value, shape)

    def _product(self, a, a_shape, ta, b, b_shape, tb, out_shape, bias=None, addend=None, relu=False):
        """-> (op(a) op(b) + bias + addend, its Relu or None); arrays of more than two axes are matrices of the last one's columns."""
        if self._can("matmul_add"):
            return self.b.matmul_add(a, ta, b, tb, out_shape, bias, addend, relu)
        flat = [_shaped(self.b.reshape(v, sh) if v is not None and sh != whole else v, sh)
                for v, whole, sh in ((v, sh, (_prod(sh[:-1]), sh[-1])) for v, sh in ((a, a_shape), (b, b_shape)))]
        rows = (_prod(out_shape[:-1]), out_shape[-1])
        y = self.b.matmul(flat[0], ta, flat[1], tb, rows)
        if bias is not None:
            y = self.b.add(y, self.b.broadcast_to(bias, rows), rows)
        if len(out_shape) > 2:
            y = self.b.reshape(y, out_shape)
        if addend is not None:
            y = self.b.add(y, addend, out_shape)
        return y, self.b.relu(y, out_shape) if relu else None

    def _acc_product(self, var, a, a_shape, ta, b, b_shape, tb):
        """Adds op(a) op(b) to var's gradient."""
        if not var.needs_grad:
            return
        n = self._call_of(var)
        if n in self._gates and self._readers[n] == 1 and var.grad is None:
            # a Relu's output that goes nowhere else: its gradient behind the product that makes it
            var.grad = self.b.matmul_add(a, ta, b, tb, var.shape, gate=self._gates[n].value)[0]
            self._owns(var, True)
            self._gated.add(n)
        elif var.own:
            self.b.matmul_add(a, ta, b, tb, var.shape, addend=var.grad, out=var.grad)
        else:
            var.grad = self._product(a, a_shape, ta, b, b_shape, tb, var.shape, addend=var.grad)[0]
            self._owns(var, True)

    def _heads_product(self, a, a_shape, ta, b, b_shape, tb, out_shape, heads, alpha=1.0, mask=None, mask_value=0.0, causal=False,
                       fill=0.0, addend=None):
        """For every sample and head alpha * op(a) op(b), + mask_value where mask (a value a column) is 0, `fill` right of the
        diagonal with causal, + addend.  A shape of three axes holds the heads' columns side by side in its rows."""
        # (a matrix one launch cannot address goes the long way: 2^31 bytes, and 128 rows of it)
        reach = all(_prod(sh[1:]) < (1 << 29) and sh[-1] < (1 << 22) for sh in (a_shape, b_shape, out_shape))
        if self._can("heads_matmul") and reach:
            return self.b.heads_matmul(a, ta, b, tb, out_shape, heads, alpha, mask, mask_value, causal, fill, addend)

        def split(v, sh):
            if len(sh) == 4:
                return v, sh
            v = self.b.reshape(v, (sh[0], sh[1], heads, sh[2] // heads))
            sh = (sh[0], heads, sh[1], sh[2] // heads)
            return self.b.transpose(v, [0, 2, 1, 3], sh), sh

        def side(v, sh):
            return _shaped(*split(v, sh))
        n = out_shape[0]
        four = out_shape if len(out_shape) == 4 else (n, heads, out_shape[1], out_shape[2] // heads)
        y = self.b.batch_matmul(side(a, a_shape), ta, side(b, b_shape), tb, four)
        if alpha != 1.0:
            y = self.b.mul_const(y, alpha, four)
        if mask is not None:
            cols = (n, four[3])
            m = self.b.where(mask, self.b.zeros(cols), self.b.add_const(self.b.zeros(cols), mask_value, cols), cols)
            y = self.b.add(y, self.b.broadcast_shape(self.b.reshape(m, (n, 1, 1, four[3])), four), four)
        if causal:
            tril = self.b.broadcast_shape(self.b.from_numpy(np.tril(np.ones(four[2:], np.float32))), four)
            y = self.b.where(tril, y, self.b.add_const(self.b.zeros(four), fill, four), four)
        if len(out_shape) == 3:
            y = self.b.reshape(self.b.transpose(y, [0, 2, 1, 3], (n, four[2], heads, four[3])), out_shape)
        return y if addend is None else self.b.add(y, addend, out_shape)

    # ---- operators (reference gradient rules cited)
    @_op
    def conv2d(self, x, w, ph, pw, stride):
        """gpu_ops/Conv2d.py:100-118 (compute), :120 (gradient: a data-gradient and a filter-gradient node)."""
        y = self.b.conv2d(x.value, w.value, x.shape, w.shape, ph, pw, stride)
        ys = (x.shape[0], w.shape[0], conv_out(x.shape[2], w.shape[2], ph, stride), conv_out(x.shape[3], w.shape[3], pw, stride))

        def back(g):
            if w.needs_grad:
                self._acc(w, self.b.conv2d_grad_filter(x.value, g, w.shape, ph, pw, stride), fresh=True)
            if x.needs_grad and x.grad is not None and self._adds_data_gradient(w.shape, ph, pw, stride):
                x.grad = self.b.conv2d_grad_data_add(w.value, g, x.shape, ph, pw, stride, x.grad, x.grad if x.own else None)
                if not x.own:
                    self._owns(x, True)
            elif x.needs_grad:
                self._acc(x, self.b.conv2d_grad_data(w.value, g, x.shape, ph, pw, stride), fresh=True)
        return self._out(y, ys, [x, w], back, saved=[x, w])

    def _adds_data_gradient(self, ws, ph, pw, stride):
        """Whether a data gradient's launch can add to what is there: filters of one tap (others would be two launches all the same)."""
        return ws[2:] == (1, 1) and not ph and not pw and stride <= 2 and self._ahead and self._can("conv2d_grad_data_add")

    @_op
    def batch_norm(self, x, gamma, beta, eps=0.01):
        """gpu_ops/BatchNorm.py:54-83 (compute), :166-227 (gradient node; statistics recomputed, no
        saved arrays); gamma / beta receive their gradients as in gpu_ops/BatchNorm2.py:104-114."""
        def fwd():
            return self.b.bn(x.value, gamma.value, beta.value, x.shape, eps)

        def back(g):
            dx, dg, db = self.b.bn_grad(g, x.value, gamma.value, x.shape, eps)
            self._acc(x, dx)
            self._acc(gamma, dg)
            self._acc(beta, db)
        return self._out(fwd(), x.shape, [x, gamma, beta], back, saved=[x, gamma], redo=fwd)

    @_op
    def batch_norm_relu(self, x, gamma, beta, eps=0.01, exact=False, residual=None):
        """BatchNorm and the Relu behind it as one node (TSplit_BatchNormRelu / _gradient; the reference's graph
        has two nodes, gpu_ops/BatchNorm.py and gpu_ops/Relu.py): the BatchNorm output is never written, and
        the gradient reads the BatchNorm's input, the parameters and the two saved statistics vectors.
        exact (device backends): with the bits of the two nodes.  residual (likewise, and not on a tape that accounts for every
        value): a Var that is added behind the Relu."""
        stats, form = [None, None], {"exact": True} if exact else {}

        def fwd():
            if residual is not None:
                r = self.b.bn_relu_add(x.value, gamma.value, beta.value, residual.value, x.shape, eps, **form)
            else:
                r = self.b.bn_relu(x.value, gamma.value, beta.value, x.shape, eps, **form)
            if r is None:                      # a backend that only records shapes
                return None
            y, stats[0], stats[1] = r
            return y

        def back(g):
            if residual is not None:
                self._acc(residual, g)
            dx, dg, db = self.b.bn_relu_grad(g, x.value, gamma.value, beta.value, stats[0], stats[1], x.shape, eps)
            self._acc(x, dx)
            self._acc(gamma, dg)
            self._acc(beta, db)
        inputs = [x, gamma, beta] + ([] if residual is None else [residual])
        return self._out(fwd(), x.shape, inputs, back, saved=[x, gamma, beta], redo=fwd)

    def bn_relu_then_add(self, x, gamma, beta, residual, eps=0.01):
        """bn_then_relu and the sum with `residual` behind it; where that is one node, the sum is part of it."""
        if self._ahead and self._can("bn_relu_add") and (self.fuse_bn_relu or getattr(type(self.b), "fuses_pairs", False)):
            assert residual.shape == x.shape, (residual.shape, x.shape)
            return self.batch_norm_relu(x, gamma, beta, eps, not self.fuse_bn_relu, residual)
        return self.add(self.bn_then_relu(x, gamma, beta, eps), residual)

    def bn_then_relu(self, x, gamma, beta, eps=0.01):
        """The pair as the reference's graph has it (two nodes), or as one node: when the tape was asked to fuse, and on the device
        on a tape that accounts for no value, where nothing can read the BatchNorm's output (the same values from two passes of
        five less going forward, three of eight less going back)."""
        if self.fuse_bn_relu:
            return self.batch_norm_relu(x, gamma, beta, eps)
        if self._ahead and getattr(type(self.b), "fuses_pairs", False):
            return self.batch_norm_relu(x, gamma, beta, eps, exact=True)
        return self.relu(self.batch_norm(x, gamma, beta, eps))

    @_op
    def relu(self, x):
        """gpu_ops/Relu.py:51,117."""
        def fwd():
            return self.b.relu(x.value, x.shape)
        y = self._ready.pop(self._call_of(x), None)
        out = None

        def back(g):
            if out.node in self._gated:
                self._acc(x, g, fresh=True)
            else:
                self._acc(x, self.b.relu_grad(x.value, g, x.shape))
        out = self._out(fwd() if y is None else y, x.shape, [x], back, redo=fwd)
        if out.node >= 0 and self._ahead and self._can("matmul_add"):
            self._gates[out.node] = x
        return out

    @_op
    def max_pool(self, x, k, pad, stride):
        """gpu_ops/MaxPool.py:119 (compute), :146 (gradient)."""
        y = self.b.max_pool(x.value, x.shape, k, pad, stride)
        ys = (x.shape[0], x.shape[1], conv_out(x.shape[2], k, pad, stride), conv_out(x.shape[3], k, pad, stride))
        out = None
        out = self._out(y, ys, [x], lambda g: self._acc(x, self.b.max_pool_grad(x.value, out.value, g, x.shape, k, pad, stride)),
                        saved=[x, SELF])
        return out

    @_op
    def avg_pool(self, x, k, pad, stride):
        """gpu_ops/AvgPool.py:78 (compute), :103-104 (gradient)."""
        y = self.b.avg_pool(x.value, x.shape, k, pad, stride)
        ys = (x.shape[0], x.shape[1], conv_out(x.shape[2], k, pad, stride), conv_out(x.shape[3], k, pad, stride))
        out = None
        out = self._out(y, ys, [x], lambda g: self._acc(x, self.b.avg_pool_grad(x.value, out.value, g, x.shape, k, pad, stride)),
                        saved=[x, SELF])
        return out

    @_op
    def add(self, a, b):
        """gpu_ops/AddElewise.py:54 (compute), :95 (gradient: both inputs receive the output gradient)."""
        assert a.shape == b.shape, (a.shape, b.shape)

        def fwd():
            return self.b.add(a.value, b.value, a.shape)

        def back(g):
            self._acc(a, g)
            self._acc(b, g)
        return self._out(fwd(), a.shape, [a, b], back, saved=[], redo=fwd)

    @_op
    def scale(self, a, c):
        """gpu_ops/MultiplyConst.py:45 (compute), :63 (gradient: the output gradient times the constant)."""
        def fwd():
            return self.b.mul_const(a.value, c, a.shape)
        return self._out(fwd(), a.shape, [a], lambda g: self._acc(a, self.b.mul_const(g, c, a.shape)), saved=[], redo=fwd)

    @_op
    def shift(self, a, c):
        def fwd():
            return self.b.add_const(a.value, c, a.shape)
        return self._out(fwd(), a.shape, [a], lambda g: self._acc(a, g), saved=[], redo=fwd)

    @_op
    def mul(self, a, b):
        """gpu_ops/MultiplyElewise.py (compute; gradient: each input receives the other times the
        output gradient)."""
        assert a.shape == b.shape, (a.shape, b.shape)

        def fwd():
            return self.b.mul(a.value, b.value, a.shape)

        def back(g):
            self._acc(a, self.b.mul(b.value, g, a.shape))
            self._acc(b, self.b.mul(a.value, g, a.shape))
        return self._out(fwd(), a.shape, [a, b], back, redo=fwd)

    @_op
    def sigmoid(self, x):
        """gpu_ops/Sigmoid.py:58-61: gradient s * (1 + -1 * s) * g, built from the same elementwise
        operators the reference's gradient graph uses."""
        y = self.b.sigmoid(x.value, x.shape)
        out = None

        def back(g):
            one_minus = self.b.add_const(self.b.mul_const(out.value, -1.0, x.shape), 1.0, x.shape)
            self._acc(x, self.b.mul(self.b.mul(out.value, one_minus, x.shape), g, x.shape))
        out = self._out(y, x.shape, [x], back, saved=[SELF])
        return out

    @_op
    def tanh(self, x):
        """gpu_ops/Tanh.py:59-61: gradient (1 + (-1 * t) * t) * g."""
        y = self.b.tanh(x.value, x.shape)
        out = None

        def back(g):
            d = self.b.add_const(self.b.mul(self.b.mul_const(out.value, -1.0, x.shape), out.value, x.shape), 1.0, x.shape)
            self._acc(x, self.b.mul(d, g, x.shape))
        out = self._out(y, x.shape, [x], back, saved=[SELF])
        return out

    @_op
    def slice(self, x, begin, size):
        """gpu_ops/Slice.py:47-81: tf.slice semantics, a size of -1 runs to the end; the gradient
        writes the output gradient into zeros at `begin` (:126-141)."""
        begin = tuple(int(v) for v in begin)
        shape = tuple(int(x.shape[d] - begin[d] if n == -1 else n) for d, n in enumerate(size))
        y = self.b.slice(x.value, begin, shape)
        return self._out(y, shape, [x], lambda g: self._acc(x, self.b.slice_grad(g, begin, x.shape)), saved=[])

    @_op
    def reshape(self, a, shape):
        """gpu_ops/Reshape.py:42 (compute: a copy there), :61 (gradient: reshaped back)."""
        shape = list(shape)
        if -1 in shape:
            known = _prod([s for s in shape if s != -1])
            shape[shape.index(-1)] = _prod(a.shape) // known
        shape = tuple(shape)
        # this tape's outputs and gradients are written once, so another shape of one is a view of it; parameters, inputs and what
        # other tapes left are the caller's to write again, so they are copied
        made_here = self._call_of(a) >= 0

        def fwd():
            return self._seen_as(a.value, shape) if made_here else self.b.reshape(a.value, shape)
        return self._out(fwd(), shape, [a], lambda g: self._acc(a, self._seen_as(g, a.shape)), saved=[], redo=fwd)

    @_op
    def concat(self, a, b, axis):
        """gpu_ops/Concat.py:47-60 (compute), :65 (gradient: two concat_gradient nodes, idx 0 and 1)."""
        shape = list(a.shape)
        shape[axis] += b.shape[axis]
        shape = tuple(shape)
        def fwd():
            return self.b.concat(a.value, b.value, shape, axis)
        y = fwd()

        def back(g):
            if a.needs_grad:
                self._acc(a, self.b.concat_grad(g, a.shape, axis, 0))
            if b.needs_grad:
                self._acc(b, self.b.concat_grad(g, b.shape, axis, 1))
        return self._out(y, shape, [a, b], back, saved=[], redo=fwd)

    def concat_all(self, parts, axis):
        """The parts one behind the other: one node where the backend joins any number and the whole is within one launch's reach, else
        chained concats of two (examples/imagenet_inceptionv4.py concatenates in pairs)."""
        values = sum(_prod(p.shape) for p in parts)
        if 2 < len(parts) <= 8 and self._ahead and self._can("join") and values < (1 << 32) - (1 << 10):
            return self.join(parts, axis)
        x = parts[0]
        for p in parts[1:]:
            x = self.concat(x, p, axis)
        return x

    @_op
    def join(self, parts, axis):
        """The parts one behind the other along `axis`; the gradient is cut up again."""
        shape = list(parts[0].shape)
        shape[axis] = sum(p.shape[axis] for p in parts)
        shape = tuple(shape)

        def fwd():
            return self.b.join([p.value for p in parts], shape, axis)

        def back(g):
            for p, gp in zip(parts, self.b.part(g, [p.shape for p in parts], axis)):
                if p.needs_grad:
                    self._acc(p, gp, fresh=True)
        return self._out(fwd(), shape, list(parts), back, saved=[], redo=fwd)

    @_op
    def matmul(self, a, b, trans_a=False, trans_b=False):
        """gpu_ops/MatrixMult.py:57-86 (compute), :95-124 (gradient)."""
        m = a.shape[1] if trans_a else a.shape[0]
        n = b.shape[0] if trans_b else b.shape[1]
        y = self.b.matmul(a.value, trans_a, b.value, trans_b, (m, n))

        def back(g):
            gs = (m, n)
            if not trans_a:
                self._acc_product(a, g, gs, False, b.value, b.shape, not trans_b)
            else:
                self._acc_product(a, b.value, b.shape, trans_b, g, gs, True)
            if not trans_b:
                self._acc_product(b, a.value, a.shape, not trans_a, g, gs, False)
            else:
                self._acc_product(b, g, gs, True, a.value, a.shape, trans_a)
        return self._out(y, (m, n), [a, b], back)

    # whether a launch may leave a later operator's output as well (not on a tape that accounts for every value where it is made)
    _ahead = True

    @_op
    def dense(self, x, w, bias=None, residual=None, relu_follows=False):
        """x [..., fan_in] w [fan_in, fan_out] + bias + residual as one node; the reference's graph has MatrixMult, Broadcast and
        AddElewise nodes (examples/transformer.py:56-69, :174-181).  relu_follows: relu() of the output comes next, and the launch may
        leave that too."""
        ys = tuple(x.shape[:-1]) + (w.shape[1],)
        relu = relu_follows and self._ahead and self._can("matmul_add")
        y, r = self._product(x.value, x.shape, False, w.value, w.shape, False, ys, bias.value if bias is not None else None,
                             residual.value if residual is not None else None, relu)

        def back(g):
            if residual is not None:
                self._acc(residual, g)
            both = bias is not None and bias.needs_grad and w.needs_grad and bias.grad is None and w.grad is None and self._can("matmul_sums")
            if both:
                w.grad, bias.grad = self.b.matmul_sums(x.value, g, w.shape, bias.shape)
                self._owns(w, True)
                self._owns(bias, True)
            else:
                self._acc_product(w, x.value, x.shape, True, g, ys, False)
            if bias is not None and bias.needs_grad and not both:
                rows = self._seen_as(g, (_prod(ys[:-1]), ys[-1])) if len(ys) > 2 else g
                self._acc(bias, self.b.reduce_sum_axis_zero(rows, bias.shape), fresh=True)
            self._acc_product(x, g, ys, False, w.value, w.shape, True)
        out = self._out(y, ys, [v for v in (x, w, bias, residual) if v is not None], back, saved=[x, w])
        if r is not None:
            self._ready[out.node] = r
        return out

    @_op
    def head_scores(self, q, k, heads, scale, mask_ids=None, mask_value=0.0, causal=False):
        """Attention scores [N, heads, tq, tk] of projections [N, t, heads * dh] whose heads lie side by side: scale * q k', mask_value
        added in the columns of padding (ids of 0), mask_value in place of what lies in the future.  The reference's graph spells
        this out (examples/transformer.py:93-160: reshape, transpose, BatchMatrixMultiply, MultiplyConst, Where, Broadcast, Add)."""
        n, tq, tk = q.shape[0], q.shape[1], k.shape[1]
        ys = (n, heads, tq, tk)
        y = self._heads_product(q.value, q.shape, False, k.value, k.shape, True, ys, heads, scale,
                                mask_ids.value if mask_ids is not None else None, mask_value, causal, mask_value)
        out = None

        def back(g):
            if out.node in self._scaled:
                self._scaled.discard(out.node)
            elif self._can("heads_scale"):      # (a gradient that nothing else holds in place: a planner counts no other array there)
                g = self.b.heads_scale(g, scale, causal, ys, g if out.own else None)
            else:
                if causal:
                    tril = self.b.broadcast_shape(self.b.from_numpy(np.tril(np.ones((tq, tk), np.float32))), ys)
                    g = self.b.where(tril, g, self.b.zeros(ys), ys)
                g = self.b.mul_const(g, scale, ys)
            for var, ta, other in ((q, False, k), (k, True, q)):
                if var.needs_grad:
                    var.grad = self._heads_product(g, ys, ta, other.value, other.shape, False, var.shape, heads, addend=var.grad)
                    self._owns(var, True)
        out = self._out(y, ys, [v for v in (q, k, mask_ids) if v is not None], back, saved=[q, k])
        if out.node >= 0:
            self._scores[out.node] = (scale, causal)
        return out

    @_op
    def head_context(self, scores, v, heads, residual=None):
        """scores [N, heads, tq, tk] times v [N, tk, heads * dh], the heads side by side again: [N, tq, heads * dh], + residual
        (examples/transformer.py:161-171)."""
        ys = (v.shape[0], scores.shape[2], v.shape[2])
        y = self._heads_product(scores.value, scores.shape, False, v.value, v.shape, False, ys, heads,
                                addend=residual.value if residual is not None else None)

        def back(g):
            if residual is not None:
                self._acc(residual, g)
            if v.needs_grad:
                v.grad = self._heads_product(scores.value, scores.shape, True, g, ys, False, v.shape, heads, addend=v.grad)
                self._owns(v, True)
            if scores.needs_grad:
                # scores that go nowhere else take their scale and their selection behind this product
                n = self._call_of(scores)
                alone = n in self._scores and self._readers[n] == 1 and scores.grad is None
                scale, causal = self._scores[n] if alone else (1.0, False)
                scores.grad = self._heads_product(g, ys, False, v.value, v.shape, True, scores.shape, heads, scale, causal=causal,
                                                  addend=scores.grad)
                self._owns(scores, True)
                if alone:
                    self._scaled.add(n)
        return self._out(y, ys, [u for u in (scores, v, residual) if u is not None], back, saved=[scores, v])

    def takes_cells(self, x, initial, steps, units):
        """Whether lstm_cells() is there for these operands: the data get no gradient, every value of x is a frame's, and the sizes
        are those TSplit_Lstm addresses."""
        return (self._ahead and self._can("lstm") and not x.needs_grad and not initial.needs_grad and initial.shape == (1,)
                and len(x.shape) == 2 and 0 < x.shape[0] < 1 << 20 and x.shape[1] % steps == 0 and 0 < x.shape[1] // steps < 1 << 24
                and x.shape[0] * steps < (1 << 31) - 64 and units < 1 << 20 and (x.shape[0] // 16 + 1) * (units // 16 + 1) < 1 << 30)

    @_op
    def lstm_cells(self, x, params, initial, steps):
        """The last hidden state of `steps` LSTM cells on the frames of x, from a state of one value everywhere; params: W, U and b of
        the forget, input, output and candidate gates.  The reference's graph spells out every cell (examples/LSTM.py:52-84)."""
        if x.needs_grad or initial.needs_grad:
            raise ValueError("lstm_cells gives the frames and the initial state no gradient: spell the cells out (takes_cells)")
        values = [p.value for p in params]
        y, saved = self.b.lstm(x.value, values, initial.value, steps)

        def back(g):
            for p, gp in zip(params, self.b.lstm_grad(g, x.value, values, initial.value, steps, saved)):
                self._acc(p, gp, fresh=True)
        return self._out(y, (x.shape[0], params[1].shape[0]), [x] + list(params) + [initial], back)

    @_op
    def batch_matmul(self, a, b, trans_a=False, trans_b=False):
        """gpu_ops/BatchMatrixMult.py:49-75 (compute), :77 (gradient: the four transpose cases)."""
        lead = a.shape[:-2]
        m = a.shape[-1] if trans_a else a.shape[-2]
        n = b.shape[-2] if trans_b else b.shape[-1]
        ys = tuple(lead) + (m, n)
        y = self.b.batch_matmul(a.value, trans_a, b.value, trans_b, ys)

        def back(g):
            if a.needs_grad:
                if not trans_a:
                    ga = self.b.batch_matmul(g, False, b.value, not trans_b, a.shape)
                else:
                    ga = self.b.batch_matmul(b.value, trans_b, g, True, a.shape)
                self._acc(a, ga)
            if b.needs_grad:
                if not trans_b:
                    gb = self.b.batch_matmul(a.value, not trans_a, g, False, b.shape)
                else:
                    gb = self.b.batch_matmul(g, True, a.value, trans_a, b.shape)
                self._acc(b, gb)
        return self._out(y, ys, [a, b], back)

    @_op
    def add_bias(self, x, bias):
        """x [rows, cols] + broadcast(bias [cols]) (gpu_ops/Broadcast.py:45-59, gradient :65 =
        reduce_sum_axis_zero)."""
        def fwd():
            return self.b.add(x.value, self.b.broadcast_to(bias.value, x.shape), x.shape)

        def back(g):
            self._acc(x, g)
            if bias.needs_grad:
                self._acc(bias, self.b.reduce_sum_axis_zero(g, bias.shape))
        return self._out(fwd(), x.shape, [x, bias], back, saved=[], redo=fwd)

    @_op
    def broadcast_like(self, x, shape):
        """gpu_ops/BroadcastTF.py:46-58 (numpy alignment from the right); gradient = reduce_sum
        over the broadcast axes (gpu_ops/BroadcastShape.py:61)."""
        shape = tuple(shape)

        def fwd():
            return self.b.broadcast_shape(x.value, shape)
        y = fwd()
        diff = len(shape) - len(x.shape)
        axes = [d for d in range(len(shape)) if d < diff or (x.shape[d - diff] == 1 and shape[d] != 1)]

        def back(g):
            if axes:
                self._acc(x, self.b.reduce_sum(g, axes, x.shape))
            else:
                self._acc(x, g)
        return self._out(y, shape, [x], back, saved=[], redo=fwd)

    @_op
    def transpose(self, x, perm):
        """gpu_ops/Transpose.py:44-58 (compute), :60 (gradient: the inverse permutation)."""
        perm = list(perm)
        ys = tuple(x.shape[p] for p in perm)
        def fwd():
            return self.b.transpose(x.value, perm, ys)
        inv = [0] * len(perm)
        for i, p in enumerate(perm):
            inv[p] = i
        return self._out(fwd(), ys, [x], lambda g: self._acc(x, self.b.transpose(g, inv, x.shape)), saved=[], redo=fwd)

    @_op
    def where(self, cond, a, b):
        """gpu_ops/Where.py:41-48 (compute), :50-55 (gradient: where(cond, g, 0) and where(cond, 0, g))."""
        def fwd():
            return self.b.where(cond.value, a.value, b.value, a.shape)
        y = fwd()

        def back(g):
            z = self.b.zeros(a.shape)
            if a.needs_grad:
                self._acc(a, self.b.where(cond.value, g, z, a.shape))
            if b.needs_grad:
                self._acc(b, self.b.where(cond.value, z, g, a.shape))
        return self._out(y, a.shape, [cond, a, b], back, saved=[cond], redo=fwd)

    @_op
    def one_hot(self, ids, classes):
        """gpu_ops/OneHot.py:44-46; no gradient."""
        ys = tuple(ids.shape) + (classes,)
        return self._out(self.b.one_hot(ids.value, ys), ys, [ids], None, saved=[])

    @_op
    def embedding(self, table, ids):
        """gpu_ops/EmbeddingLookUp.py:41-42, gradient :48-49."""
        ys = tuple(ids.shape) + (table.shape[1],)
        y = self.b.embedding(table.value, ids.value, ys)
        return self._out(y, ys, [table, ids], lambda g: self._acc(table, self.b.embedding_grad(g, ids.value, table.shape)),
                         saved=[ids])

    @_op
    def embedding_add(self, table, ids, scale, positions):
        """scale * table[id] + positions, those left out where the id is 0 (examples/transformer.py:189-232 node by node)."""
        ys = tuple(ids.shape) + (table.shape[1],)
        fused = self._can("embedding_add")

        def where_an_id(v):
            cond = self.b.broadcast_shape(self.b.reshape(ids.value, tuple(ids.shape) + (1,)), ys)
            return self.b.where(cond, v, self.b.zeros(ys), ys)
        if fused:
            y = self.b.embedding_add(table.value, ids.value, scale, positions.value, ys)
        else:
            y = self.b.add(self.b.mul_const(self.b.embedding(table.value, ids.value, ys), scale, ys), where_an_id(positions.value), ys)

        def back(g):
            if positions.needs_grad:
                self._acc(positions, where_an_id(g), fresh=True)
            if not table.needs_grad:
                return
            if fused and table.own:
                self.b.embedding_add_grad(g, ids.value, scale, table.shape, table.grad)
            elif fused:
                self._acc(table, self.b.embedding_add_grad(g, ids.value, scale, table.shape), fresh=True)
            else:
                self._acc(table, self.b.embedding_grad(self.b.mul_const(g, scale, ys), ids.value, table.shape))
        return self._out(y, ys, [table, ids, positions], back, saved=[ids])

    @_op
    def softmax_ce(self, logits, labels, weight=1.0, smoothing=None):
        """gpu_ops/SoftmaxCrossEntropy.py:46-67 (compute), :73 and :134-135 (gradient) with an adjoint of one.
        `weight` scales the loss and, through the gradient operator's adjoint argument, its gradient: the
        share of a batch micro-tensor in the mean over the whole batch.  With `smoothing` the labels are one class
        index a row (smoothed_softmax_ce)."""
        assert len(logits.shape) == 2
        if smoothing is None:
            forward, gradient, lab = self.b.softmax_ce, self.b.softmax_ce_grad, lambda: (labels.value,)
        else:
            on, off = 1.0 - smoothing, smoothing / logits.shape[1]
            forward, gradient, lab = self.b.softmax_ce_ids, self.b.softmax_ce_ids_grad, lambda: (labels.value, on, off)
        loss = forward(logits.value, *lab())
        if weight != 1.0:
            loss = self.b.mul_const(loss, weight, (1,))

        def back(g):
            if weight != 1.0:
                self._acc(logits, gradient(logits.value, *lab(), logits.shape, weight))
            else:
                self._acc(logits, gradient(logits.value, *lab(), logits.shape))
        return self._out(loss, (1,), [logits, labels], back, saved=[logits, labels])

    def smoothed_softmax_ce(self, logits, ids, smoothing):
        """The loss for labels (1 - smoothing) * one-hot(ids) + smoothing / classes (examples/transformer.py:184-186).  The label
        array is written, by the reference's three nodes, only where a planner accounts for it or the backend has no other loss."""
        if self._ahead and self._can("softmax_ce_ids"):
            return self.softmax_ce(logits, ids, smoothing=smoothing)
        classes = logits.shape[1]
        labels = self.shift(self.scale(self.one_hot(ids, classes), 1.0 - smoothing), smoothing / classes)
        return self.softmax_ce(logits, labels)

    # ---- reverse sweep
    def backward(self, loss):
        """Runs the recorded backward operators in reverse order; the loss adjoint is one
        (gpu_ops/executor.py:175), folded into softmax_ce's gradient."""
        if loss.grad is None:
            loss.grad = True
        for node in reversed(self._nodes):
            v = node.out
            self._before_backward(node)
            if node.back is not None and v.grad is not None:
                node.back(v.grad)
                if v is not loss:
                    v.grad, v.own = None, False      # interior gradients are dropped as soon as they are consumed
            self._after_backward(node)
        self._release_leaves()
        self._nodes, self._readers, self._sweep = [], [], object()
        self._ready, self._scores, self._scaled, self._gates, self._gated = {}, {}, set(), {}, set()


    def _release_leaves(self):
        for v in self._leaves:
            v.own = False
        self._leaves = []


# ---------------------------------------------------------------- batch micro-tensors on the tape
class _ShapeOnly(object):
    """Backend that computes nothing: every primitive returns None."""

    def __getattr__(self, name):
        return lambda *a, **k: None


def trace(build, inputs, binder_for, fuse_bn_relu=False):
    """Runs `build(tape, binder, cache)` on shapes only and returns the operator calls it makes, in
    order: a list of (method name, args, kwargs), Var arguments being the Vars of that run.
    inputs: name -> shape; binder_for(tape) -> a binder whose parameters need no values."""
    t = Tape(_ShapeOnly())
    t.fuse_bn_relu = fuse_bn_relu
    t._log = []
    cache = {k: t.const(None, shape) for k, shape in inputs.items()}
    build(t, binder_for(t), cache)
    return t._log


# operators whose result for one sample depends on the other samples of the batch: a graph that
# contains one cannot run that part per micro-tensor
COUPLES_SAMPLES = frozenset(["batch_norm", "batch_norm_relu"])


class _PieceTape(Tape):
    """The tape one micro-tensor of a put-off stretch runs on.  It drops a value once its last reader has
    run (`drop_after_forward[t]`: values read by no backward operator whose last forward reader is operator
    t; `drop_after_backward[j]`: values whose last backward reader is operator j) and tells its owner after
    every operator."""

    _ahead = False

    def __init__(self, backend, owner, drop_after_forward=None, drop_after_backward=None):
        Tape.__init__(self, backend)
        self._owner = owner
        self._drop_f, self._drop_b = drop_after_forward or {}, drop_after_backward or {}

    def _after_forward(self, node):
        for m in self._drop_f.get(node.index, ()):
            self._nodes[m].out.value = None
        self._owner._inside_piece()

    def _after_backward(self, node):
        for m in self._drop_b.get(node.index, ()):
            self._nodes[m].out.value = None
        self._owner._inside_piece()

    def _release_leaves(self):
        pass                 # the next piece adds to the same arrays


def _last_readers(nodes):
    """For the operators of one tape: -> (drop_after_forward, drop_after_backward) as _PieceTape takes them.
    The last operator's output (the loss) is never dropped."""
    n = len(nodes)
    last_fwd, need = list(range(n)), [[] for _ in range(n)]
    for t, node in enumerate(nodes):
        for v in node.inputs:
            if v.node >= 0:
                last_fwd[v.node] = max(last_fwd[v.node], t)
        if node.back is not None:
            for v in node.saved:
                if v.node >= 0:
                    need[v.node].append(t)
    drop_f, drop_b = {}, {}
    for m in range(n - 1):
        if need[m]:
            drop_b.setdefault(min(need[m]), []).append(m)
        else:
            drop_f.setdefault(last_fwd[m], []).append(m)
    return drop_f, drop_b


class MicroTape(Tape):
    """A Tape that runs the END of a graph per batch micro-tensor, as TSplit's executor runs a split
    operator as micro-operators on the micro-tensors of its operands (the primitives are
    DLArraySliceForMicroTensor, src/common/c_runtime_api.cc:212-271, and split_shape,
    python/athena/ndarray.py:390-409).

    Operator calls number `split_from` and later are put off while the builder runs: they return Vars
    that carry shapes only.  When call number `total_calls - 1` (the loss) arrives, the stretch runs
    `pieces` times, once per micro-tensor, depth first: for piece i every put-off call is made again
    on a plain tape with the arguments of `piece_calls` (the same builder traced at batch / pieces:
    shapes, permutations and constants of that batch size) and with values of that piece: results of
    the stretch's own earlier calls, or, for a value from outside the stretch, micro-tensor view i of
    it when the trace shows that its shape follows the batch, the whole value when it does not
    (parameters, tables).  Forward and backward of a piece run back to back, so the stretch's
    activations and their gradients exist for one micro-tensor at a time; the loss of piece i is
    weighted with 1 / pieces (equal pieces: the mean over the batch is the mean of the pieces' means).
    The gradients leave the stretch as whole arrays: of a value that follows the batch, written piece
    by piece through micro-tensor views of one array; of a parameter, accumulated over the pieces.
    On the outer tape the stretch is ONE operator whose output is the loss and whose backward
    operators have already run.  Nothing in the stretch may couple the samples of a batch
    (COUPLES_SAMPLES); the batch must divide by `pieces`."""

    _ahead = False

    def __init__(self, backend, split_from=None, pieces=1, piece_calls=None, total_calls=None):
        Tape.__init__(self, backend)
        self.split_from, self.pieces, self.piece_calls, self.total_calls = split_from, pieces, piece_calls, total_calls
        self._ncalls = 0
        self._put_off = []        # (name, args, kwargs, out Var) of the calls put off so far
        self._deferring = False
        if split_from is not None:
            assert pieces >= 1 and piece_calls is not None and total_calls == len(piece_calls)
            bad = [c[0] for c in piece_calls[split_from:] if c[0] in COUPLES_SAMPLES]
            assert not bad, "operators that couple the samples of a batch cannot run per micro-tensor: %s" % bad[:3]

    def _inside_piece(self):
        pass

    def _call(self, fn, args, kwargs):
        c = self._ncalls
        self._ncalls += 1
        if self.split_from is None or c < self.split_from:
            return Tape._call(self, fn, args, kwargs)
        # put off: the call runs on shapes only and leaves no node
        real, self.b, self._deferring = self.b, _ShapeOnly(), True
        try:
            out = fn(self, *args, **kwargs)
        finally:
            self.b, self._deferring = real, False
        self._put_off.append((fn.__name__, args, kwargs, out))
        if c == self.total_calls - 1:
            return self._run_pieces(out)
        return out

    def _out(self, value, shape, inputs, backward, saved=None, redo=None):
        if self._deferring:
            v = Var(None, shape, any(i.needs_grad for i in inputs))
            v.node = -2          # neither a leaf nor an operator of this tape
            return v
        return Tape._out(self, value, shape, inputs, backward, saved, redo)

    def _readers_of_the_stretch(self, inner_ids):
        """Runs the stretch once on shapes only (the traced calls, stand-ins for the outside values) to learn
        which operator reads each of its values last."""
        dry = Tape(_ShapeOnly())
        env, standin = {}, {}

        def arg_for(actual, traced):
            if not isinstance(actual, Var):
                return traced
            if id(actual) in inner_ids:
                return env[inner_ids[id(actual)]]
            if id(actual) not in standin:
                standin[id(actual)] = Var(None, traced.shape, actual.needs_grad)
            return standin[id(actual)]
        for n, (name, args, kwargs, _) in enumerate(self._put_off):
            _, t_args, t_kwargs = self.piece_calls[self.split_from + n]
            env[n] = getattr(dry, name)(*[arg_for(a, ta) for a, ta in zip(args, t_args)],
                                        **{key: arg_for(kwargs[key], t_kwargs[key]) for key in kwargs})
        return _last_readers(dry._nodes)

    def _run_pieces(self, loss_var):
        k, b = self.pieces, self.b
        inner_ids = {id(c[3]): n for n, c in enumerate(self._put_off)}
        drop_f, drop_b = self._readers_of_the_stretch(inner_ids)
        outside, outside_vars = {}, []          # id(Var) -> [Var, follows the batch, whole gradient array or None]
        total = None
        for i in range(k):
            piece_tape = _PieceTape(b, self, drop_f, drop_b)
            env = {}                            # put-off call -> its result for this piece
            wrapped = {}                        # id(outside Var) -> its Var on the piece's tape

            def arg_for(actual, traced):
                if not isinstance(actual, Var):
                    return traced               # shapes, permutations, constants: those of the piece's batch size
                if id(actual) in inner_ids:
                    return env[inner_ids[id(actual)]]
                if id(actual) not in wrapped:
                    follows = tuple(traced.shape) != tuple(actual.shape)
                    if follows:
                        assert tuple(traced.shape[1:]) == tuple(actual.shape[1:]) and traced.shape[0] * k == actual.shape[0], \
                            (actual.shape, traced.shape, k)
                    if id(actual) not in outside:
                        outside[id(actual)] = [actual, follows, None]
                        outside_vars.append(actual)
                    value = b.piece(actual.value, k, i) if follows else actual.value
                    wrapped[id(actual)] = w = Var(value, traced.shape, actual.needs_grad, actual.name)
                    if not follows:
                        w.grad, w.own = actual.grad, actual.own      # a parameter's pieces add to one array
                return wrapped[id(actual)]

            for n, (name, args, kwargs, _) in enumerate(self._put_off):
                t_name, t_args, t_kwargs = self.piece_calls[self.split_from + n]
                assert t_name == name and len(t_args) == len(args), "the graph differs from the traced one"
                p_args = [arg_for(a, ta) for a, ta in zip(args, t_args)]
                p_kwargs = {key: arg_for(kwargs[key], t_kwargs[key]) for key in kwargs}
                if n == len(self._put_off) - 1:
                    assert name == "softmax_ce", "a stretch run per micro-tensor ends with the loss"
                    p_kwargs["weight"] = 1.0 / k
                env[n] = getattr(piece_tape, name)(*p_args, **p_kwargs)
            piece_loss = env[len(self._put_off) - 1]
            total = piece_loss.value if total is None else b.add(total, piece_loss.value, (1,))
            piece_tape.backward(piece_loss)
            for key, w in wrapped.items():
                actual, follows, whole = outside[key]
                if not actual.needs_grad or w.grad is None:
                    continue
                if follows:
                    if whole is None:
                        whole = outside[key][2] = b.empty(actual.shape)
                    b.assign(b.piece(whole, k, i), w.grad)
                else:
                    actual.grad = w.grad                # a parameter: summed over the pieces
                    self._owns(actual, w.own)
                w.grad = None
            del piece_tape, env, wrapped, piece_loss
        for v in outside_vars:
            whole = outside[id(v)][2]
            if whole is not None:
                self._acc(v, whole, fresh=True)
        self._put_off = []
        # on this tape the stretch is one operator: it read the outside values, its output is the loss
        # and its backward operators have run
        out = Tape._out(self, total, (1,), outside_vars, None, saved=[])
        out.needs_grad = False
        return out

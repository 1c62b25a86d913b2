"""How much one launch joins or cuts up: a launch has fewer than 2^32 threads, one a word."""
import ctypes

import pytest

from tsplit_amd import graph


def _array(shape, at):
    """A struct of that shape; the call is to refuse it before anything reads the address."""
    from tsplit_amd import ndarray as nd
    dims = (ctypes.c_int64 * len(shape))(*shape)
    a = nd.DLArray(ctypes.c_void_p(at), nd.gpu(0), len(shape), dims)
    return ctypes.pointer(a), (a, dims)


# rows in words of four and not, both just out of reach
@pytest.mark.parametrize("rows,extents", [(1 << 20, (4096, 8192, 4096)), ((1 << 20) - 1, (1365, 2048, 684)), (257, (1 << 24, 1, 1))])
def test_what_one_launch_does_not_reach_is_refused_with_a_word(rows, extents, capfd):
    from tsplit_amd._base import _LIB
    from tsplit_amd import ndarray as nd
    parts = [_array((rows, e), 16 * (i + 1)) for i, e in enumerate(extents)]
    whole = _array((rows, sum(extents)), 1 << 12)
    handles = (nd.DLArrayHandle * 3)(*[p[0] for p in parts])
    for call in (lambda: _LIB.TSplit_Join(handles, 3, whole[0], 1, None), lambda: _LIB.TSplit_Part(whole[0], handles, 3, 1, None)):
        assert call() != 0
        assert "fewer than 2^32" in capfd.readouterr().err


class _Joins(graph._ShapeOnly):
    def join(self, parts, out_shape, axis):
        return None


@pytest.mark.parametrize("shape,calls", [((2, 96, 8, 8), ["join"]), ((1 << 10, 1365, 32, 32), ["join"]), ((1 << 10, 1366, 32, 32), ["concat", "concat"])])
def test_tape_joins_pair_by_pair_what_one_launch_does_not_reach(shape, calls):
    t = graph.Tape(_Joins())
    t._log = []
    out = t.concat_all([t.const(None, shape) for _ in range(3)], 1)
    assert [c[0] for c in t._log] == calls and out.shape == (shape[0], 3 * shape[1]) + shape[2:]

"""Any number of parts joined along an axis and cut up again in one launch: byte for byte the pairs' chain (numpy's concatenation)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# rows in words and not, one part, eight, parts of nothing, the first and the last axis
@pytest.mark.parametrize("shape,axis,extents", [((3, 0, 5, 4), 1, (1, 7, 2)), ((2, 0, 17, 17), 1, (96, 5, 3, 64)), ((0, 6), 0, (4, 1, 2)), ((5, 0), 1, (3, 0, 9, 1)),
                                                ((2, 0, 8, 8), 1, (4, 8, 12, 16, 4, 4, 8, 20)), ((4, 0, 3), 1, (9,))])
def test_join_and_part(shape, axis, extents, rng):
    from tsplit_amd import gpu_links as L, ndarray as nd
    ctx = nd.gpu(0)
    shapes = [tuple(e if d == axis else v for d, v in enumerate(shape)) for e in extents]
    parts = [rng.normal(size=s).astype(np.float32) for s in shapes]
    want = np.concatenate(parts, axis)
    whole, dev = nd.array(np.zeros_like(want), ctx), [nd.array(p, ctx) for p in parts]
    L.join(dev, whole, axis)
    np.testing.assert_array_equal(whole.asnumpy(), want)
    back = [nd.array(np.ones_like(p), ctx) for p in parts]
    L.part(whole, back, axis)
    for b, p in zip(back, parts):
        np.testing.assert_array_equal(b.asnumpy(), p)
    with pytest.raises(RuntimeError):
        L.join(dev * 9, whole, axis)
    with pytest.raises(RuntimeError):
        L.join(dev + [dev[0]], whole, axis)

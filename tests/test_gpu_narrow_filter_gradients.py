"""Filter gradients of 3x3 layers with at most 64 channels on a side (Winograd routine): launches of few blocks run the depth's chains of
sums on tiles of 32 rows, one chain a wave, where larger ones run four a wave.  The sums are the same, in the same order: digests recorded
where the wide tiles took every such layer, and the float64 gradient within the 1e-4 of the other convolution tests."""
import zlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# images, channels in and out, H, W: two and four k-groups, rows and columns off the tile, a depth off the chunk, one and several ranges
CASES = {
    (16, 64, 128, 32, 32): 2721739805,
    (5, 128, 64, 61, 63): 1265109624,
    (2, 64, 64, 112, 112): 3897018141,
    (1, 64, 64, 130, 131): 4247606335,
    (9, 64, 200, 47, 50): 3571719784,
    (40, 64, 64, 54, 54): 431637729,
}


def gradient(case):
    from tsplit_amd import gpu_links as L, ndarray as nd
    n, c, o, h, w = case
    rng, ctx = np.random.RandomState(sum(case)), nd.gpu(0)
    x, dy = rng.normal(size=(n, c, h, w)).astype(np.float32), rng.normal(size=(n, o, h, w)).astype(np.float32)
    assert L.conv_takes_winograd(n, c, o, h, w, filter_gradient=True)
    dw = nd.empty((o, c, 3, 3), ctx)
    L.CuDNN_conv2d_gradient_of_filter(nd.array(x, ctx), nd.array(dy, ctx), dw, 1, 1, 1)
    return x, dy, dw.asnumpy()


@pytest.mark.parametrize("case", CASES)
def test_few_blocks_give_the_bits_of_wide_tiles(case):
    import torch
    x, dy, dw = gradient(case)
    n, c, o, h, w = case
    padded = torch.nn.functional.pad(torch.from_numpy(x).cuda().double(), (1, 1, 1, 1))
    grads = torch.from_numpy(dy).cuda().double().permute(1, 0, 2, 3).reshape(o, -1).contiguous()
    ref = np.empty(dw.shape)
    for i in range(3):
        for j in range(3):
            ref[:, :, i, j] = (grads @ padded[:, :, i:i + h, j:j + w].permute(0, 2, 3, 1).reshape(-1, c).contiguous()).cpu().numpy()
    assert np.abs(dw - ref).max() <= 1e-4 * np.abs(ref).max()
    assert zlib.crc32(np.ascontiguousarray(dw).tobytes()) == CASES[case]

"""What 32-bit byte offsets reach of a convolution's tensors (csrc/conv_reach.h), compiled for the host: every range of depth the
filter gradient plans, and every run of images, stays within the bytes its kernel may address."""
import ctypes
import itertools
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tsplit_amd", "csrc")
FULL = (1 << 31) - 1
SOURCE = """
#include "conv_reach.h"
using namespace tsplit;
extern "C" int takes(const ConvTileGeo *g, long long reach) { return filter_gradient_in_reach(*g, reach); }
extern "C" int range(const ConvTileGeo *g, long long reach, int S) { return range_depth(*g, reach, S); }
extern "C" int images(const ConvTileGeo *g, long long values, long long reach) { return images_per_launch(*g, values, reach); }
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    where = tmp_path_factory.mktemp("reach")
    (where / "reach.cpp").write_text(SOURCE)
    out = str(where / "reach.so")
    done = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, str(where / "reach.cpp"), "-o", out],
                          capture_output=True, text=True)
    assert done.returncode == 0, done.stderr
    return ctypes.CDLL(out)


def _geo(n, c, h, w, o, kh, kw, ph, pw, s):
    return (ctypes.c_int * 12)(n, c, h, w, o, kh, kw, ph, pw, s, (h + 2 * ph - kh) // s + 1, (w + 2 * pw - kw) // s + 1)


def _ranges_stay_in_reach(host, g, reach, asked):
    n, c, h, w, o, oh, ow = g[0], g[1], g[2], g[3], g[4], g[10], g[11]
    if not host.takes(g, ctypes.c_longlong(reach)):
        return False
    depth, per_image = host.range(g, ctypes.c_longlong(reach), asked), (oh * ow + 3) // 4 * 4
    assert depth >= 32 and depth % 32 == 0
    for begin in range(0, n * per_image, depth):
        images = (min(begin + depth, n * per_image) - 1) // per_image - begin // per_image
        # the last value a block may load: the last row of a tile of 128 that begins at the last channel
        assert 4 * (images * o + o + 127) * oh * ow <= reach, (tuple(g), begin, depth)
        assert 4 * (images * c + c + 127) * h * w <= reach, (tuple(g), begin, depth)
    return True


def test_ranges_of_depth_stay_within_what_a_block_addresses(host):
    # 2 x 2 positions of large images: a step of 32 would cover eight of them, four lie within reach
    far = _geo(8, 300, 512, 512, 16, 3, 3, 1, 1, 256)
    assert not host.takes(far, ctypes.c_longlong(FULL))
    taken = 0
    for oh, ow, images in itertools.product(range(1, 6), range(1, 7), (1, 3, 4, 5, 9, 40, 300)):
        for span in (2, 3, 4, 5, 8, 17, 34):
            g = _geo(images, 20, oh * 3, ow * 3, 24, 3, 3, 0, 0, 3)
            reach = span * 4 * (20 + 128) * 9 * oh * ow
            taken += sum(_ranges_stay_in_reach(host, g, reach, S) for S in (1, 2, 7, 1000))
    assert taken > 2000
    rng = random.Random(5)
    for _ in range(300):
        g = _geo(rng.randint(1, 64), rng.randint(1, 600), rng.randint(8, 300), rng.randint(8, 300), rng.randint(1, 600), 3, 3, 1, 1, rng.choice((1, 2, 8)))
        for reach in (FULL, 1 << 24):
            _ranges_stay_in_reach(host, g, reach, rng.choice((1, 3, 50)))


def test_runs_of_images_stay_in_reach_with_the_base_moved_back(host):
    """Both passes move the base of the gathered tensor back and address the run's bytes and that distance.  Wide padding of narrow
    images makes the data gradient's distance, a filter's height times the OUTPUT's width, the larger one."""
    rng, narrow = random.Random(6), 0
    for _ in range(4000):
        kh, kw = rng.choice(((64, 1), (32, 2), (8, 8), (7, 7), (3, 3), (1, 1)))
        h, w, ph, pw = rng.randint(1, 40), rng.randint(1, 40), rng.randint(0, 40), rng.randint(0, 120)
        if h + 2 * ph < kh or w + 2 * pw < kw:
            continue
        g = _geo(1 << 20, rng.randint(1, 64), h, w, rng.randint(1, 64), kh, kw, ph, pw, rng.choice((1, 1, 2, 3)))
        for values, back in ((g[1] * h * w, ph * w + pw), (g[4] * g[10] * g[11], (kh - 1) * g[11] + kw - 1)):
            for reach in (FULL, 1 << 20):
                per = host.images(g, ctypes.c_longlong(values), ctypes.c_longlong(reach))
                assert per == 0 or 4 * (per * values + back) <= reach, (tuple(g), per)
                narrow += per > 0 and back > ph * w + pw + kh * w + kw
    assert narrow > 100

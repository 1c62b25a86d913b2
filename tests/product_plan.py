"""Which kernel a matrix product runs on, and in which ranges of its depth: csrc/tile_plan.h compiled for the host, as csrc/gemm.hip asks it."""
import ctypes
import functools
import os
import subprocess
import tempfile
from collections import namedtuple

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tsplit_amd", "csrc")
SOURCE = """
#include "tile_plan.h"
using namespace tsplit;
extern "C" void plan(long long M, long long N, long long K, long long batch, int *got) {
  const int64_t cols = N;
  const int steps = std::max(1ll, (K + 31) / 32);
  const TilePlan t = plan_tiles(M, &cols, &steps, 1, batch, batch > 1 ? 1 : 64, static_cast<double>(M) * N, kProductCost);
  const WavesPlan w = plan_waves(M, N, K, batch, t, batch > 1);
  const int range = (steps + t.S - 1) / t.S * 32;
  const int values[] = {t.tile, range, w.tile, w.waves, w.S, w.kchunk};
  for (int i = 0; i < 6; ++i) got[i] = values[i];
}
"""
TILES = ((128, 128), (64, 128), (128, 64), (64, 64))            # of gemm_tile.h
WAVE_TILES = ((16, 16), (16, 32), (32, 16), (32, 32))           # of gemm_waves.h
# tile: of the kernel that runs, range: values of the depth in one of its ranges; tile_range: what the tile kernel's would be
Plan = namedtuple("Plan", "waves tile range tile_range")


@functools.lru_cache(maxsize=None)
def _library():
    with tempfile.TemporaryDirectory() as where:
        src, out = os.path.join(where, "plan.cpp"), os.path.join(where, "plan.so")
        with open(src, "w") as f:
            f.write(SOURCE)
        done = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, src, "-o", out], capture_output=True, text=True)
        assert done.returncode == 0, done.stderr
        return ctypes.CDLL(out)


def plan(M, N, K, batch=1):
    got = (ctypes.c_int * 6)()
    _library().plan(*(ctypes.c_longlong(v) for v in (M, N, K, batch)), got)
    tile, tile_range, wave_tile, waves, S, kchunk = got
    if waves:
        assert S == -(-K // kchunk) and waves in (4, max(2, min(4, S)))
        return Plan(waves, WAVE_TILES[wave_tile], kchunk, tile_range)
    return Plan(0, TILES[tile], tile_range, tile_range)

"""The choice of tile and ranges (csrc/tile_plan.h), compiled for the host, against times of the same launches on all four tiles and many
counts of ranges, taken on an MI355X."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tsplit_amd", "csrc")
COSTS = ["kProductCost", "kOneTapCost", "kGatheredCost", "kPairsCost", "kFilterWordsCost", "kFilterTapsCost"]
SOURCE = """
#include "tile_plan.h"
using namespace tsplit;
extern "C" void plan(int cost, long long M, const long long *cols, const int *steps, int parts, long long batch, int most, double out, int *got) {
  static const TileCost costs[] = {%s};
  int64_t c[64];
  for (int i = 0; i < parts; ++i) c[i] = cols[i];
  const TilePlan p = plan_tiles(M, c, steps, parts, batch, most, out, costs[cost]);
  got[0] = p.tile;
  got[1] = p.S;
}
""" % ", ".join(COSTS)

# name, cost, rows, columns and steps of each part, most ranges, values of the result, us by ranges on 128x128, 64x128, 128x64, 64x64
MEASURED = [
    ("18 x 25088 x 4096, second operand transposed", "kProductCost", 18, [25088], [128], 64, 451584,
     [{2: 240, 4: 244, 5: 203, 7: 223, 8: 228, 9: 236, 10: 210, 12: 224, 13: 208, 14: 206, 16: 231, 20: 240, 24: 235, 28: 227, 32: 241, 40: 241},
      {2: 128, 3: 129, 4: 139, 6: 134, 7: 120, 8: 126, 9: 141, 10: 126, 11: 121, 12: 135, 14: 135, 16: 133, 20: 131, 24: 135, 28: 136, 32: 143, 40: 143, 48: 146},
      {1: 245, 3: 211, 4: 223, 5: 206, 6: 220, 7: 210, 8: 212, 10: 215, 12: 219, 14: 213, 16: 216, 20: 231, 24: 231, 28: 234, 32: 242, 40: 244},
      {2: 129, 4: 130, 5: 108, 6: 129, 7: 121, 8: 122, 10: 117, 12: 126, 14: 119, 16: 127, 24: 131}]),
    ("64 x 25088 x 4096, the same", "kProductCost", 64, [25088], [128], 64, 1605632,
     [{2: 242, 4: 249, 5: 209, 7: 230, 8: 236, 9: 246, 10: 222, 12: 239, 13: 222, 14: 219, 16: 246, 28: 250},
      {2: 133, 3: 134, 4: 146, 6: 143, 7: 131, 8: 141, 9: 151, 10: 139, 11: 136, 12: 158, 14: 152, 16: 154, 20: 156},
      {1: 246, 3: 212, 4: 227, 5: 208, 6: 224, 7: 218, 8: 220, 10: 223, 12: 230, 14: 227, 16: 231, 20: 246, 24: 250},
      {1: 137, 2: 138, 4: 135, 5: 123, 6: 137, 7: 131, 8: 134, 10: 131, 12: 146, 14: 139}]),
    ("1x1, 2048 -> 512 at 7 x 7", "kOneTapCost", 512, [3136], [64], 32, 1605632,
     [{2: 89, 4: 80, 5: 74},
      {2: 76, 3: 83, 4: 88, 5: 85, 6: 79, 7: 88, 8: 87, 10: 92},
      {1: 90, 2: 85, 3: 82, 4: 84, 5: 82, 6: 74, 7: 79, 8: 79, 9: 80, 10: 81, 11: 81, 12: 81, 14: 86, 16: 89, 20: 89},
      {1: 69, 2: 75, 3: 78, 4: 71, 5: 69, 6: 73, 7: 75, 8: 76, 10: 83, 12: 82}]),
    ("3x3, 512 -> 512 at 7 x 7, data gradient", "kGatheredCost", 512, [3136], [144], 32, 1605632,
     [{2: 202, 4: 195, 5: 166, 6: 201, 7: 183, 8: 200, 10: 184, 12: 192},
      {2: 202, 3: 195, 4: 202, 5: 170, 6: 183, 7: 185, 8: 186, 10: 186, 12: 195, 14: 199, 16: 203},
      {3: 179, 4: 186, 5: 181, 6: 161, 7: 164, 8: 171, 9: 158, 10: 168, 12: 174, 13: 173, 14: 177, 16: 178, 20: 177, 24: 192, 28: 190},
      {2: 190, 3: 172, 4: 171, 5: 162, 6: 170, 7: 167, 8: 172, 10: 178, 12: 177, 14: 187, 16: 186, 20: 188}]),
    ("3x3 stride 2, 224 -> 256 at 35 x 35", "kGatheredCost", 256, [9248], [63], 32, 2367488,
     [{3: 120, 4: 135, 5: 118, 6: 129, 7: 116, 8: 125, 10: 132, 12: 136, 14: 139},
      {2: 133, 3: 128, 4: 122, 5: 119, 6: 123, 7: 120, 8: 130, 10: 130, 12: 135, 14: 139},
      {2: 119, 3: 115, 4: 110, 5: 108, 6: 110, 7: 108, 8: 119, 10: 118, 12: 126, 14: 127},
      {1: 129, 2: 117, 3: 109, 4: 116, 5: 116, 6: 119, 7: 117, 8: 124, 10: 125}]),
    ("3x3 stride 2, 384 -> 384 at 35 x 35, data gradient", "kPairsCost", 384, [10368, 9792], [72, 36], 32, 15052800,
     [{1: 375, 2: 441},
      {1: 384, 2: 424, 3: 455},
      {1: 357, 2: 387, 3: 406, 4: 418, 5: 435},
      {1: 360, 2: 378, 3: 405, 4: 426, 5: 439}]),
    ("1x1, 64 -> 256 at 56 x 56, filter gradient", "kFilterWordsCost", 256, [64], [6272], 1024, 16384,
     [{128: 121, 256: 120, 512: 130},
      {64: 134, 128: 113, 192: 113, 256: 134, 384: 124},
      {128: 72, 256: 71, 384: 73},
      {64: 84, 128: 70, 192: 70, 256: 69, 384: 72, 448: 74}]),
    ("3x3, 512 -> 512 at 28 x 28, filter gradient", "kFilterTapsCost", 512, [4608], [441], 1024, 2359296,
     [{3: 658, 5: 615, 6: 667, 7: 575, 8: 639, 10: 620, 12: 603, 14: 593, 16: 578, 17: 603, 20: 642, 24: 639, 28: 640, 32: 632, 40: 657, 48: 700},
      {3: 707, 4: 658, 5: 620, 6: 619, 7: 602, 8: 601, 10: 646, 12: 622, 14: 624, 16: 608, 20: 649, 24: 650, 28: 669, 32: 662, 40: 686, 48: 715},
      {3: 673, 4: 626, 5: 599, 6: 592, 7: 576, 8: 579, 10: 619, 12: 601, 14: 600, 16: 584, 20: 623, 24: 622, 28: 636, 32: 632, 40: 657, 48: 687},
      {2: 700, 3: 626, 4: 607, 5: 641, 6: 626, 7: 616, 8: 615, 10: 635, 12: 614, 14: 634, 16: 621, 20: 646, 24: 656, 28: 665, 32: 666, 40: 688, 48: 723}]),
    ("3x3 stride 2, 64 -> 96 at 147 x 147, filter gradient", "kFilterTapsCost", 96, [576], [5332], 1024, 55296,
     [{48: 302, 51: 288, 96: 276, 102: 262, 128: 313, 153: 276, 204: 275, 256: 278, 307: 285, 358: 285},
      {48: 305, 51: 287, 64: 308, 76: 267, 96: 289, 102: 277, 128: 273, 153: 272, 179: 279, 204: 284, 230: 286, 256: 284},
      {56: 245, 80: 234, 85: 223, 96: 270, 113: 238, 128: 253, 142: 238, 170: 235, 199: 237, 227: 244, 256: 240},
      {28: 282, 40: 267, 42: 252, 48: 282, 56: 244, 64: 279, 71: 253, 80: 261, 85: 249, 96: 251, 99: 245, 113: 249, 128: 249, 142: 248}]),
]


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    where = tmp_path_factory.mktemp("plan")
    (where / "plan.cpp").write_text(SOURCE)
    out = str(where / "plan.so")
    done = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, str(where / "plan.cpp"), "-o", out],
                          capture_output=True, text=True)
    assert done.returncode == 0, done.stderr
    lib = ctypes.CDLL(out)

    def call(cost, M, cols, steps, batch=1, most=64, values=1.0):
        got = (ctypes.c_int * 2)()
        lib.plan(COSTS.index(cost), ctypes.c_longlong(M), (ctypes.c_longlong * len(cols))(*cols), (ctypes.c_int * len(steps))(*steps), len(cols),
                 ctypes.c_longlong(batch), most, ctypes.c_double(values), got)
        return tuple(got)
    return call


@pytest.mark.parametrize("case", MEASURED, ids=lambda c: c[0])
def test_choices_are_near_the_best_of_all_tiles_and_ranges(case, plan):
    _, cost, M, cols, steps, most, values, times = case
    tile, S = plan(cost, M, cols, steps, 1, most, values)
    nearest = min(times[tile], key=lambda s: abs(s - S))
    assert abs(nearest - S) <= 0.1 * S, (tile, S)
    assert times[tile][nearest] <= 1.08 * min(min(t.values()) for t in times), (tile, S)


@pytest.mark.parametrize("cost", COSTS)
def test_choices_stay_in_their_bounds(cost, plan):
    for M in (1, 16, 65, 1000, 8192, 1 << 22):
        for cols in ([1], [300], [5000, 4000], [1 << 21], [7, 7, 7, 0]):
            for deep in (0, 1, 2, 31, 144, 30000):
                for most in (1, 32, 1024):
                    tile, S = plan(cost, M, cols, [deep] * len(cols), 1, most, float(M) * sum(cols))
                    bm, bn = ((128, 128), (64, 128), (128, 64), (64, 64))[tile]
                    tiles = sum(-(-M // bm) * -(-c // bn) for c in cols)
                    assert 1 <= S <= max(1, min(most, deep)) and (S == 1 or tiles <= 1024)
                    assert S == 1 or -(-deep // -(-deep // S)) == S      # no range is empty

"""Which workgroup computes which row tile (csrc/prompt_tiles.h, host code as well as device code)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tinyllmforge_amd", "csrc")
SOURCE = """
#define __host__
#define __device__
#include "prompt_tiles.h"
extern "C" int place(long xtiles, long planes, long seqs, int together, int most, int *out) {
  tlf::PromptTiles t;
  const int blocks = tlf::prompt_tiles_make(t, xtiles, planes, seqs, together);
  for (int b = 0; b < blocks && b < most; ++b)
    if (!tlf::prompt_tile(t, b, out[3 * b], out[3 * b + 1], out[3 * b + 2])) out[3 * b] = -1;
  return blocks;
}
struct Grid {
  long x, y;
  Grid(long x, long y = 1) : x(x), y(y) {}
};
// The grid, and how many of its workgroups behind the last one have a tile, or of those before have none but should
extern "C" void limits(long xtiles, long planes, long seqs, long *out) {
  tlf::PromptTiles t;
  const int blocks = tlf::prompt_tiles_make(t, xtiles, planes, seqs);
  const Grid g = tlf::prompt_grid<Grid>(blocks);
  long tiles = 0, beyond = 0;
  for (long y = 0; y < g.y; ++y)
    for (long x = 0; x < g.x && blocks; ++x) {
      const int b = tlf::prompt_block(x, y);
      int s, p, i;
      if (!tlf::prompt_tile(t, b, s, p, i)) continue;
      ++tiles;
      beyond += b >= blocks || s < 0 || s >= seqs || p < 0 || p >= planes || i < 0 || i >= xtiles;
    }
  out[0] = blocks; out[1] = g.x; out[2] = g.y; out[3] = beyond + (blocks ? tiles - xtiles * planes * seqs : 0);
}
"""


@pytest.fixture(scope="module")
def place(tmp_path_factory):
    at = tmp_path_factory.mktemp("tiles")
    (at / "place.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-O2", "-I", CSRC, str(at / "place.cpp"), "-o", str(at / "place.so")], check=True)
    lib = ctypes.CDLL(str(at / "place.so"))
    call = lib.place
    call.argtypes = [ctypes.c_long] * 3 + [ctypes.c_int] * 2 + [ctypes.c_void_p]

    def table(xtiles, planes, seqs, together=4):
        most = 8 * (xtiles + 7) * planes * seqs
        out = np.full((most, 3), -1, dtype=np.int32)
        blocks = call(xtiles, planes, seqs, together, most, out.ctypes.data)
        assert 0 < blocks <= most
        return out[:blocks]

    def limits(xtiles, planes, seqs):
        out = (ctypes.c_long * 4)()
        lib.limits(ctypes.c_long(xtiles), ctypes.c_long(planes), ctypes.c_long(seqs), out)
        return list(out)
    table.limits = limits
    return table


@pytest.mark.parametrize("planes", [1, 2, 3, 4, 5, 6, 8, 12, 16, 24])
def test_every_tile_once_and_every_xcd_its_share(place, planes):
    for xtiles in (1, 2, 3, 4, 7, 8, 9, 10, 16, 17, 33, 64):
        for seqs in (1, 2, 3, 8, 15, 16, 64, 100):
            t = place(xtiles, planes, seqs, 1 if seqs == 15 else 4)
            xcd, used = np.arange(len(t)) % 8, t[:, 0] >= 0
            seq, plane, tile = t[used].T
            assert seq.max() < seqs and plane.min() >= 0 and plane.max() < planes and tile.min() >= 0 and tile.max() < xtiles
            where = (seq * planes + plane) * xtiles + tile
            assert len(where) == len(np.unique(where)) == seqs * planes * xtiles
            load = np.bincount(xcd[used], weights=tile + 1, minlength=8)       # a tile's keys grow with its place
            if len(where) >= 8 * 32:                                        # enough for the kinds of tiles to come out even
                assert load.max() <= 1.1 * load.mean(), (xtiles, seqs, load)


def test_a_grid_of_many_workgroups(place):
    """2^23 workgroups of 512 threads and more, which one dimension of a launch does not hold."""
    places = place.limits
    for xtiles, planes, seqs in ((683, 8, 2000), (1366, 3, 3000), (1, 1, 1 << 22), (100000, 8, 100)):
        blocks, x, y, beyond = places(xtiles, planes, seqs)
        assert blocks >= xtiles * planes * seqs and x * 512 < 1 << 32 and y <= 65535 and x * y >= blocks and x % 8 == 0
        assert beyond == 0
    assert places(1 << 20, 8, 1 << 12)[0] == 0

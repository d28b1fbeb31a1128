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
extern "C" int place(long xtiles, long planes, long seqs, int most, int *out) {
  tlf::PromptTiles t;
  const int blocks = tlf::prompt_tiles_make(t, xtiles, planes, seqs);
  for (int b = 0; b < blocks && b < most; ++b)
    if (!tlf::prompt_tile(t, b, out[3 * b], out[3 * b + 1], out[3 * b + 2])) out[3 * b] = -1;
  return blocks;
}
"""


@pytest.fixture(scope="module")
def place(tmp_path_factory):
    at = tmp_path_factory.mktemp("tiles")
    (at / "place.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-O1", "-I", CSRC, str(at / "place.cpp"), "-o", str(at / "place.so")], check=True)
    call = ctypes.CDLL(str(at / "place.so")).place
    call.argtypes = [ctypes.c_long] * 3 + [ctypes.c_int, ctypes.c_void_p]

    def table(xtiles, planes, seqs):
        most = 8 * (xtiles + 7) * planes * seqs
        out = np.full((most, 3), -1, dtype=np.int32)
        blocks = call(xtiles, planes, seqs, most, out.ctypes.data)
        assert 0 < blocks <= most
        return out[:blocks]
    return table


@pytest.mark.parametrize("planes", [1, 2, 3, 4, 5, 6, 8, 12, 16, 24])
def test_every_tile_once_and_every_xcd_its_share(place, planes):
    for xtiles in (1, 2, 3, 4, 7, 8, 9, 10, 16, 17, 33, 64):
        for seqs in (1, 2, 3, 8, 15, 16, 64, 100):
            t = place(xtiles, planes, seqs)
            xcd, used = np.arange(len(t)) % 8, t[:, 0] >= 0
            seq, plane, tile = t[used].T
            assert seq.max() < seqs and plane.min() >= 0 and plane.max() < planes and tile.min() >= 0 and tile.max() < xtiles
            where = (seq * planes + plane) * xtiles + tile
            assert len(where) == len(np.unique(where)) == seqs * planes * xtiles
            load = np.bincount(xcd[used], weights=tile + 1, minlength=8)       # a tile's keys grow with its place
            if len(where) >= 8 * 32:                                        # enough for the kinds of tiles to come out even
                assert load.max() <= 1.1 * load.mean(), (xtiles, seqs, load)

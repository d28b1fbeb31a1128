"""How the key ranges of row tiles are cut (csrc/talk_split.h, host code as well as device code)."""
import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tinyllmforge_amd", "csrc")
SOURCE = """
#define __host__
#define __device__
#include "talk_split.h"
using namespace tlf;
extern "C" int cuts(long portions, long tokens, long keys, int tq) { return talk_cuts(portions, tokens, keys, tq); }
extern "C" int pays(long portions, long tokens, long rows, long keys, int tq) { return talk_cuts_pay(portions, tokens, rows, keys, tq); }
extern "C" int steps(int start, int tokens, int tq, int x) { return talk_steps(start, tokens, tq, x); }
extern "C" int tiles(int tokens, int tq) { return talk_tiles(tokens, tq); }
extern "C" int extras(int n, int per) { return talk_extras(n, per); }
extern "C" int length_class(int n, int per) { return talk_class(n, per); }
extern "C" int per(const int *steps, int n) {
  long all = 0;
  for (int i = 0; i < n; ++i) all += steps[i];
  return talk_per(all, n, [&](int per) {
    long e = 0;
    for (int i = 0; i < n; ++i) e += talk_extras(steps[i], per) < kTalkExtras ? talk_extras(steps[i], per) : kTalkExtras;
    return static_cast<int>(e);
  });
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    at = tmp_path_factory.mktemp("split")
    (at / "split.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-O2", "-I", CSRC, str(at / "split.cpp"), "-o", str(at / "split.so")], check=True)
    lib = ctypes.CDLL(str(at / "split.so"))
    lib.cuts.argtypes = [ctypes.c_long] * 3 + [ctypes.c_int]
    lib.pays.argtypes = [ctypes.c_long] * 4 + [ctypes.c_int]
    return lib


@pytest.mark.parametrize("tq", [16, 32, 64])
def test_parts_cover_every_step_once(lib, tq):
    rng = random.Random(tq)
    batches = [[(0, 1)], [(4095, 1)], [(0, 8192)], [(1 << 20, 40)], [(31, tq), (32, tq), (33, tq + 1)]]
    batches += [[(rng.choice([0, 64, rng.randrange(5000)]), rng.randint(1, 3000)) for _ in range(rng.randint(1, 12))] for _ in range(200)]
    for batch in batches:
        most = max(n for _, n in batch)
        if not lib.cuts(len(batch), most, max(a + n for a, n in batch), tq):
            continue
        steps = [lib.steps(a, n, tq, x) for a, n in batch for x in range(lib.tiles(n, tq))]
        assert steps == [(a + min((x + 1) * tq, n) - 1) // 32 + 1 for a, n in batch for x in range(-(-n // tq))] and len(steps) <= 512
        per = lib.per((ctypes.c_int * len(steps))(*steps), len(steps))
        assert per >= 3
        extras = [lib.extras(s, per) for s in steps]
        assert sum(extras) <= 256                                    # what the workspace has room for
        for s, e in zip(steps, extras):
            assert 1 <= s - e * per <= per                           # the rest, behind e whole parts
            assert 0 <= lib.length_class(s - e * per, per) <= 127 and lib.length_class(per, per) == 0
        assert all(lib.length_class(n, per) >= lib.length_class(n + 1, per) for n in range(1, min(per, 300)))


def test_which_launches_are_cut(lib):
    assert lib.cuts(1, 5000, 5000, 32) and lib.cuts(8, 2048, 2048, 32) and lib.cuts(1, 130, 2178, 32)
    assert not lib.cuts(1, 90, 96, 32) and not lib.cuts(16, 300, 4000, 16) and not lib.cuts(9, 2048, 2048, 32) and not lib.cuts(64, 128, 128, 32)


# portions, their longest, rows of all, keys at most, rows of a tile
@pytest.mark.parametrize("launch", [(1, 8000, 8000, 8000, 16), (4, 2048, 8192, 2048, 16), (3, 2600, 7800, 2624, 16), (24, 250, 6000, 256, 32), (48, 128, 6144, 1152, 32),
                                    (24, 128, 3072, 1152, 16), (12, 250, 3000, 256, 16), (9, 2048, 18432, 2048, 32)], ids=str)
def test_launches_that_whole_tiles_do_better(lib, launch):
    assert not lib.pays(*launch)


@pytest.mark.parametrize("launch", [(1, 8000, 8000, 8000, 32), (8, 2048, 12000, 2048, 32), (4, 2048, 6143, 2048, 16), (6, 1300, 7800, 1344, 16), (1, 130, 130, 2240, 32),
                                    (12, 400, 4800, 448, 32), (1, 4000, 4000, 4032, 16), (20, 600, 9000, 640, 32)], ids=str)
def test_launches_that_parts_do_better(lib, launch):
    assert lib.pays(*launch) and lib.cuts(launch[0], launch[1], launch[3], launch[4])       # which is what the workspace is sized for

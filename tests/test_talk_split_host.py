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
extern "C" int pays(const long *l, int tq) { return talk_cuts_pay({l[0], l[1], l[2], l[3], l[4]}, tq); }
extern "C" int route(int singles, const long *s, const long *l, int heads, int tq) {
  return talk_route(singles, {s[0], s[1], s[2], s[3], s[4]}, {l[0], l[1], l[2], l[3], l[4]}, heads, tq);
}
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


# portions as (tokens held before, tokens brought), rows of a tile; measured, us in parts and whole
WHOLE = [([(0, 8000)], 16), ([(0, 2048)] * 4, 16), ([(0, 2600)] * 3, 16),                                     # 1530, 1421; 483, 449; 565, 535
         ([(1024, 600)] * 8, 16), ([(0, 800)] * 7, 16), ([(1024, 600)] * 7, 16), ([(2048, 2000)] * 4, 16),    # 484, 448; 227, 199; 480, 432; 1279, 1205
         ([(0, 250)] * 24, 32), ([(1024, 128)] * 48, 32), ([(1024, 128)] * 24, 16), ([(0, 250)] * 12, 16),    # 93, 89; 272, 251; 267, 230; 93, 88
         ([(0, 2048)] * 9, 32)]                                                                               # more tiles than a plan holds
PARTS = [([(0, 8000)], 32), ([(0, n) for n in range(1061, 2048, 141)], 32), ([(2048, 130)], 32), ([(0, 400)] * 12, 32),      # 795, 1280; 353, 399; 92, 355; 99, 106
         ([(0, n) for n in (1024, 1365, 1706, 2048)], 16), ([(0, 4000)], 16), ([(0, 1500)] * 5, 16), ([(0, 1300)] * 6, 16),  # 347, 375; 453, 640; 419, 506; 388, 422
         ([(0, 850)] * 9, 16), ([(0, 640)] * 12, 16), ([(4096, 300)] * 4, 16), ([(0, n) for n in range(300, 601, 15)], 32)]  # 288, 345; 235, 247; 357, 696; 153, 166
load = lambda ps: (ctypes.c_long * 5)(len(ps), max([n for _, n in ps], default=0), sum(n for _, n in ps), sum(n * a + n * (n + 1) // 2 for a, n in ps),
                                      max([a + n for a, n in ps], default=0))


@pytest.mark.parametrize("portions,tq,pays", [(*v, False) for v in WHOLE] + [(*v, True) for v in PARTS], ids=[f"whole {i}" for i in range(len(WHOLE))] + [f"parts {i}" for i in range(len(PARTS))])
def test_launches_that_parts_do_better(lib, portions, tq, pays):
    v = load(portions)
    assert lib.pays(v, tq) == pays
    if pays:                                                         # which is what the workspace is sized for
        assert lib.cuts(v[0], v[1], v[4], tq)


ROWS, TOGETHER, APART = range(3)


# short and long portions as (tokens held before, tokens brought), single tokens, heads; measured, one by one in us: row by row, together, apart
STEPS = [([(0, 9)] * 7, [], 0, 16, ROWS), ([(2048, 2)] * 33, [], 0, 16, ROWS),              # fewer than 64 rows; 128, 158
         ([(0, 100)], [], 0, 16, ROWS), ([(4096, 100)], [], 0, 16, TOGETHER),               # 26, 43; 237, 146
         ([(64, 4)] * 16, [], 0, 32, ROWS), ([(1024, 4)] * 64, [], 0, 32, TOGETHER),        # 22, 37; 194, 143
         ([(2048, 3)] * 100, [], 0, 16, TOGETHER), ([(2048, 2)] * 200, [], 0, 32, TOGETHER),  # 445, 320; 683, 570
         ([(64, 20)] * 30, [(0, 200)], 0, 16, TOGETHER), ([(1024, 20)] * 30, [(0, 200)], 0, 16, APART),         # 118, 66, 87; 399, 210, 140
         ([(1024, 20)] * 40, [(0, 1000)], 0, 32, APART), ([(0, 100)] * 10, [(0, 300)] * 3, 0, 16, TOGETHER),    # 591, 376, 243; 158, 70, 100
         ([(64, 10)] * 60, [(0, 4000)], 0, 32, APART), ([(2048, 2)] * 33, [(0, 4000)], 0, 32, ROWS),            # 533, 1419, 498; 585, 996, 649
         ([(1024, 20)] * 4, [(0, 300)], 0, 32, TOGETHER), ([(0, 16)] * 4, [(64, 130)], 2, 16, TOGETHER)]        # 126, 79, 120; not measured


@pytest.mark.parametrize("short,long,singles,heads,want", STEPS, ids=[str(i) for i in range(len(STEPS))])
def test_how_short_portions_run(lib, short, long, singles, heads, want):
    assert lib.route(singles, load(short), load(long), heads, 16 if heads > 16 else 32) == want

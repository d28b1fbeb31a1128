"""Which rows the preparation of attention with sinks works on in runs (csrc/sink_runs.h)."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tinyllmforge_amd", "csrc")
SOURCE = """
#include "sink_runs.h"
extern "C" long from(long n, long singles, long seqs, long hy, int conv) { return tlf::sink_runs_from(n, singles, seqs, hy, conv); }
extern "C" int run_rows(long rows, long hy) { return tlf::sink_run_rows(rows, hy); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    at = tmp_path_factory.mktemp("runs")
    (at / "runs.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-O2", "-I", CSRC, str(at / "runs.cpp"), "-o", str(at / "runs.so")], check=True)
    lib = ctypes.CDLL(str(at / "runs.so"))
    lib["from"].argtypes, lib["from"].restype = [ctypes.c_long] * 4 + [ctypes.c_int], ctypes.c_long
    lib.run_rows.argtypes = [ctypes.c_long] * 2
    return lib


# rows, single tokens, sequences, workgroups of a row
@pytest.mark.parametrize("step", [(512 + 600, 512, 513, 3), (9000, 9000, 9000, 3), (9000, 0, 4500, 3), (1500, 0, 500, 3), (1500, 0, 1, 2), (1100, 0, 275, 2), (4000, 0, 0, 3),
                                  (1024, 0, 1, 16), (128 + 1500, 128, 129, 2), (8 + 3000, 8, 9, 3)], ids=str)
def test_steps_without_runs(lib, step):
    assert lib["from"](*step, 1) == step[0]


@pytest.mark.parametrize("step", [(12237, 0, 8, 3), (1100, 0, 1, 3), (1600, 0, 1, 2), (1100, 0, 275, 3), (9000, 0, 3000, 3), (2 + 2000, 2, 3, 2), (4 + 3000, 4, 5, 3)], ids=str)
def test_steps_of_runs_alone(lib, step):
    assert lib["from"](*step, 1) == 0


@pytest.mark.parametrize("step", [(64 + 12000, 64, 65, 3), (500 + 6000, 500, 501, 2), (8 + 6000, 8, 9, 2)], ids=str)
def test_single_tokens_apart(lib, step):
    assert lib["from"](*step, 1) == step[1]


def test_without_a_convolution_only_the_number_of_rows_counts(lib):
    for seqs, singles in ((0, 0), (1, 0), (4000, 4000)):
        assert [lib["from"](n, singles, seqs, 3, 0) for n in (1025, 1500, 1800, 4000, 8000, 9000)] == [1025, 1500, 0, 0, 0, 9000]


def test_runs_fit_their_arrays(lib):
    assert [lib.run_rows(n, 3) for n in (1, 1500, 4095, 4096, 8191, 8192, 100000)] == [8, 8, 8, 16, 16, 24, 24]

"""Launch shapes of the streaming scans (manta_amd/csrc/stream_plan.hpp),
checked on the CPU."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "manta_amd", "csrc")

DRIVER = r"""
#include "stream_plan.hpp"
extern "C" int rounds(int64_t tiles, int64_t nq, int64_t wgs) { return manta::choose_rounds(tiles, nq, wgs); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("stream_plan")
    src, so = d / "plan.cpp", d / "plan.so"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-fPIC", "-shared", "-I" + CSRC, str(src), "-o",
                    str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.rounds.argtypes = [C.c_int64, C.c_int64, C.c_int64]
    return lib


def test_rounds_stay_within_the_rows(lib):
    for tiles in (1, 2, 3, 4, 5, 7, 16, 63, 64, 65, 1000, 40000):
        for nq in (1, 2, 7, 8, 64, 512, 1024, 65535):
            for wgs in (256, 512):
                r = lib.rounds(tiles, nq, wgs)
                assert 1 <= r <= 64 and r <= tiles, (tiles, nq, wgs, r)
                # as many as spread the work over wgs workgroups, where there are that many
                assert r >= min(64, tiles, -(-tiles * nq // wgs)), (tiles, nq, wgs, r)

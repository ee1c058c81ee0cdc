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
extern "C" int buffered(int64_t tiles, int64_t nq, int64_t wgs, int rounds, int pitch) {
    return manta::buffered_rounds(tiles, nq, wgs, rounds, 512, pitch);
}
extern "C" int stream(int q8, int64_t n, int64_t d, int64_t nq) {
    return manta::stream_is_faster(q8 != 0, n, d, nq);
}
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
    lib.buffered.argtypes = [C.c_int64, C.c_int64, C.c_int64, C.c_int, C.c_int]
    lib.stream.argtypes = [C.c_int, C.c_int64, C.c_int64, C.c_int64]
    return lib


def test_rounds_stay_within_the_rows(lib):
    for tiles in (1, 2, 3, 4, 5, 7, 16, 63, 64, 65, 1000, 40000):
        for nq in (1, 2, 7, 8, 64, 512, 1024, 65535):
            for wgs in (256, 512):
                r = lib.rounds(tiles, nq, wgs)
                assert 1 <= r <= 64 and r <= tiles, (tiles, nq, wgs, r)
                # as many as spread the work over wgs workgroups, where there are that many
                assert r >= min(64, tiles, -(-tiles * nq // wgs)), (tiles, nq, wgs, r)


def test_buffered_rounds_leave_no_short_wave_of_long_parts(lib):
    """Few workgroups past a whole wave only where the parts are short."""
    for tiles in (1, 5, 16, 100, 1013, 1172, 2735, 4688, 9766, 19531, 32768):
        for nq in (1, 2, 3, 5, 6, 7, 20, 64, 300, 1000):
            for pitch in (16, 32, 64, 128, 192, 336, 1008):
                rounds = lib.rounds(tiles, nq, 256)
                r = lib.buffered(tiles, nq, 256, rounds, pitch)
                parts, most = -(-tiles // r), max(512, -(-tiles // rounds))
                assert 1 <= r <= min(64, tiles) and parts <= most, (tiles, nq, pitch, rounds, r)
                short = max(24, -(-tiles // 512))
                assert r <= short or nq * parts <= 512, (tiles, nq, pitch, rounds, r)
                if nq * -(-tiles // rounds) <= 256:
                    assert r == rounds
    assert lib.buffered(2735, 6, 256, 64, 32) == 33


# Whole calls timed both ways, us: format, n, d, nq, in passes, streaming.
TIMED = [
    ("q8", 159505, 128, 8, 55, 41), ("q8", 23925, 384, 32, 56, 42), ("q8", 79753, 512, 8, 59, 50),
    ("q8", 156251, 384, 8, 62, 99), ("q8", 78125, 1024, 8, 75, 129), ("q8", 11963, 1024, 32, 62, 52),
    ("q8", 500, 256, 512, 37, 33), ("q8", 3739, 768, 128, 45, 52), ("q8", 1200, 768, 200, 39, 52),
    ("q8", 1200, 1024, 200, 42, 61), ("q8", 2400, 768, 200, 44, 69), ("q8", 4001, 256, 64, 41, 31),
    ("q8", 2400, 512, 200, 46, 59), ("q8", 1831, 384, 128, 41, 30), ("q8", 915, 1024, 128, 39, 37),
    ("q8", 28089, 100, 32, 54, 44), ("q8", 7959, 333, 32, 54, 33), ("q8", 12203, 333, 32, 54, 37),
    ("q8", 25475, 480, 8, 54, 43), ("q8", 11683, 600, 32, 59, 45), ("q8", 17889, 600, 32, 59, 55),
    ("q8", 12191, 1000, 32, 62, 55), ("q8", 3047, 1000, 128, 45, 55), ("q8", 19905, 1000, 32, 63, 73),
    ("q8", 5477, 600, 32, 58, 35), ("q8", 16219, 900, 8, 56, 37), ("q8", 3311, 900, 128, 46, 56),
    ("q4", 39877, 128, 32, 56, 39), ("q4", 83221, 480, 8, 63, 59), ("q4", 49079, 992, 8, 79, 61),
    ("q4", 156251, 384, 8, 69, 84), ("q4", 24415, 768, 32, 67, 90), ("q4", 3739, 768, 128, 48, 69),
    ("q4", 2400, 256, 300, 74, 42), ("q4", 1200, 768, 300, 51, 66), ("q4", 1200, 1024, 300, 59, 97),
]


@pytest.mark.parametrize("fmt,n,d,nq,passes,stream", TIMED)
def test_the_streaming_line_follows_the_times(lib, fmt, n, d, nq, passes, stream):
    assert bool(lib.stream(fmt == "q8", n, d, nq)) == (stream < passes)

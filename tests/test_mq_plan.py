"""The row ranges of the multi-query passes (manta_amd/csrc/mq_plan.hpp),
walked on the CPU as the kernels walk them: the passes cover every row once,
and every chunk's copy of q4 block scales (4 bytes at a time) starts on a word
and stays inside the allocation, whatever the block count of a row."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from manta_amd import synth
from oracle import oracle as orc

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "manta_amd", "csrc")

DRIVER = r"""
#include "mq_plan.hpp"
extern "C" int plan(int64_t n, int64_t k, int chunk, int groups, int wgs, int wide, int shadow, int64_t* out) {
    const auto p = manta::mq_topk_passes(n, k, chunk, groups, wgs, wide != 0, shadow != 0);
    for (size_t i = 0; i < p.size(); i++) {
        const int64_t v[4] = {p[i].begin, p[i].end, p[i].rows_per_wg, p[i].R};
        for (int j = 0; j < 4; j++) out[4 * i + j] = v[j];
    }
    return (int)p.size();
}
extern "C" int scale_limit(int left, int nb) { return manta::mq4_scale_limit(left, nb); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("mq_plan")
    src, so = d / "plan.cpp", d / "plan.so"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-fPIC", "-shared", "-I" + CSRC, str(src), "-o",
                    str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.plan.argtypes = [C.c_int64, C.c_int64, C.c_int, C.c_int, C.c_int, C.c_int, C.c_int, C.POINTER(C.c_int64)]
    return lib


def _passes(lib, n, k, chunk, groups, wide=0, shadow=0):
    buf = (C.c_int64 * 256)()
    count = lib.plan(n, k, chunk, groups, 256 if wide else 512, wide, shadow, buf)
    return [tuple(buf[4 * i:4 * i + 4]) for i in range(count)]


SIZES = [1, 31, 4095, 4096, 4097, 35055, 60001, 100003, 262147, 300000, 524288, 1048575, 4194304]
KS = [1, 7, 50, 129, 500, 513, 1031, 2048]


@pytest.mark.parametrize("wide,shadow,chunk", [(0, 0, 32), (0, 0, 64), (0, 0, 128), (1, 0, 64), (1, 0, 128),
                                               (1, 1, 64), (1, 1, 128)])
def test_passes_cover_the_rows_in_whole_chunks(lib, wide, shadow, chunk):
    for n in SIZES:
        for k in KS:
            if k > n:
                continue
            for groups in (1, 3, 64):
                passes = _passes(lib, n, k, chunk, groups, wide, shadow)
                at = 0
                for begin, end, per, R in passes:
                    assert begin == at and end > begin
                    assert begin % chunk == 0, (n, k, passes)
                    assert per % chunk == 0 and (R - 1) * per < end - begin <= R * per
                    at = end
                assert at == n


@pytest.mark.parametrize("chunk", [32, 64, 128])
def test_q4_scale_copies_stay_aligned_and_inside(lib, chunk):
    for n in SIZES:
        if n > 600000:
            continue
        for nb in (1, 2, 3, 5, 7, 12, 15, 31):
            allocated = (n * nb * 2 + 3) // 4 * 4
            for k in (129, 500):
                if k > n:
                    continue
                for begin, end, per, R in _passes(lib, n, k, chunk, 1):
                    for w in range(R):
                        r0 = begin + w * per
                        r1 = min(r0 + per, end)
                        for c0 in {r0, r1 - ((r1 - r0 - 1) % chunk + 1)}:  # its first and last chunk
                            left = min(chunk, r1 - c0)
                            first = c0 * nb * 2
                            last = first + lib.scale_limit(left, nb)
                            assert first % 4 == 0, (n, nb, k, begin, c0)
                            assert first <= last and last + 4 <= allocated, (n, nb, k, begin, c0)
                            assert last + 4 >= (c0 + left) * nb * 2  # the copy holds every row's


@pytest.mark.gpu
@pytest.mark.parametrize("nq,n,d,k", [(16, 300000, 96, 500), (9, 200001, 480, 500)])
def test_q4_odd_block_counts_over_three_passes(rt, nq, n, d, k):
    """Row counts whose prefixes would grow to odd row numbers."""
    q = synth.normal_f16(61, d, nq, d, 1.0)
    packed, scales = synth.q4_rows(61, 1000 + d, n, d)
    cands = rt.bind_q4(packed, scales, d)
    rt.set_timing(True)
    rt.timing(reset=True)
    ids, sc, _ = rt.score_topk(cands, "l2_distance", rt.to_device(q), k, smallest=True, quantized=True)
    passes = rt.timing("mq_select")[0]
    rt.set_timing(False)
    assert passes == 3
    want_scores = orc.score_q4("l2_distance", q, packed, scales, d)
    want = orc.topk(want_scores, k, smallest=True)
    np.testing.assert_array_equal(ids.download(), want)
    np.testing.assert_array_equal(sc.download(), np.take_along_axis(want_scores, want, 1))
    cands.close()

"""The reference score matrix's tiles and the candidates' rescore at their
edges, bit for bit against the oracle's sequential sums: rows and queries
around every tile size, row widths around the staged columns, queries whose
squares span more than f64 holds exactly, zero rows and queries, ties.
"""
import numpy as np
import pytest

from manta_amd import synth
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

OPS = ["dot", "cosine", "l2_distance"]


def _queries(seed, nq, d):
    q = synth.normal_f16(700 + seed, 0, nq, d, 1.0, normalize=False).reshape(nq, d).copy()
    # one of subnormals and large values side by side, one of zeros
    wide = q[0].view(np.float16)
    wide[:] = np.where(np.arange(d) % 3 == 0, wide * np.float16(500), wide * np.float16(6e-5))
    if nq > 2:
        q[2] = 0
    return q


def _bind(rt, fmt, seed, n, d, sets=1):
    pack = synth.q8_rows if fmt == "q8" else synth.q4_rows
    parts = [pack(700 + seed, 1 + s, n, d, normalize=False) for s in range(sets)]
    codes = np.stack([np.asarray(p[0]).reshape(n, -1) for p in parts])
    scales = np.stack([np.asarray(p[1]).reshape((n,) if fmt == "q8" else (n, -1)) for p in parts])
    codes[:, n // 2] = 0           # a zero row
    if n > 4:
        codes[:, 1] = codes[:, 0]  # a tie
        scales[:, 1] = scales[:, 0]
    if sets == 1:
        codes, scales = codes[0], scales[0]
    return rt.bind_q8(codes, scales) if fmt == "q8" else rt.bind_q4(codes, scales, d), codes, scales


def _want(fmt, op, q, codes, scales):
    if fmt == "q8":
        return orc.ref_score_q8(op, q, codes, scales)
    return orc.ref_score_q4(op, q, codes, scales, q.shape[1])


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("fmt,d", [("q8", 1), ("q8", 17), ("q8", 64), ("q8", 129), ("q8", 1024),
                                   ("q4", 32), ("q4", 96), ("q4", 1024)])
@pytest.mark.parametrize("nq,n", [(1, 1), (1, 257), (2, 63), (4, 65), (5, 33), (8, 32), (9, 255), (17, 64)])
def test_score_matrix_small_tiles(rt, op, fmt, d, nq, n):
    q = _queries(d + nq, nq, d)
    cands, codes, scales = _bind(rt, fmt, d + nq, n, d)
    got = rt.score(cands, op, rt.to_device(q)).download()
    np.testing.assert_array_equal(got, _want(fmt, op, q, codes, scales))
    cands.close()


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("fmt,d,nq,n", [("q8", 33, 1, 65537), ("q4", 64, 1, 40001), ("q4", 32, 2, 20000),
                                        ("q8", 1024, 5, 104861), ("q8", 100, 8, 65536), ("q4", 96, 7, 75001),
                                        ("q8", 1024, 16, 32769), ("q8", 65, 9, 58303), ("q4", 160, 19, 30001),
                                        ("q8", 300, 1, 262147), ("q4", 1024, 9, 60001),
                                        ("q8", 960, 12, 43691)])
def test_score_matrix_large_tiles(rt, op, fmt, d, nq, n):
    """Checked on the first and last rows and a stretch of the middle."""
    q = _queries(d + nq, nq, d)
    cands, codes, scales = _bind(rt, fmt, d + nq, n, d)
    got = rt.score(cands, op, rt.to_device(q)).download()
    for lo in (0, n // 2 - 150, n - 300):
        at = slice(lo, lo + 300)
        np.testing.assert_array_equal(got[:, at], _want(fmt, op, q, codes[at], scales[at]))
    cands.close()


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("d,n", [(40, 130), (256, 23000)])
def test_score_matrix_sets(rt, op, d, n):
    """A set per query: below and above the one-row-a-thread line."""
    q = _queries(d, 3, d)
    cands, codes, scales = _bind(rt, "q8", d, n, d, sets=3)
    got = rt.score(cands, op, rt.to_device(q)).download()
    for j in range(3):
        for at in (slice(0, 130), slice(n - 130, n)):
            np.testing.assert_array_equal(got[j, at], _want("q8", op, q[j:j + 1], codes[j, at], scales[j, at])[0])
    cands.close()


@pytest.mark.parametrize("op", OPS)
@pytest.mark.parametrize("fmt,d", [("q8", 24), ("q8", 384), ("q8", 1024), ("q4", 32), ("q4", 416), ("q4", 1024)])
@pytest.mark.parametrize("nq,k", [(1, 1), (3, 9), (5, 100)])
def test_rescored_candidates(rt, op, fmt, d, nq, k):
    n = 3000
    q = _queries(d + nq, nq, d)
    cands, codes, scales = _bind(rt, fmt, d + nq, n, d)
    want = _want(fmt, op, q, codes, scales)
    smallest = op == "l2_distance"
    ids, sc, _ = rt.score_topk(cands, op, rt.to_device(q), k, smallest=smallest)
    want_ids = orc.topk(want, k, smallest=smallest)
    np.testing.assert_array_equal(ids.download(), want_ids)
    np.testing.assert_array_equal(sc.download(), np.take_along_axis(want, want_ids, 1))
    cands.close()


@pytest.mark.parametrize("fmt,op,d,nq,k", [("q8", "dot", 100, 130, 200), ("q8", "dot", 1024, 90, 300),
                                           ("q8", "cosine", 40, 90, 100), ("q8", "cosine", 128, 130, 256),
                                           ("q8", "l2_distance", 24, 100, 150), ("q8", "l2_distance", 100, 140, 300),
                                           ("q4", "dot", 96, 1, 1), ("q4", "dot", 1024, 9, 260),
                                           ("q4", "cosine", 160, 140, 220), ("q4", "l2_distance", 64, 190, 230)])
def test_many_rescored_candidates(rt, fmt, op, d, nq, k):
    """Past the line where a row a thread rescores them."""
    n = 1500
    q = _queries(d + nq, nq, d)
    cands, codes, scales = _bind(rt, fmt, d + nq, n, d)
    want = _want(fmt, op, q, codes, scales)
    smallest = op == "l2_distance"
    ids, sc, _ = rt.score_topk(cands, op, rt.to_device(q), k, smallest=smallest)
    want_ids = orc.topk(want, k, smallest=smallest)
    np.testing.assert_array_equal(ids.download(), want_ids)
    np.testing.assert_array_equal(sc.download(), np.take_along_axis(want, want_ids, 1))
    cands.close()

"""GPU parity of the quantized-query scans over row widths and selection paths
that the config-shaped tests do not reach: rows of any number of 16-byte
pieces (q8) or blocks (q4), streamed a query at a time or through the
multi-query kernels (k past 192 always takes those with 8 or more queries),
and the buffered selection of the streaming scans (k <= 192; on fixed-width q8
rows past the lists' k) on tied and
clustered rows.  Bar: ids and scores bit-exact with the oracle."""
import numpy as np
import pytest

from manta_amd import synth
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _check(rt, cands, want_scores, op, q, k):
    smallest = op == "l2_distance"
    ids, sc, _ = rt.score_topk(cands, op, rt.to_device(q), k, smallest=smallest, quantized=True)
    want = orc.topk(want_scores, k, smallest=smallest)
    np.testing.assert_array_equal(ids.download(), want)
    np.testing.assert_array_equal(sc.download(), np.take_along_axis(want_scores, want, 1))


@pytest.mark.parametrize("nq,k", [(2, 5), (3, 100), (9, 200)])
@pytest.mark.parametrize("op", ["dot", "cosine", "l2_distance"])
@pytest.mark.parametrize("d", [8, 24, 40, 100, 333, 520, 600, 768, 900, 1024])
def test_q8_row_widths(rt, d, op, nq, k):
    n = 2777
    q = synth.normal_f16(51, d, nq, d, 1.0)
    codes, scales = synth.q8_rows(51, 1000 + d, n, d)
    cands = rt.bind_q8(codes, scales)
    want = orc.score_q8(op, q, codes, scales)
    _check(rt, cands, want, op, q, k)
    if nq == 9:
        got = rt.score(cands, op, rt.to_device(q), quantized=True).download()
        np.testing.assert_array_equal(got, want)
    cands.close()


@pytest.mark.parametrize("nq,k", [(1, 20), (2, 150), (17, 200)])
@pytest.mark.parametrize("op", ["dot", "cosine", "l2_distance"])
@pytest.mark.parametrize("d", [32, 96, 160, 224, 416, 544, 800, 1024])
def test_q4_row_widths(rt, d, op, nq, k):
    n = 3001  # odd: with an odd number of blocks the scales end half way through a word
    q = synth.normal_f16(52, d, nq, d, 1.0)
    packed, scales = synth.q4_rows(52, 1000 + d, n, d)
    cands = rt.bind_q4(packed, scales, d)
    want = orc.score_q4(op, q, packed, scales, d)
    _check(rt, cands, want, op, q, k)
    if nq == 17:
        got = rt.score(cands, op, rt.to_device(q), quantized=True).download()
        np.testing.assert_array_equal(got, want)
    cands.close()


@pytest.mark.parametrize("rows", ["tied", "ascending", "clustered"])
@pytest.mark.parametrize("fmt", ["q8", "q8_wide", "q4"])
@pytest.mark.parametrize("n,k", [(200, 192), (5000, 65), (70000, 100), (300000, 192)])
def test_buffered_selection(rt, fmt, rows, n, k):
    """Rows all equal, best last, or the best ones in one thread's slots."""
    d = 160 if fmt == "q8_wide" else 128
    rng = np.random.default_rng(n + k)
    q = synth.normal_f16(53, 0, 1, d, 1.0)
    base = rng.integers(-100, 101, size=d).astype(np.int8)
    f = np.full(n, 0.5, np.float32)
    if rows == "ascending":
        f = np.linspace(0.01, 1.0, n, dtype=np.float32)
    elif rows == "clustered":
        f = np.where(np.arange(n) % 256 == 7, np.float32(1.0) + np.arange(n, dtype=np.float32) / n, np.float32(0.25))
    if fmt == "q4":
        codes = np.clip(base // 15, -7, 7).astype(np.int8)
        nib = (codes.view(np.uint8) & 15)
        packed = np.broadcast_to(nib[0::2] | (nib[1::2] << 4), (n, d // 2)).copy()
        scales = np.repeat(f.astype(np.float16).view(np.uint16)[:, None], d // 32, axis=1)
        cands = rt.bind_q4(packed, scales, d)
        want = orc.score_q4("dot", q, packed, scales, d)
    else:
        codes = np.broadcast_to(base, (n, d)).copy()
        cands = rt.bind_q8(codes, f.astype(np.float32))
        want = orc.score_q8("dot", q, codes, f.astype(np.float32))
    _check(rt, cands, want, "dot", q, min(k, n))
    cands.close()


def _tiled_rows(rows, n):
    """n rows that repeat `rows` with scales of their own, so that the oracle
    scores few rows and the device reads many."""
    return np.tile(rows, (-(-n // len(rows)), 1))[:n]


@pytest.mark.parametrize("op,k", [("dot", 12), ("cosine", 100), ("l2_distance", 250)])
@pytest.mark.parametrize("fmt,d,nq,n", [("q8", 100, 4, 500001), ("q8", 500, 1, 530001), ("q8", 840, 1, 330001),
                                        ("q4", 256, 1, 1050001), ("q4", 416, 2, 90001), ("q4", 1024, 3, 22001)])
def test_rows_in_pieces(rt, fmt, d, nq, n, op, k):
    """Past the line where a row per lane streams them (the widths above are
    below it), in pieces of 16 bytes."""
    rng = np.random.default_rng(d)
    q = synth.normal_f16(54, d, nq, d, 1.0)
    if fmt == "q8":
        codes = _tiled_rows(rng.integers(-127, 128, (20011, d), dtype=np.int8), n)
        scales = rng.uniform(0.5, 1.5, n).astype(np.float32) / np.float32(127 * 30)
        cands = rt.bind_q8(codes, scales)
        want = orc.score_q8(op, q, codes, scales)
    else:
        nib = rng.integers(-7, 8, (20011, d), dtype=np.int8).view(np.uint8) & 15
        packed = _tiled_rows(nib[:, 0::2] | (nib[:, 1::2] << 4), n)
        scales = (rng.uniform(0.5, 1.5, (n, d // 32)) / 200).astype(np.float16).view(np.uint16)
        cands = rt.bind_q4(packed, scales, d)
        want = orc.score_q4(op, q, packed, scales, d)
    _check(rt, cands, want, op, q, k)
    cands.close()


@pytest.mark.parametrize("sets,n,k", [(3, 300, 64), (64, 500, 20), (20, 6000, 21), (20, 6000, 22), (2, 256, 33)])
def test_q8_lists_of_few_parts(rt, sets, n, k):
    """Lists and buffered selections on both sides of the line, a set each."""
    d = 128
    codes = np.empty((sets, n, d), np.int8)
    scales = np.empty((sets, n), np.float32)
    for s in range(sets):
        codes[s], scales[s] = synth.q8_rows(55, 1 + s, n, d)
    codes[:, n // 2:] = codes[:, :n - n // 2]  # ties
    q = synth.normal_f16(55, 0, sets, d, 1.0)
    cands = rt.bind_q8(codes, scales)
    _check(rt, cands, orc.score_q8("dot", q, codes, scales), "dot", q, k)
    cands.close()

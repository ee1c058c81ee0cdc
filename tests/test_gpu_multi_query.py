"""GPU parity of the multi-query passes where they are the route: every K-step
and block count of the kernels at their exact row width and on shorter rows,
over a first pass and at least two that append above a threshold, in each
query-group shape; rows ordered worst first (regions fill and are compacted);
and shapes of few queries whose work is past the streaming scans' line.

Bar: ids and scores bit-exact.  The wide sweeps compare every query with the
streaming scans (fewer than 8 queries a call: other kernels, held to the oracle
by tests/test_gpu_scan_shapes.py) and two queries with the oracle; the others
compare with the oracle alone.  Each test asserts the launches it is about."""
import numpy as np
import pytest

from manta_amd import synth
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


class Launches:
    """Launch counts of a block of calls, by kernel family."""

    def __init__(self, rt):
        self.rt = rt

    def __enter__(self):
        self.rt.set_timing(True)
        self.rt.timing(reset=True)
        return self

    def __exit__(self, *exc):
        self.selects = self.rt.timing("mq_select")[0]
        self.scans = self.rt.timing("q8_scan")[0] + self.rt.timing("q4_scan")[0]
        self.rt.set_timing(False)


def _topk(rt, cands, op, q, k, smallest, quantized=True):
    ids, sc, _ = rt.score_topk(cands, op, rt.to_device(q), k, smallest=smallest, quantized=quantized)
    return ids.download(), sc.download()


def _check(rt, cands, op, q, k, smallest, want_s, quantized=True, passes=None):
    with Launches(rt) as n:
        ids, sc = _topk(rt, cands, op, q, k, smallest, quantized)
    assert n.scans == 0 and n.selects >= (passes or 1), (n.scans, n.selects)
    want = orc.topk(want_s, k, smallest=smallest)
    np.testing.assert_array_equal(ids, want)
    np.testing.assert_array_equal(sc, np.take_along_axis(want_s, want, 1))


def _sweep(rt, cands, q, ops, k, oracle):
    """9, 65 and 130 queries (each group shape of the kernels), one op each."""
    for nq, op in zip((9, 65, 130), ops):
        smallest = op == "l2_distance"
        with Launches(rt) as n:
            ids, sc = _topk(rt, cands, op, q[:nq], k, smallest)
        assert n.scans == 0 and n.selects >= 3, (nq, op, n.scans, n.selects)
        for a in range(0, nq, 7):
            with Launches(rt) as n:
                want_ids, want_sc = _topk(rt, cands, op, q[a:min(nq, a + 7)], k, smallest)
            assert n.scans == 1 and n.selects == 0, (nq, op, n.scans, n.selects)
            np.testing.assert_array_equal(ids[a:a + 7], want_ids, err_msg="%d %s" % (nq, op))
            np.testing.assert_array_equal(sc[a:a + 7], want_sc, err_msg="%d %s" % (nq, op))
        pick = [0, nq - 1]
        want_s = oracle(op, q[pick])
        want = orc.topk(want_s, k, smallest=smallest)
        np.testing.assert_array_equal(ids[pick], want)
        np.testing.assert_array_equal(sc[pick], np.take_along_axis(want_s, want, 1))


OPS = ["dot", "cosine", "l2_distance"]
ROWS, K = 150001, 500  # 4,096 rows, then two growth passes


@pytest.mark.parametrize("i,d", enumerate([64, 40, 128, 100, 256, 200, 384, 333, 512, 480, 768, 600, 1024, 1000]))
def test_q8_widths_over_three_passes(rt, i, d):
    """Each K-step count, at its exact width and on shorter rows."""
    rng = np.random.default_rng(d)
    codes = rng.integers(-127, 128, (ROWS, d), dtype=np.int8)
    scales = rng.uniform(0.5, 1.5, ROWS).astype(np.float32) / (127 * np.sqrt(d)).astype(np.float32)
    q = synth.normal_f16(71, d, 130, d, 1.0)
    cands = rt.bind_q8(codes, scales)
    _sweep(rt, cands, q, [OPS[(i // 2 + j) % 3] for j in range(3)], K,
           lambda op, qs: orc.score_q8(op, qs, codes, scales))
    cands.close()


@pytest.mark.parametrize("i,nb", enumerate([1, 2, 4, 3, 8, 5, 12, 9, 16, 13, 24, 17, 32, 25]))
def test_q4_widths_over_three_passes(rt, i, nb):
    """Each block count, at its exact width and on shorter rows (odd counts:
    a row's scales then end half way through a word)."""
    d = 32 * nb
    rng = np.random.default_rng(nb)
    codes = rng.integers(-7, 8, (ROWS, d), dtype=np.int8).view(np.uint8) & 15
    packed = codes[:, 0::2] | (codes[:, 1::2] << 4)
    scales = (rng.uniform(0.5, 1.5, (ROWS, nb)) / (7 * np.sqrt(d))).astype(np.float16).view(np.uint16)
    q = synth.normal_f16(72, d, 130, d, 1.0)
    cands = rt.bind_q4(packed, scales, d)
    _sweep(rt, cands, q, [OPS[(i // 2 + j) % 3] for j in range(3)], K,
           lambda op, qs: orc.score_q4(op, qs, packed, scales, d))
    cands.close()


@pytest.mark.parametrize("nq", [24, 130])
@pytest.mark.parametrize("fmt,d", [("q8", 333), ("q8", 1000), ("q4", 160), ("q4", 416)])
def test_worst_first_rows_of_short_widths(rt, fmt, d, nq):
    """One row's codes under scales that grow with the index: every pass lets
    the later rows through, so regions fill and are compacted."""
    n, k = 60001, 300
    rng = np.random.default_rng(d)
    base = rng.standard_normal(d)
    q = orc.f32_to_f16((base + 0.05 * rng.standard_normal((nq, d))).astype(np.float32))
    grow = 1.0 + np.arange(n, dtype=np.float64) / n
    if fmt == "q8":
        codes1, s1 = orc.pack_q8_rows((base / np.linalg.norm(base)).astype(np.float32).reshape(1, -1))
        codes, scales = np.repeat(codes1, n, axis=0), (s1[0] * grow).astype(np.float32)
        cands = rt.bind_q8(codes, scales)
        want_s = orc.score_q8("dot", q, codes, scales)
    else:
        packed1, s1 = orc.pack_q4_blocks(base.astype(np.float32).reshape(1, -1))
        packed = np.repeat(packed1, n, axis=0)
        scales = orc.f32_to_f16((orc.f16_to_f32(s1) * grow[:, None]).astype(np.float32))
        cands = rt.bind_q4(packed, scales, d)
        want_s = orc.score_q4("dot", q, packed, scales, d)
    _check(rt, cands, "dot", q, k, False, want_s, passes=2)
    cands.close()


# Shapes past the line where the streaming scans are faster: k within their
# reach, a growth pass in each.

@pytest.mark.parametrize("op,smallest", [("dot", False), ("cosine", False), ("l2_distance", True),
                                         ("dot", True), ("l2_distance", False)])
@pytest.mark.parametrize("nq,n,d,k", [(8, 200001, 128, 10), (33, 30000, 384, 50), (40, 33000, 256, 100),
                                      (64, 33333, 64, 1)])
def test_q8_topk_past_the_streaming_line(rt, op, smallest, nq, n, d, k):
    q = synth.normal_f16(73, d, nq, d, 1.0, normalize=op != "l2_distance")
    codes, scales = synth.q8_rows(73, 1000 + d, n, d, normalize=op != "l2_distance")
    cands = rt.bind_q8(codes, scales)
    _check(rt, cands, op, q, k, smallest, orc.score_q8(op, q, codes, scales), passes=2)
    if (op, smallest) in (("cosine", False), ("l2_distance", True)):
        # the reference arithmetic on the rows the passes rank
        _check(rt, cands, op, q, k, smallest, orc.ref_score_q8(op, q, codes, scales), quantized=False, passes=2)
    cands.close()


@pytest.mark.parametrize("op,smallest", [("cosine", False), ("l2_distance", True), ("dot", False), ("dot", True)])
@pytest.mark.parametrize("nq,n,d,k", [(8, 270001, 32, 10), (37, 45000, 128, 50), (129, 9001, 384, 100),
                                      (9, 230000, 64, 1)])
def test_q4_topk_past_the_streaming_line(rt, op, smallest, nq, n, d, k):
    q = synth.normal_f16(74, d, nq, d, 1.0, normalize=op != "l2_distance")
    packed, scales = synth.q4_rows(74, 1000 + d, n, d, normalize=op != "l2_distance")
    cands = rt.bind_q4(packed, scales, d)
    _check(rt, cands, op, q, k, smallest, orc.score_q4(op, q, packed, scales, d), passes=2)
    cands.close()


@pytest.mark.parametrize("op,smallest", [("dot", False), ("cosine", False), ("l2_distance", True),
                                         ("cosine", True), ("l2_distance", False)])
def test_zero_rows_and_a_partial_group(rt, op, smallest):
    """All-zero rows (cosine's zero denominator) among normal ones, with a
    query count that leaves most of the last query group empty: the empty
    slots never append keys, and zero rows score like the oracle's."""
    nq, n, d, k = 19, 90000, 128, 40
    q = synth.normal_f16(75, 0, nq, d, 1.0, normalize=op != "l2_distance")
    codes, scales = synth.q8_rows(75, 1, n, d, normalize=op != "l2_distance")
    codes, scales = codes.copy(), scales.copy()
    zero = np.arange(0, n, 7)
    codes[zero] = 0
    scales[zero[::2]] = 0.0
    cands = rt.bind_q8(codes, scales)
    _check(rt, cands, op, q, k, smallest, orc.score_q8(op, q, codes, scales), passes=2)
    cands.close()


def test_repeated_calls_start_afresh(rt):
    """Thresholds and counts are reset between calls: a second call with
    fewer rows matches the oracle too."""
    for n, nq in ((200000, 12), (60000, 32)):
        q = synth.normal_f16(76, n, nq, 128, 1.0)
        codes, scales = synth.q8_rows(76, 1, n, 128)
        cands = rt.bind_q8(codes, scales)
        _check(rt, cands, "l2_distance", q, 100, True, orc.score_q8("l2_distance", q, codes, scales), passes=2)
        cands.close()


def test_small_calls_build_no_shadow(rt):
    """A q4 call of many queries that streams leaves the bound matrix as it
    is; the first one past the line builds the shadow and keeps it."""
    d, k = 64, 10
    q = synth.normal_f16(77, 0, 256, d, 1.0, normalize=True)
    for n, built in ((3000, False), (12000, True)):
        packed, scales = synth.q4_rows(77, 1, n, d, normalize=True)
        cands = rt.bind_q4(packed, scales, d)
        before = rt.stats()["candidate_bytes"]
        ids, sc = _topk(rt, cands, "cosine", q, k, False)
        want_s = orc.score_q4("cosine", q, packed, scales, d)
        want = orc.topk(want_s, k)
        np.testing.assert_array_equal(ids, want)
        np.testing.assert_array_equal(sc, np.take_along_axis(want_s, want, 1))
        assert (rt.stats()["candidate_bytes"] > before) == built, n
        cands.close()

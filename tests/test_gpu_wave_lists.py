"""GPU parity at the largest part counts: the register lists for 16 < k <= 64, which the
streaming q8 scan takes where a query's parts are too many for the merge by a
floor and ranks (more than 512 workgroups of 64 rounds: over 8,388,608 rows)."""
import numpy as np
import pytest

from manta_amd import synth
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rows():
    n, d = 8388608 + 20001, 64  # 514 parts, the last one partial
    rng = np.random.default_rng(81)
    codes = rng.integers(-127, 128, (n, d), dtype=np.int8)
    scales = rng.uniform(0.5, 1.5, n).astype(np.float32) / np.float32(1016)
    return codes, scales


@pytest.mark.parametrize("op,k", [("dot", 17), ("dot", 64), ("cosine", 40), ("l2_distance", 33)])
def test_lists_of_many_parts(rt, rows, op, k):
    codes, scales = rows
    q = synth.normal_f16(81, 0, 1, codes.shape[1], 1.0)
    cands = rt.bind_q8(codes, scales)
    smallest = op == "l2_distance"
    ids, sc, _ = rt.score_topk(cands, op, rt.to_device(q), k, smallest=smallest, quantized=True)
    want_s = orc.score_q8(op, q, codes, scales)
    want = orc.topk(want_s, k, smallest=smallest)
    np.testing.assert_array_equal(ids.download(), want)
    np.testing.assert_array_equal(sc.download(), np.take_along_axis(want_s, want, 1))
    cands.close()


@pytest.mark.parametrize("d", [64, 48])
def test_buffered_selection_of_the_most_parts(rt, rows, d):
    """512 parts of 64 rounds, the largest query the buffered selection takes
    (the fixed-width kernel, and the one of any width)."""
    codes, scales = np.ascontiguousarray(rows[0][:8388608, :d]), rows[1][:8388608]
    k = 192
    q = synth.normal_f16(82, 0, 1, d, 1.0)
    cands = rt.bind_q8(codes, scales)
    ids, sc, _ = rt.score_topk(cands, "dot", rt.to_device(q), k, quantized=True)
    want_s = orc.score_q8("dot", q, codes, scales)
    want = orc.topk(want_s, k)
    np.testing.assert_array_equal(ids.download(), want)
    np.testing.assert_array_equal(sc.download(), np.take_along_axis(want_s, want, 1))
    cands.close()

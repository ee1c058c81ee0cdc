"""GPU parity of the score-matrix top-k (manta_rocm_topk) with the oracle's
topKTensor: ids equal, values bit-exact (keys are a total order, so there is
no tolerance), over segment edges, ties, sorted rows and rows whose best
scores all sit in few threads (the reservoir behind the one-launch path)."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _rows(kind, rows, cols, seed):
    rng = np.random.default_rng(seed)
    s = rng.standard_normal((rows, cols)).astype(np.float32)
    if kind == "ties":
        s = np.round(s)  # few values, -0 and +0 among them
    elif kind == "ascending":
        s = np.sort(s, axis=1)
    elif kind == "equal":
        s[:] = 0.25
    elif kind == "clustered":
        # the columns of the first 99 threads (four in a row of every 1,024) above all others
        c = np.arange(cols)
        s[:, (c % 1024) // 4 < 99] += 100.0
    return np.ascontiguousarray(s)


@pytest.mark.parametrize("smallest", [False, True])
@pytest.mark.parametrize("kind", ["normal", "ties", "ascending", "equal", "clustered"])
@pytest.mark.parametrize("rows,cols,k", [
    (1, 1, 1), (3, 255, 192), (2, 257, 193), (5, 4096, 100), (1, 4097, 1), (7, 8193, 150),
    # 32 and 64 scores a thread, and rows whose length is not a multiple of 4
    (200, 50000, 10), (130, 60001, 100), (700, 16384, 100), (2, 300000, 192), (1, 70001, 700)])
def test_topk_rows(rt, rows, cols, k, kind, smallest):
    if rows * cols > 2000000 and kind not in ("normal", "clustered"):
        rows = 3
    s = _rows(kind, rows, cols, cols + k)
    ids, vals = rt.topk(rt.to_device(s), k, smallest=smallest)
    want = orc.topk(s, k, smallest=smallest)
    np.testing.assert_array_equal(ids.download(), want)
    np.testing.assert_array_equal(vals.download(), np.take_along_axis(s, want, 1) + np.float32(0))

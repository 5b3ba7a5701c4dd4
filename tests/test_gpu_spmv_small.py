"""SpMV of few entries (the merge path's one-launch form): row lengths
around a lane group's share, rows that the workgroup adds up together, empty
rows, and entry counts on both sides of the limit, against the FP64 oracle."""
import numpy as np
import pytest

import oracle
from taco_amd import _lib
from taco_amd import workloads as W
from tests import gpu_util as G

pytestmark = pytest.mark.gpu
LIMIT = 1 << 16
TOL = {"f64": 1e-12, "f32": 1e-5}


def _counts(name):
    rng = np.random.default_rng(3)
    if name == "one_row":
        return [5000]
    if name == "one_row_all":
        return [LIMIT]
    if name == "empty":
        return [0] * 77
    if name == "edges":  # mean near 8: 4 lanes a row, 64 entries a row's own
        return list(rng.choice([0, 1, 3, 4, 5, 15, 16, 17], 700)) + [63, 64, 65, 257, 4096, 4097]
    if name == "long_rows":
        return list(rng.choice([1, 2, 2000], 61))
    if name == "wide_rows":  # 64 lanes a row
        return list(rng.integers(150, 400, 300))
    if name == "at_limit":
        return [8] * (LIMIT // 8)
    return [8] * (LIMIT // 8) + [1]  # over_limit


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("name", ["one_row", "one_row_all", "empty", "edges", "long_rows",
                                  "wide_rows", "at_limit", "over_limit"])
def test_small(name, dtype):
    counts = np.array(_counts(name), np.int32)
    A = W.csr_from_counts(len(counts), LIMIT + 5, counts, 11)
    x = W.uniform(A.n, 12, W.STREAM_X)
    for s in (None, G.sched(_lib.MERGE_PATH, 256, items=16)):
        y = G.spmv(A, x, s, dtype=dtype)
        ye, cond = oracle.exact_spmv(A, x)
        rep = oracle.error_report(y, ye, cond, TOL[dtype])
        assert rep["ok"], rep
    assert np.array_equal(y, G.spmv(A, x, s, dtype=dtype))


def test_unsupported_items_refused():
    A = W.csr_fixed(10, 10, 2, 1)
    with pytest.raises(_lib.TacoHipError):
        G.spmv(A, np.ones(10), G.sched(_lib.MERGE_PATH, 256, items=5))

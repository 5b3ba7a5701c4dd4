"""SpMV of few entries (the merge path's one-launch form): row lengths
around a lane group's share, rows that the workgroup adds up together, empty
rows, and entry counts on both sides of the limit, against the FP64 oracle."""
import numpy as np
import pytest
import torch

import oracle
from taco_amd import _lib, descriptors as D
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


# Row lengths on both sides of the lines between a lane group's own rows and
# those of a team of 16 lanes, a wave and the workgroup, and of the column
# counts up to which the form is taken (16,384 in f64, 24,576 in f32).
SHAPES = {
    "teams": ([2] * 9000 + [31, 32, 33, 34, 64, 65, 128, 129, 255, 256], 16384),
    "waves": ([1] * 9000 + [256, 257, 258, 1023, 1024, 1025, 2047, 2048], 16384),
    "workgroup": ([1] * 9000 + [2048, 2049, 4096, 4097, 8193], 16384),
    "more_than_the_teams": ([33] * 1900 + [0] * 9000, 16384),
    "more_than_the_waves": ([1] * 300 + [257] * 250, 16384),
    "same_workgroup": (([2100] + [1] * 32) * 25, 16384),
    "n_f64": ([16384, 1, 0, 5], 16384),
    "over_n_f64": ([16385, 1, 0, 5], 16385),
    "n_f32": ([24576] * 2 + [1, 0, 5], 24576),
    "over_n_f32": ([24577] * 2 + [1, 0, 5], 24577),
    "tall": ([0, 0, 1, 0, 0, 0, 0, 0] * (1 << 15), 300),
    "over_tall": ([0, 0, 1, 0, 0, 0, 0, 0] * (1 << 15) + [7], 300),
}


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("name", list(SHAPES))
def test_long_rows(name, dtype):
    counts, n = SHAPES[name]
    A = W.csr_from_counts(len(counts), n, np.array(counts, np.int32), 21)
    assert A.nnz <= LIMIT and np.diff(A.pos).max() == max(counts)
    x = W.uniform(A.n, 22, W.STREAM_X)
    y = G.spmv(A, x, None, dtype=dtype)
    ye, cond = oracle.exact_spmv(A, x)
    rep = oracle.error_report(y, ye, cond, TOL[dtype])
    assert rep["ok"], rep
    assert np.array_equal(y, G.spmv(A, x, None, dtype=dtype))


def _microseconds(A, x, sched, calls=100):
    a, xd = G.csr_desc(A), G.dev(x)
    y = torch.empty(A.m, dtype=torch.float64, device="cuda")
    ad, yd = D.dense(xd), D.dense(y)
    L = _lib.lib()
    best = []
    for _ in range(5):
        t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        t0.record()
        for _ in range(calls):
            _lib.check(L.taco_hip_spmv_compute(yd.ptr, a.ptr, ad.ptr, sched))
        t1.record()
        torch.cuda.synchronize()
        best.append(t0.elapsed_time(t1) / calls * 1e3)
    return min(best)


@pytest.mark.parametrize("counts", [[64] * 512 + [3] * 10500, [128] * 512 + [0] * 15000,
                                    [2000] * 30, [40] * 1000 + [1] * 15000],
                         ids=["dense_block", "block_among_empty", "few_long", "many_short_long"])
def test_long_rows_together_keep_their_pace(counts):
    """Long rows side by side are summed side by side: the default schedule
    stays within 4 times an equal split of the entries (0.4 to 0.7 times;
    one after another it was 5 to 90 times)."""
    A = W.csr_from_counts(len(counts), 16384, np.array(counts, np.int32), 31)
    x = W.uniform(A.n, 32, W.STREAM_X)
    split = _microseconds(A, x, G.sched(_lib.NNZ_SPLIT, 256, items=8))
    assert _microseconds(A, x, None) < 4 * split

"""Merge-path SpMM at the edges of its lane layout (columns a lane, lane
groups, lanes left over) and of its teams and carries, in every value form,
against the FP64 oracle."""
import numpy as np
import pytest
import torch

import oracle
from taco_amd import _lib, descriptors as D
from taco_amd import workloads as W
from tests import gpu_util as G

pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-12, "f32": 1e-5, "bf16": 1e-2}


def _matrix():
    """Empty and short rows, rows around a block of 8 .. 64 entries, and
    rows over many teams (runs of more than 16 carries)."""
    counts = np.random.default_rng(5).choice([0, 0, 1, 3, 7, 8, 9, 16, 31, 33, 63, 64, 65, 130], 900)
    counts[[5, 400, 899]] = [6000, 5000, 4500]
    return W.csr_from_counts(900, 7000, counts.astype(np.int32), 6)


@pytest.mark.parametrize("dtype", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 8, 9, 16, 17, 20, 31, 33, 48, 64, 65, 96, 128, 129, 255, 256])
def test_widths(K, dtype):
    A = _matrix()
    B = W.uniform(A.n * K, 7, W.STREAM_B).reshape(A.n, K)
    group = min(64, max(8, 1 << (K - 1).bit_length()))
    for items in (256, 32):
        print(f"merge spmm K={K} {dtype} items={items}", flush=True)
        C = G.spmm(A, B, G.sched(_lib.MERGE_PATH, 256, items=items, group=group), dtype=dtype)
        Ce, cond = oracle.exact_spmm(A, B)
        rep = oracle.error_report(C, Ce, cond, TOL[dtype])
        assert rep["ok"], rep


@pytest.mark.parametrize("K", [16, 33, 64])
def test_infinities_stay_in_their_rows(K):
    """B rows of infinities and NaN reach only the rows that name them."""
    A = _matrix()
    B = W.uniform(A.n * K, 8, W.STREAM_B).reshape(A.n, K)
    bad = np.unique(A.crd)[::97]
    B[bad[::2]] = np.inf
    B[bad[1::2]] = np.nan
    C = G.spmm(A, B, dtype="f32")
    touched = np.zeros(A.m, bool)
    rows = np.repeat(np.arange(A.m), np.diff(A.pos))
    touched[rows[np.isin(A.crd, bad)]] = True
    assert np.isfinite(C[~touched]).all() and not np.isfinite(C[touched]).any()


@pytest.mark.parametrize("K", [3, 64])
def test_no_entries(K):
    A = W.Csr(300, 0, np.zeros(301, np.int32), np.zeros(0, np.int32), np.zeros(0))
    assert not G.spmm(A, np.zeros((0, K))).any()


@pytest.mark.parametrize("group", [8, 16, 32, 64])
@pytest.mark.parametrize("items", [1, 3, 16, 31, 64, 255])
def test_items_of_small_teams(items, group):
    """Items a wave takes for teams of every size, below the default of 256."""
    A = _matrix()
    B = W.uniform(A.n * 6, 10, W.STREAM_B).reshape(A.n, 6)
    C = G.spmm(A, B, G.sched(_lib.MERGE_PATH, 256, items=items, group=group))
    Ce, cond = oracle.exact_spmm(A, B)
    rep = oracle.error_report(C, Ce, cond, TOL["f64"])
    assert rep["ok"], rep


def test_few_items_keep_their_pace():
    """16 items a team of 8 lanes take at most twice as long as the default
    (1.1 times; 3.3 times where a wave took the 16 items of one team)."""
    m, K = 200_000, 4
    A = W.csr_fixed(m, m, 16, 11)
    a = G.csr_desc(A)
    x, c = D.dense(torch.rand(m, K, dtype=torch.float64, device="cuda")), D.dense(
        torch.empty(m, K, dtype=torch.float64, device="cuda"))
    took = []
    for s in (None, G.sched(_lib.MERGE_PATH, 256, items=16, group=8)):
        best = []
        for _ in range(5):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            for _ in range(10):
                _lib.check(_lib.lib().taco_hip_spmm_compute(c.ptr, a.ptr, x.ptr, s))
            t1.record()
            torch.cuda.synchronize()
            best.append(t0.elapsed_time(t1))
        took.append(min(best))
    assert took[1] < 2 * took[0], took


def test_same_result_every_time():
    A = _matrix()
    B = W.uniform(A.n * 40, 9, W.STREAM_B).reshape(A.n, 40)
    first = G.spmm(A, B)
    assert all(np.array_equal(first, G.spmm(A, B)) for _ in range(3))
    torch.cuda.synchronize()

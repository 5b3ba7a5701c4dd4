"""Merge-path SpMM at the edges of its lane layout (columns a lane, lane
groups, lanes left over) and of its teams and carries, in every value form,
against the FP64 oracle."""
import numpy as np
import pytest
import torch

import oracle
from taco_amd import _lib
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


def test_same_result_every_time():
    A = _matrix()
    B = W.uniform(A.n * 40, 9, W.STREAM_B).reshape(A.n, 40)
    first = G.spmm(A, B)
    assert all(np.array_equal(first, G.spmm(A, B)) for _ in range(3))
    torch.cuda.synchronize()

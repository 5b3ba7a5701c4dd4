"""Merge-path corners: matrices whose rows are far from alike, so that the
corner search's first guess is far off, on both sides of the row count up to
which it guesses; rows over many tiles (carries added by a wave)."""
import numpy as np
import pytest

import oracle
from taco_amd import _lib
from taco_amd import workloads as W
from tests import gpu_util as G

pytestmark = pytest.mark.gpu
ROWS = 1 << 19


def _counts(name):
    if name == "front":  # every entry in the first rows, the rest empty
        c = np.zeros(ROWS, np.int32)
        c[:300] = 1000
    elif name == "back":
        c = np.zeros(ROWS, np.int32)
        c[-300:] = 1000
    elif name == "middle":
        c = np.ones(100_000, np.int32)
        c[50_000:50_003] = 60_000  # some 29 tiles each
    elif name == "above":  # one row past the guessing range
        c = np.ones(ROWS + 1, np.int32)
        c[7] = 70_000
    elif name == "run_lengths":  # runs of 7 .. 66 carries
        c = np.repeat(np.array([14_000, 16_400, 18_500, 20_500, 131_000, 135_000], np.int32), 2)
    elif name == "wave_edges":  # carry runs that end and start at slots 63, 64, 65 of 512 items
        t = 512
        c = np.array([64 * t - 1, 64 * t - 1, 63 * t - 1, 2 * t, t, 65 * t + 3, 0, 128 * t - 8, 9 * t,
                      16 * t, 5, 129 * t], np.int32)
    else:  # few rows
        c = np.array([40_000, 0, 0, 40_000], np.int32)
    return c


@pytest.mark.parametrize("dtype,tol", [("f64", 1e-12), ("f32", 1e-5)])
@pytest.mark.parametrize("name", ["front", "back", "middle", "above", "run_lengths", "few",
                                  "wave_edges"])
def test_corners(name, dtype, tol):
    counts = _counts(name)
    A = W.csr_from_counts(len(counts), 150_000, counts, 21)
    x = W.uniform(A.n, 22, W.STREAM_X)
    ye, cond = oracle.exact_spmv(A, x)
    for items in (2, 8):
        print(f"corners {name} {dtype} items={items}", flush=True)
        y = G.spmv(A, x, G.sched(_lib.MERGE_PATH, 256, items=items), dtype=dtype)
        rep = oracle.error_report(y, ye, cond, tol)
        assert rep["ok"], rep
        assert np.array_equal(y, G.spmv(A, x, G.sched(_lib.MERGE_PATH, 256, items=items), dtype=dtype))

"""SpGEMM rows of more than 64 candidates: every route of the wave-per-row
kernels (flags, bits, register sorts of 2 to 16 values a lane, hash set;
sums by column, by staged and by unstaged search), at the edges between them,
against the oracle: pos and crd bit for bit, and the values too, since every
column sums separately rounded products in encounter order."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from taco_amd import _lib, descriptors as D
from taco_amd import workloads as W
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


def _csr(rows, n, seed):
    pos = np.zeros(len(rows) + 1, np.int32)
    pos[1:] = np.cumsum([len(r) for r in rows])
    crd = np.concatenate([np.asarray(r, np.int64) for r in rows]).astype(np.int32)
    vals = W.uniform(len(crd), seed, W.STREAM_VALS)
    return W.Csr(len(rows), n, pos, crd, vals)


def _case(span, la, lb, distinct, seed, reverse=False):
    """C rows of la * lb candidates of exactly `distinct` columns, which span
    exactly `span`; 37 rows of C.  Every column is dealt to one of the row's
    la B rows, which are then filled up to lb with others."""
    rng = np.random.default_rng(seed)
    m, n = 37, span + 4096
    brows, arows = [], []
    for i in range(m):
        lo = int(rng.integers(0, n - span + 1))
        cols = np.concatenate([[0], rng.choice(span - 2, distinct - 2, replace=False) + 1, [span - 1]])
        cols = rng.permutation(lo + cols)
        arows.append(range(i * la, (i + 1) * la))
        for q in range(la):
            own = cols[q::la]
            assert len(own) <= lb
            more = rng.choice(np.setdiff1d(cols, own), lb - len(own), replace=False)
            r = np.sort(np.concatenate([own, more])).astype(np.int64)
            brows.append(r[::-1] if reverse else r)
    return _csr(arows, m * la, seed), _csr(brows, n, seed + 1)


def _shape_of(A, B, i):
    """Row i of C: its candidates, its distinct columns and their span."""
    cols = np.concatenate([B.crd[B.pos[j]:B.pos[j + 1]] for j in A.crd[A.pos[i]:A.pos[i + 1]]])
    return len(cols), len(np.unique(cols)), int(cols.max()) - int(cols.min()) + 1


CASES = [
    # span, A entries, entries of a B row, distinct columns
    ("flags_small", (65, 3, 64, 65)), ("flags_edge", (1024, 5, 70, 300)),
    ("flags_full", (1024, 16, 64, 1024)), ("bits_edge", (1025, 5, 70, 300)),
    ("bits_mid", (20000, 9, 33, 250)), ("bits_top", (32768, 12, 40, 400)),
    ("sort_2_65", (40000, 13, 5, 60)), ("sort_2", (32769, 2, 64, 128)),
    ("sort_4", (40000, 3, 43, 120)), ("sort_4_top", (40000, 4, 64, 256)),
    ("sort_8", (70000, 257, 1, 257)), ("sort_8_top", (70000, 4, 128, 500)),
    ("sort_16", (70000, 9, 57, 513)), ("sort_16_top", (70000, 8, 128, 1000)),
    ("hash", (70000, 41, 25, 900)), ("hash_full", (70000, 11, 100, 1024)),
    # distinct columns around the staged search (682) and the sums in LDS (1024)
    ("staged_top", (60000, 11, 62, 682)), ("unstaged", (60000, 11, 63, 683)),
    ("slots", (50000, 8, 128, 1024)), ("over_slots", (50000, 41, 25, 1025)),
    ("staged_top_bits", (20000, 11, 62, 682)), ("unstaged_bits", (20000, 11, 63, 683)),
    ("over_slots_bits", (20000, 41, 25, 1025)),
    ("far_over_slots", (300000, 30, 60, 1700)), ("long_b", (900, 3, 700, 800)),
    ("many_a", (1000, 200, 3, 400)),
]


def test_cases_are_what_they_are_called():
    """Candidates, columns and spans of the cases, counted on the host."""
    for name, (span, la, lb, distinct) in CASES:
        A, B = _case(span, la, lb, distinct, seed=len(name) * 31 + span)
        for i in (0, 17, 36):
            assert _shape_of(A, B, i) == (la * lb, distinct, span), name
        route = ("flags" if span <= 1024 else "bits" if span <= 32768 else
                 "sort" if la * lb <= 1024 else "hash")
        kind = name.split("_")[0]
        if kind in ("flags", "bits", "sort", "hash"):
            assert kind == route, name
        if kind == "sort":
            values = int(name.split("_")[1])  # a lane: at most 64 times as many candidates
            assert max(32 * values, 64) < la * lb <= 64 * values, name


@pytest.mark.parametrize("name,shape", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("reverse", [False, True], ids=["sorted", "reversed"])
def test_mid_rows(name, shape, reverse):
    A, B = _case(*shape, seed=len(name) * 31 + shape[0], reverse=reverse)
    print(f"spgemm mid {name} reverse={reverse}", flush=True)
    pos, crd, vals = G.spgemm(A, B)
    opos, ocrd = oracle.spgemm_assemble(A, B)
    assert np.array_equal(pos, opos) and np.array_equal(crd, ocrd)
    assert np.array_equal(vals, oracle.spgemm_compute(A, B, opos, ocrd))


@pytest.mark.parametrize("m", [1, 7, 63, 65, 300])
def test_mid_rows_among_short_and_empty(m):
    """Rows of every kind interleaved, at row counts around a workgroup's
    share."""
    rng = np.random.default_rng(m)
    k, n = 500, 3000
    B = _csr([np.sort(rng.choice(n, int(c), replace=False))
              for c in rng.choice([0, 1, 5, 40, 90], k)], n, m + 1)
    A = _csr([np.sort(rng.choice(k, int(c), replace=False))
              for c in rng.choice([0, 1, 3, 10, 70], m)], k, m + 2)
    pos, crd, vals = G.spgemm(A, B)
    opos, ocrd = oracle.spgemm_assemble(A, B)
    assert np.array_equal(pos, opos) and np.array_equal(crd, ocrd)
    assert np.array_equal(vals, oracle.spgemm_compute(A, B, opos, ocrd))


def test_subnormal_sums():
    """Products and sums of multiples of 2^-1074 are exact: sums in LDS must
    not flush them.  Compared as integers (a host in flush-to-zero mode would
    compare the floats as equal)."""
    k = np.arange(1, 211, dtype=np.int64)
    B = W.Csr(70, 3, np.arange(0, 211, 3, dtype=np.int32), np.tile(np.arange(3, dtype=np.int32), 70),
              k.view(np.float64))
    A = W.Csr(1, 70, np.array([0, 70], np.int32), np.arange(70, dtype=np.int32), np.ones(70))
    _, crd, vals = G.spgemm(A, B)
    assert crd.tolist() == [0, 1, 2]
    assert vals.view(np.int64).tolist() == k.reshape(70, 3).sum(0).tolist()


def _check(A, B):
    pos, crd, vals = G.spgemm(A, B)
    opos, ocrd = oracle.spgemm_assemble(A, B)
    assert np.array_equal(pos, opos) and np.array_equal(crd, ocrd)
    assert np.array_equal(vals, oracle.spgemm_compute(A, B, opos, ocrd))


@pytest.mark.parametrize("m", [1, 3, 4, 5, 1023, 1024, 1025, 4095, 4096, 4097, 8191, 65536, 70001])
def test_every_row_listed(m):
    """Row counts around what a workgroup lists at a time (1024), the resident
    grid's waves (4096, past which neighbouring pieces stay on an XCD) and 64
    entries of the list for each workgroup (65,536).  66 candidates a row."""
    rng = np.random.default_rng(m)
    B = _csr([np.sort(rng.choice(500, 33, replace=False)) for _ in range(90)], 500, m)
    A = _csr(np.sort(np.stack([rng.integers(0, 45, m), rng.integers(45, 90, m)], 1), 1), 90, m + 1)
    _check(A, B)


@pytest.mark.parametrize("every", [1, 2, 7])
def test_long_rows_without_products(every):
    """Rows of more than 64 entries that all name empty rows of B, alone and
    among rows with products."""
    m, k = 1300, 200
    B = _csr([[], *([[5, 9, 11]] * 99)] + [[]] * 100, 20, 3)
    A = _csr([np.arange(100, 200) if i % every == 0 else np.arange(i % 100) for i in range(m)], k, 4)
    _check(A, B)


def test_heavy_rows_together_keep_their_pace():
    """Heavy rows that lie together (an operand sorted by degree) take about
    as long as the same rows spread out; with neighbouring
    rows left to a wave, 6 times."""
    m, heavy = 500_000, 256
    B = W.csr_from_counts(m, m, np.full(m, 8, np.int32), 41, W.STRUCT_BANDED, 64)
    took = {}
    for name, rows in (("together", np.arange(heavy)),
                       ("spread", np.arange(heavy) * (m // heavy))):
        counts = np.ones(m, np.int32)
        counts[rows] = 1000
        A = W.csr_from_counts(m, 20_000, counts, 42)
        A.n = m  # heavy rows name 20,000 of B's rows
        a, b, c = G.csr_desc(A), G.csr_desc(B), D.csr_empty((m, m))
        L = _lib.lib()
        _lib.check(L.taco_hip_spgemm_assemble(c.ptr, a.ptr, b.ptr))
        best = []
        for _ in range(4):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            _lib.check(L.taco_hip_spgemm_compute(c.ptr, a.ptr, b.ptr))
            t1.record()
            torch.cuda.synchronize()
            best.append(t0.elapsed_time(t1))
        took[name] = min(best)
        for p in (c.level_ptr(1, 0), c.level_ptr(1, 1), c.vals_ptr()):
            L.taco_hip_unified_free(ctypes.c_void_p(p))
    assert took["together"] < 3 * took["spread"], took


@pytest.mark.parametrize("ends,outside", [((10, 900), 5000), ((10, 900), 2), ((10, 30000), 60000),
                                          ((10, 30000), 2)],
                         ids=["flags_above", "flags_below", "bits_above", "bits_below"])
@pytest.mark.parametrize("long", [False, True], ids=["hash", "over_hash"])
def test_columns_outside_the_ends(ends, outside, long):
    """B rows that are not sorted inside and hold columns beyond their first
    and last ones: noticed while the columns are collected, and the row is
    done again by the hash set (of up to 1024 columns) or the global sort."""
    rng = np.random.default_rng(outside)
    m, la = 11, 40
    lb = 40 if long else 20
    brows, arows = [], []
    for i in range(m):
        arows.append(range(i * la, (i + 1) * la))
        for q in range(la):
            inner = rng.choice(np.arange(ends[0] + 1, ends[1]), lb - 2, replace=False)
            if (i + q) % 3 == 0:
                inner[rng.integers(0, lb - 2)] = outside
            brows.append(np.concatenate([[ends[0]], rng.permutation(inner), [ends[1]]]))
    A, B = _csr(arows, m * la, 5), _csr(brows, 70000, 6)
    if long:
        assert ends[1] < 1024 or _shape_of(A, B, 0)[1] > 1024
    else:
        assert _shape_of(A, B, 0)[1] <= 1024
    _check(A, B)

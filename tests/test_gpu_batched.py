"""Batched uneven SpMV/SpMM in one persistent launch: every instance against
the oracle, identical results for every schedule, hipGraph replays equal to
eager launches, and the autotuner's per-instance choice."""
import numpy as np
import pytest
import torch

import oracle
from taco_amd import batch as BT
from taco_amd import autotune

pytestmark = pytest.mark.gpu

TOL32 = 1e-5


@pytest.fixture(scope="module")
def wl():
    w = BT.BatchedWorkload(ninst=48, rmin=100, rmax=4000, seed=7, width=32, keep_host=True)
    assert set(w.structure.tolist()) == {0, 1, 2}
    return w


def check_spmv(wl, insts):
    for i in insts:
        A, x, _ = wl.instance(i)
        ye, cond = oracle.exact_spmv(A, x)
        rep = oracle.error_report(wl.y_of(i), ye, cond, TOL32)
        assert rep["ok"], (i, rep)


def check_spmm(wl, insts):
    for i in insts:
        A, _, B = wl.instance(i)
        Ce, cond = oracle.exact_spmm(A, B)
        rep = oracle.error_report(wl.c_of(i), Ce, cond, TOL32)
        assert rep["ok"], (i, rep)


def test_generated_patterns_match_host(wl):
    for i in (0, 7, 31):
        pos, crd = BT.instance_pattern(i, int(wl.m[i]), int(wl.structure[i]), wl.seed,
                                       wl.kmin, wl.kmax)
        A, _, _ = wl.instance(i)
        assert np.array_equal(A.pos, pos) and np.array_equal(A.crd, crd)


@pytest.mark.parametrize("lanes", BT.SPMV_LANES)
def test_batched_spmv_every_schedule(wl, lanes):
    wl.y.zero_()
    b = BT.Batch(wl, 0, np.full(wl.ninst, lanes, np.int32), rows_per_task=128)
    b.run()
    torch.cuda.synchronize()
    check_spmv(wl, range(wl.ninst))


@pytest.mark.parametrize("lanes", BT.SPMM_LANES)
def test_batched_spmm_every_schedule(wl, lanes):
    wl.C.zero_()
    b = BT.Batch(wl, 1, np.full(wl.ninst, lanes, np.int32), rows_per_task=64)
    b.run()
    torch.cuda.synchronize()
    check_spmm(wl, range(0, wl.ninst, 3))


def test_mixed_schedules_and_graph_replay(wl):
    rng = np.random.default_rng(3)
    sched = rng.choice(BT.SPMV_LANES, size=wl.ninst).astype(np.int32)
    b = BT.Batch(wl, 0, sched)
    wl.y.zero_()
    b.run()
    torch.cuda.synchronize()
    eager = wl.y.clone()
    check_spmv(wl, range(wl.ninst))
    b.capture()
    for rep in range(4):
        wl.y.fill_(float("nan"))
        b.launch_graph()
        torch.cuda.synchronize()
        # eager work between replays, then compare every replay
        assert torch.equal(wl.y, eager), rep
        b.run()
        torch.cuda.synchronize()


def test_batched_equals_unbatched(wl):
    """Per-instance results of the batch equal a one-instance batch."""
    b = BT.Batch(wl, 0, np.full(wl.ninst, 8, np.int32))
    wl.y.zero_()
    b.run()
    torch.cuda.synchronize()
    full = wl.y.clone()
    single = BT.BatchedWorkload(ninst=1, rmin=int(wl.m[0]), rmax=int(wl.m[0]), seed=wl.seed,
                                width=32, keep_host=True)
    # instance 0 of both workloads has the same seed-derived pattern and values
    assert np.array_equal(single.instance(0)[0].crd, wl.instance(0)[0].crd)
    sb = BT.Batch(single, 0, np.full(1, 8, np.int32))
    sb.run()
    torch.cuda.synchronize()
    assert np.array_equal(single.y_of(0), full[:int(wl.m[0])].cpu().numpy().astype(np.float64))


def test_run_range_writes_only_its_instances(wl):
    b = BT.Batch(wl, 0, np.full(wl.ninst, 4, np.int32))
    wl.y.zero_()
    b.run_range(5, 9)
    torch.cuda.synchronize()
    check_spmv(wl, range(5, 9))
    r0, r1 = int(wl.row_off[5]), int(wl.row_off[9])
    assert not wl.y[:r0].any() and not wl.y[r1:].any()
    b.run_range(9, 9)  # empty range: no launch, no error
    t = b.time_instances(2)
    assert t.shape == (wl.ninst,) and np.all(np.isfinite(t)) and np.all(t > 0)


def test_autotune_batch(wl):
    best, times, cands, rejected = autotune.tune_batch(wl, 0, reps=2)
    assert rejected == []
    assert best.shape == (wl.ninst,) and set(best.tolist()) <= set(cands)
    race = autotune.tune_batch.last_race
    assert set(race) == {"per_instance"} | {f"all_{l}" for l in cands}
    per_inst = np.array(cands, np.int32)[np.argmin(times, axis=0)]
    # the choice is the fastest whole launch: the per-instance minimum or
    # one candidate for every instance
    winner = min(race, key=race.get)
    if winner == "per_instance":
        assert np.array_equal(best, per_inst)
    else:
        assert np.all(best == int(winner.split("_")[1]))
    b = BT.Batch(wl, 0, best)
    wl.y.zero_()
    b.run()
    torch.cuda.synchronize()
    check_spmv(wl, range(wl.ninst))


@pytest.mark.parametrize("ninst", [1, 3, 11])
def test_batch_fewer_instances_than_queues(ninst):
    """Per-XCD queues with empty queues: every task still runs exactly once."""
    w = BT.BatchedWorkload(ninst=ninst, rmin=70, rmax=300, seed=20 + ninst, width=32,
                           keep_host=True)
    for lanes in (0, 4):
        w.y.fill_(float("nan"))
        b = BT.Batch(w, 0, np.full(w.ninst, lanes, np.int32), rows_per_task=16)
        b.run()
        torch.cuda.synchronize()
        check_spmv(w, range(w.ninst))
        del b


class _Rows:
    """A batch's workload: instances of n rows and n columns with the given row
    lengths, random columns."""

    def __init__(self, lengths, n, width, seed):
        rng = np.random.default_rng(seed)
        self.ninst, self.width = len(lengths), width
        self.m = np.array([len(c) for c in lengths])
        self.n = self.m
        self.nnz = np.array([sum(c) for c in lengths])
        assert all(len(c) == n for c in lengths)
        pos, crd = [], []
        for c in lengths:
            pos.append(np.concatenate([[0], np.cumsum(c)]))
            crd += [np.sort(rng.choice(n, k, replace=False)) for k in c]
        self.host = [(p, np.concatenate(crd[i * n:(i + 1) * n])) for i, p in enumerate(pos)]
        self.host_vals = rng.uniform(-1, 1, int(self.nnz.sum())).astype(np.float32)
        self.host_x = rng.uniform(-1, 1, (self.ninst, n, width)).astype(np.float32)
        self.pos = torch.tensor(np.concatenate(pos), dtype=torch.int32, device="cuda")
        self.crd = torch.tensor(np.concatenate(crd), dtype=torch.int32, device="cuda")
        self.vals = torch.tensor(self.host_vals, device="cuda")
        self.x = self.B = torch.tensor(self.host_x, device="cuda").reshape(-1)
        self.y = self.C = torch.full_like(self.x, float("nan"))

    def expect(self):
        """The products and, per row, the sum of their magnitudes, in 64 bits."""
        out = np.zeros(self.host_x.shape)
        size = np.zeros(self.host_x.shape)
        e = 0
        for i, (pos, crd) in enumerate(self.host):
            rows = np.repeat(np.arange(len(pos) - 1), np.diff(pos))
            v = self.host_vals[e:e + len(crd)].astype(np.float64)[:, None]
            with np.errstate(invalid="ignore"):
                p = v * self.host_x[i].astype(np.float64)[crd]
            np.add.at(out[i], rows, p)
            np.add.at(size[i], rows, np.abs(p))
            e += len(crd)
        return out, size


def _run(w, op, lanes):
    b = BT.Batch(w, op, lanes, rows_per_task=256)
    b.capture()
    for _ in range(3):
        w.y.fill_(float("nan"))
        b.launch_graph()
        torch.cuda.synchronize()
        out, size = w.expect()
        got = w.y.cpu().numpy().astype(np.float64).reshape(out.shape)
        # f32 sums of at most 65 products, each rounding at most 65 times.
        assert np.all(np.abs(got - out) <= 65 * 2.0 ** -24 * size + 1e-30)


# Rows of 1, 2, 3 and 4 entries make passes of 256, 512, 768 and 1024
# entries, one more or less moves a pass over the edge of two, four or eight
# entries in flight; 256 rows a task.
@pytest.mark.parametrize("lanes", [0, 8])
@pytest.mark.parametrize("length", [1, 2, 3, 4, 5, 16])
def test_short_rows_spmv(length, lanes):
    c = [[length] * 300, [length] * 255 + [length + 1] + [length] * 44,
         [max(length - 1, 0)] + [length] * 299]
    _run(_Rows(c, 300, 1, 5), 0, np.full(3, lanes, np.int32))


# Rows around the eight B rows that a team of lanes has in flight, at widths
# of four columns a lane and others, alone and in one batch.
@pytest.mark.parametrize("width,lanes", [(32, 8), (64, 16), (128, 32), (256, 64), (16, 8), (20, 8),
                                         (48, 16), (33, 16), (100, 32)])
def test_rows_around_a_block_spmm(width, lanes):
    rng = np.random.default_rng(width)
    c = [rng.choice([0, 1, 2, 7, 8, 9, 15, 16, 17, 64, 65], 120).tolist() for _ in range(3)]
    _run(_Rows(c, 120, width, 6), 1, np.full(3, lanes, np.int32))
    if 8 * lanes <= 256 and width == 4 * lanes:
        _run(_Rows(c, 120, width, 7), 1, np.array([lanes, 2 * lanes, lanes], np.int32))


@pytest.mark.parametrize("width,lanes", [(32, 8), (20, 8)])
def test_spmm_schedules_replaced_after_capture(width, lanes):
    """A captured launch stays right when the lane counts change."""
    c = [[5] * 64, [9] * 64]
    w = _Rows(c, 64, width, 8)
    b = BT.Batch(w, 1, np.full(2, lanes, np.int32))
    b.capture()
    for again in (16, 8, 32):
        b.set_schedules(np.array([lanes, again], np.int32))
        w.y.fill_(float("nan"))
        b.launch_graph()
        torch.cuda.synchronize()
        out, size = w.expect()
        got = w.y.cpu().numpy().astype(np.float64).reshape(out.shape)
        assert np.all(np.abs(got - out) <= 65 * 2.0 ** -24 * size)


@pytest.mark.parametrize("op,width,lanes", [(0, 1, 0), (0, 1, 8), (1, 32, 8), (1, 20, 8)])
def test_infinities_stay_in_their_rows(op, width, lanes):
    """x values and B rows of infinities and NaN reach only the rows that name
    them, also where a block is filled up past a row's end."""
    c = [[3, 8, 1, 11, 0, 7, 9, 2] * 20] * 2
    w = _Rows(c, 160, width, 9)
    w.host_x[:, 5] = np.inf
    w.host_x[:, 77] = np.nan
    w.x.copy_(torch.tensor(w.host_x).reshape(-1))
    b = BT.Batch(w, op, np.full(2, lanes, np.int32))
    b.run()
    torch.cuda.synchronize()
    got = w.y.cpu().numpy().reshape(w.host_x.shape)
    for i, (pos, crd) in enumerate(w.host):
        rows = np.repeat(np.arange(160), np.diff(pos))
        hit = np.unique(rows[np.isin(crd, [5, 77])])
        clean = np.setdiff1d(np.arange(160), hit)
        assert hit.size and np.isfinite(got[i][clean]).all() and not np.isfinite(got[i][hit]).any()

// Two-phase SpGEMM on the GPU, C(i,k) = A(i,j) * B(j,k), all CSR, f64.
//
// taco has no GPU SpGEMM (its default GPU schedule bails out on the dense
// workspace, reference transformations.cpp:1578-1583); this follows the
// semantics of its CPU two-phase code (lowerer_impl_imperative.cpp:
// 2197-2271, 2554-2561, 2616-2779; mode_format_compressed.cpp:217-271):
//   assemble  row i's pattern is the sorted set of distinct structural
//             columns {crd_B[kB] : jA in row i of A, kB in row crd_A[jA] of
//             B} (structural: numeric zeros are kept);  pos is the prefix sum
//             of the per-row counts; crd holds each row sorted ascending.
//   compute   C(i,k) accumulates A_ij * B_jk over that row's candidates in
//             encounter order (jA outer, kB inner), first product stored,
//             later ones added — the order of taco's workspace loop.
//
// Assemble sorts each row once:
//   1. per-row candidate counts (sum of the B row lengths A's row names) and
//      their prefix sum give every row a scratch region that holds all of
//      its candidates;
//   2. one symbolic pass writes each row's sorted distinct columns into its
//      region and its distinct count;
//   3. the prefix sum of the distinct counts is C's pos; a compaction
//      copies each region's sorted columns to crd.
// Rows with more distinct columns than the LDS row set holds are listed by
// pass 2 and sorted in global memory: their candidates are written out in
// encounter order, sorted per row by a segmented radix sort (rocPRIM) and
// deduplicated into their regions.  When the candidate total exceeds the
// int32 range the two-pass protocol of taco (count, then fill, each
// building the row set) is used instead, with the LDS row-set limit.
//
// Row kernels, one 64-lane wave per row, built on the row helpers of
// include/taco_hip_rt.h (shared with modules emitted by CodeGen_HIP):
//   short rows (<= 64 candidates): candidates in lanes, bitonic sort across
//     the wave by register moves (DPP, lane-half swaps).  The numeric phase
//     sorts (column, encounter index) keys, in 32 bits when the columns
//     allow, so equal columns come out in encounter order and are summed
//     sequentially in that order.  The hand-written short-row kernels take
//     three rows a wave at a time, staging their loads together, and leave
//     longer rows to a second pass.
//   longer rows (k_spgemm_symbolic_mid, k_spgemm_numeric_mid): flags or bits
//     by column where the columns lie close together, a register sort up to
//     TACO_HIP_ROW_CAP candidates, else a per-wave LDS hash set of up to
//     TACO_HIP_ROW_CAP distinct columns and an in-LDS bitonic sort; the
//     numeric phase adds the products into LDS, one A entry after another
//     (rows of more than TACO_HIP_ROW_CAP columns accumulate in C's values
//     in global memory, in the same order).

#include <climits>
#include <vector>

#include <rocprim/device/device_segmented_radix_sort.hpp>

#include "common.h"
#include "device.h"
#include "taco_hip_rt.h"

namespace taco_hip {
namespace {

constexpr int kWavesPerBlock = TACO_HIP_ROW_WAVES;
constexpr int kHashCap = TACO_HIP_ROW_CAP;

// Symbolic pass.  FILL == false: counts[i] = distinct columns of row i.
// FILL == true: writes row i's sorted columns to ccrd[cpos[i] ...].
// status bit 1 is set when a long row exceeds kHashCap distinct columns.
template <bool FILL>
__global__ __launch_bounds__(256) void k_spgemm_symbolic(
    int32_t m, const int32_t* __restrict__ apos, const int32_t* __restrict__ acrd,
    const int32_t* __restrict__ bpos, const int32_t* __restrict__ bcrd,
    int32_t* __restrict__ counts, const int32_t* __restrict__ cpos,
    int32_t* __restrict__ ccrd, int32_t* __restrict__ status) {
  const int64_t i = (int64_t)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
  if (i >= m) return;
  const int32_t c = taco_hip_spgemm_row_symbolic<FILL>(
      apos, acrd, bpos, bcrd, (int32_t)i, FILL ? cpos[i] : 0, ccrd, status);
  if (!FILL && __lane_id() == 0) counts[i] = c;
}

// Rows per wave taken together by the short-row kernels: their dependent
// loads (A's row bounds, A's entries, B's row bounds, B's entries) are
// issued stage by stage for all of them, so that many rows' loads are in
// flight at once.
constexpr int kRowsTogether = 3;

// A wave's kRowsTogether short rows, rows base + q * stride (base and
// stride wave-uniform), staged: each stage issues its loads for every row
// before the next stage waits for them.  Every load reads a valid address
// (indices clamped, A and B each holding at least one entry), so no load
// sits under a branch, and lanes past a row's end mask what they loaded.
// Lane t < la[q] holds A's entry t of row q; a row of more than 64
// candidates (or 64 A entries) has total[q] = 65 and no candidates in
// lanes; otherwise lane c < total[q] holds candidate c (encounter order):
// its column col[q] and, with VALS, its product prod[q].
template <int R, bool VALS>
struct ShortRows {
  bool real[R];
  int32_t a0[R], la[R], total[R], col[R];
  double prod[R];

  __device__ void load(int64_t base, int64_t stride, int32_t m, const int32_t* apos,
                       const int32_t* acrd, const double* avals, int32_t nnz_a,
                       const int32_t* bpos, const int32_t* bcrd, const double* bvals,
                       int32_t nnz_b) {
    const int lane = (int)__lane_id();
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int64_t i = base + q * stride;
      real[q] = i < m;
      const int64_t ic = real[q] ? i : m;
      a0[q] = apos[ic];
      la[q] = real[q] ? apos[ic + 1] - a0[q] : 0;
    }
    int32_t j[R];
    double av[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      int32_t e = a0[q] + (lane < la[q] ? lane : la[q] - 1);
      e = e < 0 ? 0 : (e < nnz_a ? e : nnz_a - 1);
      j[q] = acrd[e];
      av[q] = VALS ? avals[e] : 0.0;
    }
    int32_t b0[R], b1[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      if (lane >= la[q] || la[q] > 64) j[q] = 0;
      b0[q] = bpos[j[q]];
      b1[q] = bpos[j[q] + 1];
    }
    int32_t kB[R];
    double a[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const bool mine = lane < la[q] && la[q] <= 64;
      const int32_t len = (b1[q] - b0[q]) & (mine ? -1 : 0);
      // B row lengths clamped to 65: the sums stay small and a total above
      // 64 still reads as above 64.
      const int32_t lc = len < 65 ? len : 65;
      const int32_t inc = taco_hip_wave_scan_add_i32(lc);
      total[q] = la[q] > 64 ? 65 : __builtin_amdgcn_readlane(inc, 63);
      // Entry t holding candidate `lane`: the entries s < la - 1 whose
      // inclusive sum is <= lane.
      const int32_t tops = total[q] <= 64 ? la[q] - 1 : 0;
      int t = 0;
      for (int s2 = 0; s2 < tops; ++s2) t += __builtin_amdgcn_readlane(inc, s2) <= lane ? 1 : 0;
      const int32_t excl = __shfl(inc - lc, t, 64);
      const int32_t bt = __shfl(b0[q], t, 64);
      a[q] = VALS ? __shfl(av[q], t, 64) : 0.0;
      int32_t k = bt + (lane - excl);
      kB[q] = k < 0 ? 0 : (k < nnz_b ? k : nnz_b - 1);
    }
    int32_t c[R];
    double bv[R];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      c[q] = bcrd[kB[q]];
      bv[q] = VALS ? bvals[kB[q]] : 0.0;
    }
    // Masks applied arithmetically, so that every lane uses what it loaded
    // and the compiler keeps the loads where they are (a select would let
    // it move them under a branch and wait there).  Columns are
    // non-negative, so c | INT_MAX = INT_MAX; x * 1.0 is exact.
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const bool cand = total[q] <= 64 && lane < total[q];
      col[q] = c[q] | (cand ? 0 : INT_MAX);
      prod[q] = VALS ? a[q] * bv[q] * (cand ? 1.0 : 0.0) : 0.0;
    }
  }
};

// Numeric pass over the rows of at most 64 candidates, whose products stay
// in lanes: this kernel uses no LDS, so twice as many waves stay resident as
// with the general row kernel (whose long-row accumulators take 32 KB of
// LDS per workgroup), and each wave stages the loads of kRowsTogether rows
// at once.  mid[i] says of every row whether it is longer and left to
// k_spgemm_numeric_mid; *listed is cleared for k_spgemm_list_mid.
__global__ __launch_bounds__(256) void k_spgemm_numeric_short(
    int32_t m, const int32_t* __restrict__ apos, const int32_t* __restrict__ acrd,
    const double* __restrict__ avals, int32_t nnz_a, const int32_t* __restrict__ bpos,
    const int32_t* __restrict__ bcrd, const double* __restrict__ bvals, int32_t nnz_b,
    const int32_t* __restrict__ cpos, double* __restrict__ cvals, uint8_t* __restrict__ mid,
    int32_t* __restrict__ listed) {
  const int lane = (int)__lane_id();
  const int64_t stride = (int64_t)gridDim.x * kWavesPerBlock;
  const int64_t first = (int64_t)blockIdx.x * kWavesPerBlock +
                        __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  if (first == 0 && lane == 0) *listed = 0;
  const TacoHipSortMasks sm;
  for (int64_t base = first; base < m; base += kRowsTogether * stride) {
    ShortRows<kRowsTogether, true> r;
    r.load(base, stride, m, apos, acrd, avals, nnz_a, bpos, bcrd, bvals, nnz_b);
#pragma unroll
    for (int q = 0; q < kRowsTogether; ++q) {
      if (!r.real[q]) continue;
      const int64_t i = base + q * stride;
      if (lane == 0) mid[i] = r.total[q] > 64;
      if (r.total[q] > 64) continue;
      const int32_t c0 = cpos[i];
      taco_hip_spgemm_row_sum_store(r.total[q], r.col[q], r.prod[q], c0, cpos[i + 1] - c0,
                                    cvals, &sm);
    }
  }
}

// ---- rows of more than 64 candidates (or more than 64 A entries) ----
//
// One wave per row.  The rows are listed kListRows at a time: a workgroup
// finds those among its rows and appends them, in their order, with one
// atomic.  (One atomic a row took 1.07 ms for 100,003 rows.)  The list is
// dealt out in pieces of a row for each wave, piece p to workgroup p modulo
// the grid, so that heavy rows that lie together, as after a sort by degree,
// are worked on side by side: taking neighbouring rows in turn, a wave had
// up to 64 of them (256 rows of 1000 A entries first in 1,000,000 rows,
// 8,000 candidates each: compute 11.1 ms, now 1.07).  Within a workgroup the waves claim rows as they get done.

// Rows that one workgroup lists at a time, a word of flags a thread.
constexpr int kListRows = 1024;
// Appends the rows row0 + 4 * threadIdx.x + q whose bit q is set in `which`
// to list, kept in order.  The whole workgroup calls it.
__device__ __forceinline__ void list_rows(uint32_t which, int32_t row0,
                                          int32_t* __restrict__ list,
                                          int32_t* __restrict__ count) {
  __shared__ int32_t s_n[kWavesPerBlock], s_base;
  const int lane = (int)__lane_id(), wave = (int)(threadIdx.x / kWave);
  const int32_t mine = __popc(which);
  const int32_t inc = taco_hip_wave_scan_add_i32(mine);
  if (lane == kWave - 1) s_n[wave] = inc;
  __syncthreads();
  if (threadIdx.x == 0) {
    int32_t all = 0;
    for (int w = 0; w < kWavesPerBlock; ++w) all += s_n[w];
    s_base = all > 0 ? atomicAdd(count, all) : 0;
  }
  __syncthreads();
  int32_t at = s_base + inc - mine;
  for (int w = 0; w < wave; ++w) at += s_n[w];
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if ((which >> q) & 1) list[at++] = row0 + 4 * (int32_t)threadIdx.x + q;
  __syncthreads();  // s_n may be written again
}

// The rows that k_spgemm_numeric_short marked.  mid holds m bytes from a
// multiple of 4 on, up to a multiple of 4.
__global__ __launch_bounds__(256) void k_spgemm_list_mid(int32_t m,
                                                         const uint32_t* __restrict__ mid,
                                                         int32_t* __restrict__ list,
                                                         int32_t* __restrict__ listed) {
  const int32_t row0 = (int32_t)blockIdx.x * kListRows;
  const int64_t r = (int64_t)row0 + 4 * threadIdx.x;
  const uint32_t flags = r < m ? mid[r / 4] : 0u;
  uint32_t which = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    which |= r + q < m && ((flags >> (8 * q)) & 0xFF) ? 1u << q : 0u;
  list_rows(which, row0, list, listed);
}

// Grid of the kernels below: as many workgroups as are resident, 4 a CU by
// the LDS of k_spgemm_numeric_mid.  Workgroups without a row cost about 1 ns
// each (16,384 of them 16 us in a product of short rows alone, now 4), and
// 100,003 banded rows take 198, 231, 201 and 213 us in k_spgemm_numeric_mid
// and what goes with it at 1024, 1536, 2048 and 4096 workgroups.
constexpr int kMidGrid = 1024;
inline unsigned mid_grid(int32_t m) {
  const int64_t pieces = ((int64_t)m + kWavesPerBlock - 1) / kWavesPerBlock;
  return (unsigned)(pieces < kMidGrid ? (pieces > 0 ? pieces : 1) : kMidGrid);
}

// A workgroup's share of the list, claimed by its waves an entry at a time:
// entry e is list[(e / 4 * grid + slot) * 4 + e % 4].  Workgroups go to the 8
// XCDs round robin.  Where the waves have more than a row each, slots run
// over kXcdRun pieces on one XCD before they go on to the next, so that
// neighbouring rows find their B rows in its L2.
constexpr int kXcdRun = 32;
struct Share {
  int32_t count, grid, slot;
  __device__ __forceinline__ Share(int32_t n) : count(n), grid((int32_t)gridDim.x) {
    const int32_t b = (int32_t)blockIdx.x, run = 8 * kXcdRun;
    const bool runs = n / kWavesPerBlock >= grid && b < grid / run * run;
    slot = runs ? b / run * run + b % 8 * kXcdRun + b % run / 8 : b;
  }
  // INT_MAX and more past the int32 range: no entry.
  __device__ __forceinline__ int64_t at(int32_t e) const {
    return ((int64_t)(e / kWavesPerBlock) * grid + slot) * kWavesPerBlock + e % kWavesPerBlock;
  }
  // No entry of the share from e's piece on is in the list.
  __device__ __forceinline__ bool over(int32_t e) const {
    return at(e) - e % kWavesPerBlock >= count;
  }
};
__device__ __forceinline__ int32_t claim(int32_t* next) {
  int32_t e = 0;
  if (__lane_id() == 0) e = atomicAdd(next, 1);
  return __builtin_amdgcn_readfirstlane(e);
}

__device__ __forceinline__ double readlane_f64(double v, int lane) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// The first 64 entries of a row of A in lanes: each with its B row's start
// and length.  A wave loads them for its next row while it works on the
// current one, in two steps (entries, then the B rows' bounds), since each
// step waits for memory as long as a batch of B rows does.
template <bool VALS>
struct ARow {
  int32_t a0, la, j, b0, n;
  double av;

  __device__ __forceinline__ void entries(int32_t start, int32_t end,
                                          const int32_t* __restrict__ acrd,
                                          const double* __restrict__ avals) {
    a0 = start;
    la = end - start;
    const int lane = (int)__lane_id();
    const int32_t last = la < kWave ? la - 1 : kWave - 1;  // la > 0: the row has candidates
    const int32_t p = start + (lane < last ? lane : last);
    j = acrd[p];
    av = VALS ? avals[p] : 0.0;
  }
  __device__ __forceinline__ void bounds(const int32_t* __restrict__ bpos) {
    b0 = bpos[j];
    n = bpos[j + 1] - b0;
  }
};

// A row's candidates, in encounter order, 64 at a time (lane l holds
// candidate l of the step), as body(valid, column, product, t): t is the A
// entry (0 .. 63 of the entries in hand) that a lane's candidate belongs to,
// not falling from lane to lane.  A lane finds its entry by binary search
// over the prefix sums of the B row lengths, which the lanes hold.  Full
// lanes matter: with one B row to a load (17 of 64 lanes in use on a banded
// matrix) the L1's data path was busy for half of the kernel's 380 us.
// kMidSteps steps are loaded while the last kMidSteps are handed over.
// Every load is unconditional, so that the compiler waits for each only
// where it is used: lanes past the end repeat the last candidate.
// between() runs once, when the first loads have been issued.
constexpr int kMidSteps = 3;
template <bool VALS>
struct Candidates {
  int32_t col[kMidSteps], t[kMidSteps];
  double a[kMidSteps], b[kMidSteps];

  __device__ __forceinline__ void load(int32_t q0, int32_t total, int32_t inc, int32_t base,
                                       double av, const int32_t* __restrict__ bcrd,
                                       const double* __restrict__ bvals, int32_t nnz_b) {
    const int lane = (int)__lane_id();
#pragma unroll
    for (int u = 0; u < kMidSteps; ++u) {
      const int32_t q = q0 + u * kWave + lane;
      const int32_t qc = q < total ? q : total - 1;
      int at = 0;
#pragma unroll
      for (int step = 32; step > 0; step >>= 1)
        at += __builtin_amdgcn_ds_bpermute((at + step - 1) * 4, inc) <= qc ? step : 0;
      t[u] = at;
      int32_t k = __builtin_amdgcn_ds_bpermute(at * 4, base) + qc;
      k = k < 0 ? 0 : (k < nnz_b ? k : nnz_b - 1);
      col[u] = bcrd[k];
      a[u] = VALS ? __shfl(av, at, 64) : 0.0;
      b[u] = VALS ? bvals[k] : 0.0;
    }
  }
};

template <bool VALS, typename Between, typename Body>
__device__ __forceinline__ void for_each_candidate(
    const ARow<VALS>& row, const int32_t* __restrict__ acrd, const double* __restrict__ avals,
    const int32_t* __restrict__ bpos, const int32_t* __restrict__ bcrd,
    const double* __restrict__ bvals, int32_t nnz_b, Between between, Body body) {
  const int lane = (int)__lane_id();
  ARow<VALS> r = row;
  int32_t left = row.la;
  for (;;) {
    const int cnt = left < kWave ? left : kWave;
    const int32_t n = lane < cnt ? r.n : 0;
    const int32_t inc = taco_hip_wave_scan_add_i32(n);
    const int32_t base = r.b0 - (inc - n);
    const int32_t total = __builtin_amdgcn_readlane(inc, 63);
    Candidates<VALS> next;
    next.load(0, total, inc, base, r.av, bcrd, bvals, nnz_b);
    if (left == row.la) between();
    for (int32_t q0 = 0; q0 < total; q0 += kMidSteps * kWave) {
      const Candidates<VALS> now = next;
      next.load(q0 + kMidSteps * kWave, total, inc, base, r.av, bcrd, bvals, nnz_b);
#pragma unroll
      for (int u = 0; u < kMidSteps; ++u) {
        const int32_t q = q0 + u * kWave;
        if (q < total) body(q + lane < total, now.col[u], now.a[u] * now.b[u], now.t[u]);
      }
    }
    left -= cnt;
    if (left <= 0) return;
    r.entries(r.a0 + cnt, r.a0 + cnt + left, acrd, avals);
    r.bounds(bpos);
  }
}

// Adds a step's products to acc[slot], one A entry after another: the
// wave's LDS instructions run in program order, and the columns of one B
// row are distinct, so every slot sums its products in encounter order.
__device__ __forceinline__ void add_in_order(bool valid, int32_t slot, double prod, int32_t t,
                                             double* acc) {
  const int32_t t0 = __builtin_amdgcn_readfirstlane(t);
  const int32_t t1 = __builtin_amdgcn_readlane(t, kWave - 1);
  for (int32_t k = t0; k <= t1; ++k)
    if (valid && t == k) atomicAdd(acc + slot, prod);
}

// Numeric pass over the listed rows.  A row's
// sums live in LDS, 8 KB a wave (16 waves a CU):
//   columns spanning at most 1024: the sum of column c at c - (first column);
//   at most 682 columns: sums by position, found by binary search over the
//     row's columns, staged in LDS beside them;
//   at most 1024 columns: the same, searching the pattern in global memory;
//   more: taco_hip_spgemm_row_numeric_global.
// A B row's products go to LDS in one float-add instruction (add_in_order);
// one product after another with a wait for each, as these rows were summed
// before, took 2.5 ms on 100,003 banded rows of about 330 candidates (now
// 184 us: each row's chain of loads, at those 16 waves).
constexpr int kMidLdsBytes = 8192;
constexpr int kMidSlots = kMidLdsBytes / 8;
constexpr int kMidStaged = kMidLdsBytes / 12;
__global__ __launch_bounds__(256) void k_spgemm_numeric_mid(
    const int32_t* __restrict__ list, const int32_t* __restrict__ listed,
    const int32_t* __restrict__ apos, const int32_t* __restrict__ acrd,
    const double* __restrict__ avals, const int32_t* __restrict__ bpos,
    const int32_t* __restrict__ bcrd, const double* __restrict__ bvals, int32_t nnz_b,
    const int32_t* __restrict__ cpos, const int32_t* __restrict__ ccrd,
    double* __restrict__ cvals) {
  __shared__ double s_acc[kWavesPerBlock][kMidSlots];
  __shared__ int32_t s_next;
  const Share share(*listed);
  if (share.over(0)) return;
  if (threadIdx.x == 0) s_next = 0;
  __syncthreads();
  const int lane = (int)__lane_id();
  double* acc = s_acc[threadIdx.x / kWave];
  int32_t* keys = (int32_t*)(acc + kMidStaged);
  // Lane l holds what entry 64 * batch + l of the share starts from.
  int32_t batch = -1;
  int32_t hrow = -1, ha0 = 0, ha1 = 0, hc0 = 0, hnc = 0, hfirst = 0, hlast = -1;
  // The next entry with columns, as its lane; -1: none is left.
  const auto take = [&]() {
    for (;;) {
      const int32_t e = claim(&s_next);
      if (share.over(e)) return -1;
      if (e / kWave != batch) {
        batch = e / kWave;
        const int64_t q = share.at(batch * kWave + lane);
        hrow = q < share.count ? list[q] : -1;
        hnc = 0;
        if (hrow >= 0) {
          ha0 = apos[hrow];
          ha1 = apos[hrow + 1];
          hc0 = cpos[hrow];
          hnc = cpos[hrow + 1] - hc0;
          if (hnc > 0) {
            hfirst = ccrd[hc0];
            hlast = ccrd[hc0 + hnc - 1];
          }
        }
      }
      if (__builtin_amdgcn_readlane(hnc, e % kWave) > 0) return e % kWave;
    }
  };
  int from = take();
  if (from < 0) return;
  int32_t a0 = __builtin_amdgcn_readlane(ha0, from), a1 = __builtin_amdgcn_readlane(ha1, from);
  ARow<true> next;
  next.entries(a0, a1, acrd, avals);
  next.bounds(bpos);
  while (from >= 0) {
    const ARow<true> row = next;
    const int32_t i = __builtin_amdgcn_readlane(hrow, from);
    const int32_t c0 = __builtin_amdgcn_readlane(hc0, from);
    const int32_t nc = __builtin_amdgcn_readlane(hnc, from);
    const int32_t first = __builtin_amdgcn_readlane(hfirst, from);
    const int64_t span = (int64_t)__builtin_amdgcn_readlane(hlast, from) - first + 1;
    from = take();
    if (from >= 0) {  // the last row's successor is that row again
      a0 = __builtin_amdgcn_readlane(ha0, from);
      a1 = __builtin_amdgcn_readlane(ha1, from);
    }
    next.entries(a0, a1, acrd, avals);
    const auto bounds = [&]() { next.bounds(bpos); };
    const int32_t* crow = ccrd + c0;
    if (nc > kMidSlots) {
      taco_hip_spgemm_row_numeric_global(apos, acrd, avals, bpos, bcrd, bvals,
                                         i, c0, nc, ccrd, cvals);
      bounds();
    } else if (span > 0 && span <= kMidSlots) {
      const uint32_t width = (uint32_t)span;
      for (int q = lane; q < (int)width; q += kWave) acc[q] = 0.0;
      taco_hip_wave_lds_sync();
      for_each_candidate<true>(
          row, acrd, avals, bpos, bcrd, bvals, nnz_b, bounds,
          [&](bool valid, int32_t col, double prod, int32_t t) {
            const uint32_t slot = (uint32_t)col - (uint32_t)first;
            add_in_order(valid && slot < width, (int32_t)slot, prod, t, acc);
          });
      taco_hip_wave_lds_sync();
      for (int q = lane; q < nc; q += kWave) {
        const uint32_t slot = (uint32_t)crow[q] - (uint32_t)first;
        __builtin_nontemporal_store(slot < width ? acc[slot] : 0.0, cvals + c0 + q);
      }
      taco_hip_wave_lds_sync();
    } else {
      const bool staged = nc <= kMidStaged;
      for (int q = lane; q < nc; q += kWave) {
        acc[q] = 0.0;
        if (staged) keys[q] = crow[q];
      }
      taco_hip_wave_lds_sync();
      int top = 1;  // the largest power of two <= nc
      while (2 * top <= nc) top <<= 1;
      for_each_candidate<true>(
          row, acrd, avals, bpos, bcrd, bvals, nnz_b, bounds,
          [&](bool valid, int32_t col, double prod, int32_t t) {
            // The last position whose column is <= col.
            int at = 0;
            bool found;
            if (staged) {
              for (int step = top; step > 0; step >>= 1) {
                const int q = at + step < nc ? at + step : nc - 1;
                const int32_t key = keys[q];
                at = at + step < nc && key <= col ? q : at;
              }
              found = keys[at] == col;
            } else {
              for (int step = top; step > 0; step >>= 1) {
                const int q = at + step < nc ? at + step : nc - 1;
                const int32_t key = crow[q];
                at = at + step < nc && key <= col ? q : at;
              }
              found = crow[at] == col;
            }
            add_in_order(valid && found, at, prod, t, acc);
          });
      taco_hip_wave_lds_sync();
      for (int q = lane; q < nc; q += kWave)
        __builtin_nontemporal_store(acc[q], cvals + c0 + q);
      taco_hip_wave_lds_sync();
    }
  }
}

// ---- one-sort assemble ----

// cand[i] = candidates of row i (saturated at INT_MAX; the prefix sum then
// reports the overflow).  kCandLanes lanes per row, each striding the row's
// A entries, so a wave covers 64 / kCandLanes rows and a row's loads are in
// flight together.
constexpr int kCandLanes = 8;
// It also clears the assemble's status words (status[0..15]), which no
// kernel reads before the prefix sum that follows it.
__global__ __launch_bounds__(256) void k_spgemm_row_cands(
    int32_t m, const int32_t* __restrict__ apos, const int32_t* __restrict__ acrd,
    const int32_t* __restrict__ bpos, int32_t* __restrict__ cand,
    int32_t* __restrict__ status) {
  if (blockIdx.x == 0 && threadIdx.x < 16) status[threadIdx.x] = 0;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t i = t / kCandLanes;
  const int sub = (int)(t % kCandLanes);
  int64_t n = 0;
  if (i < m)
    for (int32_t p = apos[i] + sub; p < apos[i + 1]; p += kCandLanes) {
      const int32_t j = acrd[p];
      n += bpos[j + 1] - bpos[j];
    }
#pragma unroll
  for (int off = kCandLanes / 2; off > 0; off >>= 1) n += __shfl_xor(n, off, kCandLanes);
  if (i < m && sub == 0) cand[i] = n > INT_MAX ? INT_MAX : (int32_t)n;
}

// Pass 2 over the rows of at most 64 candidates (no LDS, so more waves stay
// resident): each row's sorted distinct columns go to its scratch region
// and its distinct count to counts.  Longer rows are first listed for
// k_spgemm_symbolic_mid in mid_rows (status[5] of them), the rows of A
// entries without candidates aside.  status[0] bit 4: the scratch holds
// fewer entries than the candidate total, or the candidate offsets
// overflowed (nothing done).
__global__ __launch_bounds__(256) void k_spgemm_symbolic_short(
    int32_t m, const int32_t* __restrict__ apos, const int32_t* __restrict__ acrd,
    int32_t nnz_a, const int32_t* __restrict__ bpos, const int32_t* __restrict__ bcrd,
    int32_t nnz_b, const int32_t* __restrict__ candoff, int64_t capacity,
    int32_t* __restrict__ scratch, int32_t* __restrict__ counts,
    int32_t* __restrict__ mid_rows, int32_t* __restrict__ status) {
  const int lane = (int)__lane_id();
  const int64_t first = (int64_t)blockIdx.x * kWavesPerBlock +
                        __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  // The candidate offsets overflowed int32 (status[2] bit 2: the caller
  // falls back to the two-pass form), or the scratch is too small: write
  // nothing.
  if ((status[2] & 2) || (int64_t)candoff[m] > capacity) {
    if (first == 0 && lane == 0) atomicOr(status, 4);
    return;
  }
  const int64_t stride = (int64_t)gridDim.x * kWavesPerBlock;
  if (nnz_a == 0 || nnz_b == 0) {
    // No candidates anywhere (and nothing the staged loads may read).
    for (int64_t i = first; i < m; i += stride)
      if (lane == 0) counts[i] = 0;
    return;
  }
  for (int64_t row0 = (int64_t)blockIdx.x * kListRows; row0 < m;
       row0 += (int64_t)gridDim.x * kListRows) {
    uint32_t which = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t r = row0 + 4 * threadIdx.x + q;
      if (r >= m) continue;
      const int32_t n = candoff[r + 1] - candoff[r];
      if (n > 64 || apos[r + 1] - apos[r] > 64) {
        if (n > 0)
          which |= 1u << q;
        else
          counts[r] = 0;
      }
    }
    list_rows(which, (int32_t)row0, mid_rows, status + 5);
  }
  const TacoHipSortMasks sm;
  for (int64_t base = first; base < m; base += kRowsTogether * stride) {
    ShortRows<kRowsTogether, false> r;
    r.load(base, stride, m, apos, acrd, nullptr, nnz_a, bpos, bcrd, nullptr, nnz_b);
#pragma unroll
    for (int q = 0; q < kRowsTogether; ++q) {
      if (!r.real[q]) continue;
      const int64_t i = base + q * stride;
      if (r.total[q] > 64) continue;
      const int32_t v = (int32_t)taco_hip_wave_sort_u32((uint32_t)r.col[q], sm);
      const int32_t prev = __shfl_up(v, 1, 64);
      const bool head = v != INT_MAX && (lane == 0 || prev != v);
      const uint64_t heads = __ballot(head);
      if (head) scratch[candoff[i] + __popcll(heads & ((1ull << lane) - 1))] = v;
      if (lane == 0) counts[i] = __popcll(heads);
    }
  }
}

// Bitonic sort of 64 * E values across a wave, E per lane (lane l holds
// elements l * E .. l * E + E - 1 of the result).  Exchanges between lanes are
// register moves; those of strides below E stay inside the lane.
template <int E, int K, int J>
__device__ __forceinline__ void sort_step(uint32_t (&v)[E], int lane) {
  if constexpr (J >= E) {
    constexpr int L = J / E;  // lane distance; K >= 2 * J, so "up" is the lane's
    const uint32_t keep_min = (((lane * E) & K) == 0) == ((lane & L) == 0) ? 0xFFFFFFFFu : 0u;
#pragma unroll
    for (int r = 0; r < E; ++r)
      v[r] = taco_hip_bitonic_step_masked<K, L>(v[r], keep_min);
  } else {
#pragma unroll
    for (int r = 0; r < E; ++r) {
      if (r & J) continue;
      const uint32_t lo = v[r] < v[r + J] ? v[r] : v[r + J];
      const uint32_t hi = v[r] < v[r + J] ? v[r + J] : v[r];
      if constexpr (K < E) {
        v[r] = (r & K) == 0 ? lo : hi;
        v[r + J] = (r & K) == 0 ? hi : lo;
      } else {
        const uint32_t swap = ((lane * E) & K) == 0 ? 0u : 0xFFFFFFFFu;
        const uint32_t x = (lo ^ hi) & swap;
        v[r] = lo ^ x;
        v[r + J] = hi ^ x;
      }
    }
  }
  if constexpr (J > 1) sort_step<E, K, J / 2>(v, lane);
}
template <int E, int K = 2>
__device__ __forceinline__ void wave_sort_regs(uint32_t (&v)[E], int lane) {
  sort_step<E, K, K / 2>(v, lane);
  if constexpr (K < 64 * E) wave_sort_regs<E, 2 * K>(v, lane);
}

// The n <= 64 * E columns in buf, sorted and deduplicated, to dst; returns
// their number.
template <int E>
__device__ __forceinline__ int32_t sort_distinct(const int32_t* buf, int32_t n, int32_t* dst) {
  const int lane = (int)__lane_id();
  uint32_t v[E];
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const int q = lane * E + r;
    v[r] = q < n ? (uint32_t)buf[q] : (uint32_t)INT_MAX;
  }
  wave_sort_regs<E>(v, lane);
  const uint32_t below = (uint32_t)__shfl_up((int)v[E - 1], 1, 64);
  uint32_t heads = 0;
#pragma unroll
  for (int r = 0; r < E; ++r) {
    const bool head = v[r] != (uint32_t)INT_MAX &&
                      (r == 0 ? lane == 0 || below != v[0] : v[r - 1] != v[r]);
    heads |= head ? 1u << r : 0u;
  }
  const int32_t mine = __popc(heads);
  const int32_t inc = taco_hip_wave_scan_add_i32(mine);
  int32_t at = inc - mine;
#pragma unroll
  for (int r = 0; r < E; ++r)
    if ((heads >> r) & 1) dst[at++] = (int32_t)v[r];
  return __builtin_amdgcn_readlane(inc, 63);
}

// Sorted distinct columns of the rows that k_spgemm_symbolic_short leaves,
// into their scratch regions, with 4 KB of LDS a wave.  The row's first and
// last columns come from the ends of its B rows:
//   columns spanning at most 1024: a flag per column (plain stores), read
//     back 64 at a time as a lane mask;
//   at most 32768: a bit per column, each lane emitting a run of words;
//   at most 1024 candidates: staged in LDS and sorted in registers;
//   otherwise: the LDS hash set of up to TACO_HIP_ROW_CAP distinct columns
//     (rows beyond it are listed in long_rows, status[1], for the
//     global-memory sort, their count left 0).
// Flags and bits need no sort and cost nothing for a repeated column: 123 us
// on 100,003 banded rows of about 330 candidates and 245 columns, where the
// hash set with its 1024-entry sort through LDS, which every such row took
// before, took 2.67 ms.  A B
// row that is not sorted may hold columns outside its ends: such a row of C
// is noticed and goes to the hash set.
constexpr int kMidFlags = TACO_HIP_ROW_CAP;
__global__ __launch_bounds__(256) void k_spgemm_symbolic_mid(
    const int32_t* __restrict__ mid_rows, const int32_t* __restrict__ apos,
    const int32_t* __restrict__ acrd, const int32_t* __restrict__ bpos,
    const int32_t* __restrict__ bcrd, int32_t nnz_b, const int32_t* __restrict__ candoff,
    int32_t* __restrict__ scratch, int32_t* __restrict__ counts,
    int32_t* __restrict__ long_rows, int32_t* __restrict__ status) {
  __shared__ TacoHipRowSet s_sets[kWavesPerBlock];
  __shared__ int32_t s_next;
  const Share share(status[0] & 4 ? 0 : status[5]);
  if (share.over(0)) return;
  if (threadIdx.x == 0) s_next = 0;
  __syncthreads();
  const int lane = (int)__lane_id();
  TacoHipRowSet* w = &s_sets[threadIdx.x / kWave];
  int32_t* buf = w->keys;
  // Lane l holds what entry 64 * batch + l of the share starts from.
  int32_t batch = -1;
  int32_t hrow = -1, ha0 = 0, ha1 = 0, hoff = 0, hn = 0;
  // The next entry, as its lane; -1: none is left.
  const auto take = [&]() {
    for (;;) {
      const int32_t e = claim(&s_next);
      if (share.over(e)) return -1;
      if (e / kWave != batch) {
        batch = e / kWave;
        const int64_t q = share.at(batch * kWave + lane);
        hrow = q < share.count ? mid_rows[q] : -1;
        if (hrow >= 0) {
          ha0 = apos[hrow];
          ha1 = apos[hrow + 1];
          hoff = candoff[hrow];
          hn = candoff[hrow + 1] - hoff;
        }
      }
      if (__builtin_amdgcn_readlane(hrow, e % kWave) >= 0) return e % kWave;
    }
  };
  int from = take();
  if (from < 0) return;
  // The next row's entries, bounds, and the ends of its B rows.
  ARow<false> next;
  int32_t lo, hi;
  const auto ends = [&]() {
    next.bounds(bpos);
    const int32_t k = next.n > 0 ? next.b0 : 0;
    const int32_t f = bcrd[k], l = bcrd[next.n > 0 ? next.b0 + next.n - 1 : 0];
    lo = next.n > 0 ? f : INT_MAX;
    hi = next.n > 0 ? l : -1;
  };
  int32_t a0 = __builtin_amdgcn_readlane(ha0, from), a1 = __builtin_amdgcn_readlane(ha1, from);
  next.entries(a0, a1, acrd, nullptr);
  ends();
  while (from >= 0) {
    const ARow<false> row = next;
    const int32_t i = __builtin_amdgcn_readlane(hrow, from);
    const int32_t n = __builtin_amdgcn_readlane(hn, from);
    int32_t* dst = scratch + __builtin_amdgcn_readlane(hoff, from);
    from = take();
    if (from >= 0) {  // the last row's successor is that row again
      a0 = __builtin_amdgcn_readlane(ha0, from);
      a1 = __builtin_amdgcn_readlane(ha1, from);
    }
    // A's entries past the first 64.
    for (int32_t p = row.a0 + kWave + lane; p < row.a0 + row.la; p += kWave) {
      const int32_t j = acrd[p];
      const int32_t b0 = bpos[j], b1 = bpos[j + 1];
      if (b0 < b1) {
        const int32_t f = bcrd[b0], l = bcrd[b1 - 1];
        lo = f < lo ? f : lo;
        hi = l > hi ? l : hi;
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const int32_t a = __shfl_xor(lo, off, 64), b = __shfl_xor(hi, off, 64);
      lo = a < lo ? a : lo;
      hi = b > hi ? b : hi;
    }
    const int32_t low = __builtin_amdgcn_readfirstlane(lo);
    const int64_t span64 = (int64_t)__builtin_amdgcn_readfirstlane(hi) - low + 1;
    next.entries(a0, a1, acrd, nullptr);
    int32_t cnt = -1;
    if (span64 > 0 && span64 <= kMidFlags) {
      const uint32_t span = (uint32_t)span64;
      for (int q = lane; q < (int)span; q += kWave) buf[q] = 0;
      taco_hip_wave_lds_sync();
      bool outside = false;
      for_each_candidate<false>(row, acrd, nullptr, bpos, bcrd, nullptr, nnz_b, ends,
                                [&](bool, int32_t col, double, int32_t) {
                                  // Lanes past the end repeat a column.
                                  const uint32_t at = (uint32_t)col - (uint32_t)low;
                                  if (at < span) buf[at] = 1;
                                  outside |= at >= span;
                                });
      taco_hip_wave_lds_sync();
      if (__ballot(outside) == 0) {
        cnt = 0;
        for (int q0 = 0; q0 < (int)span; q0 += kWave) {
          const int q = q0 + lane;
          const bool set = q < (int)span && buf[q] != 0;
          const uint64_t mask = __ballot(set);
          if (set) dst[cnt + __popcll(mask & ((1ull << lane) - 1))] = low + q;
          cnt += __popcll(mask);
        }
      }
      taco_hip_wave_lds_sync();
    } else if (span64 > 0 && span64 <= 32 * kMidFlags) {
      const uint32_t span = (uint32_t)span64;
      const int words = (int)((span + 31) / 32);
      for (int q = lane; q < words; q += kWave) buf[q] = 0;
      taco_hip_wave_lds_sync();
      bool outside = false;
      for_each_candidate<false>(row, acrd, nullptr, bpos, bcrd, nullptr, nnz_b, ends,
                                [&](bool valid, int32_t col, double, int32_t) {
                                  const uint32_t at = (uint32_t)col - (uint32_t)low;
                                  if (valid && at < span)
                                    atomicOr(buf + (at >> 5), 1 << (at & 31));
                                  outside |= valid && at >= span;
                                });
      taco_hip_wave_lds_sync();
      if (__ballot(outside) == 0) {
        const int per = (words + kWave - 1) / kWave;  // consecutive words a lane
        const int w0 = lane * per, w1 = w0 + per < words ? w0 + per : words;
        int32_t held = 0;
        for (int q = w0; q < w1; ++q) held += __popc((uint32_t)buf[q]);
        const int32_t inc = taco_hip_wave_scan_add_i32(held);
        int32_t at = inc - held;
        for (int q = w0; q < w1; ++q)
          for (uint32_t b = (uint32_t)buf[q]; b; b &= b - 1)
            dst[at++] = low + 32 * q + (__ffs((int)b) - 1);
        cnt = __builtin_amdgcn_readlane(inc, 63);
      }
      taco_hip_wave_lds_sync();
    } else if (n <= TACO_HIP_ROW_CAP) {
      int32_t at = 0;
      for_each_candidate<false>(row, acrd, nullptr, bpos, bcrd, nullptr, nnz_b, ends,
                                [&](bool valid, int32_t col, double, int32_t) {
                                  if (valid) buf[at + lane] = col;
                                  at += __popcll(__ballot(valid));
                                });
      taco_hip_wave_lds_sync();
      cnt = n <= 128   ? sort_distinct<2>(buf, n, dst)
            : n <= 256 ? sort_distinct<4>(buf, n, dst)
            : n <= 512 ? sort_distinct<8>(buf, n, dst)
                       : sort_distinct<16>(buf, n, dst);
      taco_hip_wave_lds_sync();
    } else {
      ends();
    }
    if (cnt < 0) {
      cnt = taco_hip_row_hash(w, apos, acrd, bpos, bcrd, i);
      if (cnt >= 0) {
        taco_hip_row_hash_sort(w);
        for (int q = lane; q < cnt; q += kWave) dst[q] = buf[q];
        taco_hip_wave_lds_sync();
      }
    }
    if (lane == 0) {
      if (cnt < 0) long_rows[atomicAdd(status + 1, 1)] = i;
      counts[i] = cnt < 0 ? 0 : cnt;
    }
  }
}

// Candidates of the listed long rows, lens[r] (candidate counts from the
// first prefix sum).
__global__ __launch_bounds__(256) void k_spgemm_long_lengths(
    int32_t nlong, const int32_t* __restrict__ long_rows, const int32_t* __restrict__ candoff,
    int32_t* __restrict__ lens) {
  const int32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nlong) return;
  const int32_t i = long_rows[r];
  lens[r] = candoff[i + 1] - candoff[i];
}

// Long row r's candidate columns, in encounter order, at keys[loff[r] ...].
__global__ __launch_bounds__(256) void k_spgemm_long_fill(
    int32_t nlong, const int32_t* __restrict__ long_rows, const uint32_t* __restrict__ loff,
    const int32_t* __restrict__ apos, const int32_t* __restrict__ acrd,
    const int32_t* __restrict__ bpos, const int32_t* __restrict__ bcrd,
    uint32_t* __restrict__ keys) {
  const int64_t r = (int64_t)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
  if (r >= nlong) return;
  const int lane = (int)__lane_id();
  const int32_t i = long_rows[r];
  uint32_t o = loff[r];
  for (int32_t p = apos[i]; p < apos[i + 1]; ++p) {
    const int32_t j = acrd[p];
    const int32_t b0 = bpos[j], b1 = bpos[j + 1];
    for (int32_t kB = b0 + lane; kB < b1; kB += kWave) keys[o + (uint32_t)(kB - b0)] = (uint32_t)bcrd[kB];
    o += (uint32_t)(b1 - b0);
  }
}

// Long row r's sorted candidates deduplicated into its scratch region;
// counts[i] = the distinct count.
__global__ __launch_bounds__(256) void k_spgemm_long_dedup(
    int32_t nlong, const int32_t* __restrict__ long_rows, const uint32_t* __restrict__ loff,
    const uint32_t* __restrict__ sorted, const int32_t* __restrict__ candoff,
    int32_t* __restrict__ scratch, int32_t* __restrict__ counts) {
  const int64_t r = (int64_t)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
  if (r >= nlong) return;
  const int lane = (int)__lane_id();
  const int32_t i = long_rows[r];
  const uint32_t q0 = loff[r], q1 = loff[r + 1];
  int32_t* dst = scratch + candoff[i];
  int32_t base = 0;
  for (uint32_t c0 = q0; c0 < q1; c0 += kWave) {
    const uint32_t q = c0 + (uint32_t)lane;
    bool head = false;
    uint32_t v = 0;
    if (q < q1) {
      v = sorted[q];
      head = q == q0 || sorted[q - 1] != v;
    }
    const uint64_t heads = __ballot(head);
    if (head) dst[base + __popcll(heads & ((1ull << lane) - 1))] = (int32_t)v;
    base += __popcll(heads);
  }
  if (lane == 0) counts[i] = base;
}

// crd: each row's sorted columns copied from its scratch region.  A
// workgroup takes kCompactRows consecutive rows, whose output range in crd
// is contiguous: their pos and region starts go to LDS, and the threads
// stride the range, each finding its row by binary search in LDS, so the
// stores are coalesced whatever the row lengths.
constexpr int kCompactRows = 256;
constexpr int kCompactUnroll = 4;
__global__ __launch_bounds__(256) void k_spgemm_compact(
    int32_t m, const int32_t* __restrict__ candoff, const int32_t* __restrict__ cpos,
    const int32_t* __restrict__ scratch, int32_t* __restrict__ ccrd) {
  __shared__ int32_t s_pos[kCompactRows + 1];
  __shared__ int32_t s_src[kCompactRows];
  const int64_t r0 = (int64_t)blockIdx.x * kCompactRows;
  const int32_t nr = (int32_t)(m - r0 < kCompactRows ? m - r0 : kCompactRows);
  for (int q = threadIdx.x; q <= nr; q += blockDim.x) s_pos[q] = cpos[r0 + q];
  for (int q = threadIdx.x; q < nr; q += blockDim.x) s_src[q] = candoff[r0 + q];
  __syncthreads();
  const int32_t e0 = s_pos[0], e1 = s_pos[nr];
  // kCompactUnroll entries per thread at a time, their row searches
  // interleaved and their loads in flight together; entries past the end
  // are clamped to the last entry of the range.
  for (int32_t e = e0 + (int32_t)threadIdx.x; e < e1;
       e += kCompactUnroll * (int32_t)blockDim.x) {
    int32_t ee[kCompactUnroll], lo[kCompactUnroll];
#pragma unroll
    for (int u = 0; u < kCompactUnroll; ++u) {
      const int32_t x = e + u * (int32_t)blockDim.x;
      ee[u] = x < e1 ? x : e1 - 1;
      lo[u] = 0;
    }
    // The row of entry ee: the largest r < nr with s_pos[r] <= ee.
#pragma unroll
    for (int step = kCompactRows / 2; step > 0; step >>= 1) {
#pragma unroll
      for (int u = 0; u < kCompactUnroll; ++u) {
        const int c = lo[u] + step;
        const int32_t pv = s_pos[c < nr ? c : nr - 1];  // read unconditionally
        lo[u] = ((c < nr) & (pv <= ee[u])) ? c : lo[u];
      }
    }
    int32_t v[kCompactUnroll];
#pragma unroll
    for (int u = 0; u < kCompactUnroll; ++u)
      v[u] = scratch[s_src[lo[u]] + (ee[u] - s_pos[lo[u]])];
    // Entries past the end store the last entry's own value again (ee is
    // clamped), so every lane stores and no load waits under a branch.
#pragma unroll
    for (int u = 0; u < kCompactUnroll; ++u) __builtin_nontemporal_store(v[u], ccrd + ee[u]);
  }
}


// ---- counts -> pos (exclusive prefix sum with pos[m] = total) ----
constexpr int kScanBlock = 256;
constexpr int kScanItems = 16;
constexpr int kScanTile = kScanBlock * kScanItems;
// Up to this many tiles every workgroup of k_scan_apply adds up the tile
// sums before its own (2048 of them: 8 loads a thread), which saves a launch
// of one workgroup (4.6 us of a 17 us scan at 500,000 counts); beyond it the
// work would grow with the square of the tiles and k_scan_tile_sums turns
// them into offsets first.
constexpr int kScanDirectTiles = 2048;

__device__ __forceinline__ int64_t block_exclusive_sum(int64_t v,
                                                       int64_t* s_tmp,
                                                       int64_t* total) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  int64_t inc = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int64_t u = __shfl_up(inc, off, kWave);
    if (lane >= off) inc += u;
  }
  if (lane == kWave - 1) s_tmp[wave] = inc;
  __syncthreads();
  int64_t wbase = 0, all = 0;
  for (int w = 0; w < kScanBlock / kWave; ++w) {
    if (w < wave) wbase += s_tmp[w];
    all += s_tmp[w];
  }
  __syncthreads();
  *total = all;
  return wbase + inc - v;
}

__global__ __launch_bounds__(kScanBlock) void k_scan_tiles(
    int32_t m, const int32_t* __restrict__ counts, int64_t* __restrict__ tile_sums) {
  __shared__ int64_t s_tmp[kScanBlock / kWave];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + threadIdx.x;
  int64_t v = 0;
#pragma unroll
  for (int q = 0; q < kScanItems; ++q)
    if (base + q * kScanBlock < m) v += counts[base + q * kScanBlock];
  int64_t total;
  block_exclusive_sum(v, s_tmp, &total);
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(kScanBlock) void k_scan_tile_sums(
    int32_t ntiles, int64_t* __restrict__ tile_sums) {
  __shared__ int64_t s_tmp[kScanBlock / kWave];
  int64_t carry = 0;
  for (int32_t t0 = 0; t0 < ntiles; t0 += kScanBlock) {
    const int32_t t = t0 + threadIdx.x;
    const int64_t v = t < ntiles ? tile_sums[t] : 0;
    int64_t total;
    const int64_t ex = block_exclusive_sum(v, s_tmp, &total);
    if (t < ntiles) tile_sums[t] = carry + ex;
    carry += total;
  }
}

// A tile's counts are read and its positions written in order of the
// threads (coalesced, whatever the arrays' alignment) and turned through
// LDS, where a thread's 16 items lie one word apart per 16 so that the lanes
// spread over the banks.  Loads and stores of 16 consecutive items a thread
// had taken 8.5 us at 500,000 counts, now 4.9.  OFFSETS: tile_sums already
// holds exclusive offsets.  total, if not null, receives pos[m].
template <bool OFFSETS>
__global__ __launch_bounds__(kScanBlock) void k_scan_apply(
    int32_t m, const int32_t* __restrict__ counts,
    const int64_t* __restrict__ tile_sums, int32_t* __restrict__ pos,
    int32_t* __restrict__ status, int32_t* __restrict__ total) {
  __shared__ int64_t s_tmp[kScanBlock / kWave];
  __shared__ int32_t s_item[kScanTile + kScanTile / kScanItems];
  const int tid = threadIdx.x;
  const int64_t tile = (int64_t)blockIdx.x * kScanTile;
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    const int e = q * kScanBlock + tid;
    s_item[e + e / kScanItems] = tile + e < m ? counts[tile + e] : 0;
  }
  int64_t before = 0;
  if (OFFSETS) {
    before = tile_sums[blockIdx.x];
  } else {
    int64_t mine = 0, all;
    for (int32_t t = tid; t < (int32_t)blockIdx.x; t += kScanBlock) mine += tile_sums[t];
    block_exclusive_sum(mine, s_tmp, &all);
    before = all;
  }
  __syncthreads();
  int32_t item[kScanItems];
  int64_t v = 0;
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    item[q] = s_item[tid * (kScanItems + 1) + q];
    v += item[q];
  }
  int64_t in_tile;
  int64_t run = before + block_exclusive_sum(v, s_tmp, &in_tile);
  if (blockIdx.x == 0 && tid == 0) pos[0] = 0;
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    run += item[q];
    s_item[tid * (kScanItems + 1) + q] = (int32_t)run;
  }
  // Counts are not negative: the thread's last sum is its largest.
  if (run > INT_MAX) atomicOr(status, 2);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < kScanItems; ++q) {
    const int e = q * kScanBlock + tid;
    if (tile + e < m) {
      const int32_t sum = s_item[e + e / kScanItems];
      pos[tile + e + 1] = sum;
      if (total && tile + e + 1 == m) *total = sum;
    }
  }
}

}  // namespace

int device_counts_to_pos(int32_t m, const int32_t* counts, int32_t* pos,
                         int32_t* status, hipStream_t st, int32_t* total) {
  const int32_t ntiles = (int32_t)(((int64_t)m + kScanTile - 1) / kScanTile);
  if (m == 0) {
    TH_CHECK(hipMemsetAsync(pos, 0, sizeof(int32_t), st));
    if (total) TH_CHECK(hipMemsetAsync(total, 0, sizeof(int32_t), st));
    return 0;
  }
  int64_t* sums = (int64_t*)workspace(sizeof(int64_t) * (size_t)ntiles, 3);
  if (!sums) return 1;
  k_scan_tiles<<<ntiles, kScanBlock, 0, st>>>(m, counts, sums);
  if (ntiles <= kScanDirectTiles) {
    k_scan_apply<false><<<ntiles, kScanBlock, 0, st>>>(m, counts, sums, pos, status, total);
  } else {
    k_scan_tile_sums<<<1, kScanBlock, 0, st>>>(ntiles, sums);
    k_scan_apply<true><<<ntiles, kScanBlock, 0, st>>>(m, counts, sums, pos, status, total);
  }
  TH_LAUNCH_CHECK("counts_to_pos");
  return 0;
}

}  // namespace taco_hip

using namespace taco_hip;

namespace {

int check_spgemm_operands(taco_tensor_t* C, taco_tensor_t* A, taco_tensor_t* B,
                          CsrView* a, CsrView* b) {
  if (int rc = view_csr(A, "A", a)) return rc;
  if (int rc = view_csr(B, "B", b)) return rc;
  TH_REQUIRE(C && C->order == 2 && C->mode_types[0] == taco_mode_dense &&
                 C->mode_types[1] == taco_mode_sparse,
             "spgemm: C must be CSR");
  TH_REQUIRE(a->n == b->m, "spgemm: A has %d columns, B has %d rows", a->n,
             b->m);
  TH_REQUIRE(C->dimensions[0] == a->m && C->dimensions[1] == b->n,
             "spgemm: C is %dx%d, expected %dx%d", C->dimensions[0],
             C->dimensions[1], a->m, b->n);
  TH_REQUIRE(a->vt == VType::F64 && b->vt == VType::F64 && C->csize == 64,
             "spgemm: f64 values only");
  return 0;
}

}  // namespace

namespace {

void publish(taco_tensor_t* C, int32_t* cpos, int32_t* ccrd, double* cvals, int32_t nnz) {
  C->indices[1][0] = (uint8_t*)cpos;
  C->indices[1][1] = (uint8_t*)ccrd;
  C->vals = (uint8_t*)cvals;
  C->vals_size = nnz;
}

// taco's two-phase protocol as it stands: a count pass and a fill pass, each
// building the row set (rows limited to kHashCap distinct columns).  Used
// when the candidate total exceeds the int32 range of the one-sort scratch.
int assemble_two_pass(const CsrView& a, const CsrView& b, taco_tensor_t* C,
                      hipStream_t st) {
  const int32_t m = a.m;
  int32_t* cpos = (int32_t*)taco_hip_unified_alloc(sizeof(int32_t) * ((size_t)m + 1));
  if (!cpos) return 1;
  // Workspace: counts[m] and a status word.
  char* ws = (char*)workspace(sizeof(int32_t) * ((size_t)m + 64), 2);
  if (!ws) {
    taco_hip_unified_free(cpos);
    return 1;
  }
  int32_t* status = (int32_t*)ws;
  int32_t* counts = (int32_t*)(ws + 256);
  int rc = 0;
  do {
    if (hipMemsetAsync(status, 0, sizeof(int32_t), st) != hipSuccess) {
      rc = fail("spgemm: memset failed");
      break;
    }
    const unsigned grid = (unsigned)(((int64_t)m + kWavesPerBlock - 1) / kWavesPerBlock);
    if (m > 0)
      k_spgemm_symbolic<false><<<grid, 256, 0, st>>>(
          m, a.pos, a.crd, b.pos, b.crd, counts, nullptr, nullptr, status);
    if ((rc = device_counts_to_pos(m, counts, cpos, status, st))) break;
    int32_t host[2] = {0, 0};
    if (hipMemcpyAsync(&host[0], cpos + m, sizeof(int32_t),
                       hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipMemcpyAsync(&host[1], status, sizeof(int32_t),
                       hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess) {
      rc = fail("spgemm: reading nnz(C) failed");
      break;
    }
    if (host[1] & 1) {
      rc = fail("spgemm: a row of C has more than %d distinct columns, the "
                "limit of the LDS row kernel (two-pass form, used when the "
                "candidate total exceeds the int32 range)", kHashCap);
      break;
    }
    if (host[1] & 2) {
      rc = fail("spgemm: nnz(C) exceeds the int32 index range");
      break;
    }
    const int32_t nnz = host[0];
    int32_t* ccrd = (int32_t*)taco_hip_unified_alloc(sizeof(int32_t) * (size_t)nnz);
    double* cvals = (double*)taco_hip_unified_alloc(sizeof(double) * (size_t)nnz);
    if (nnz > 0 && (!ccrd || !cvals)) {
      taco_hip_unified_free(ccrd);
      taco_hip_unified_free(cvals);
      rc = 1;
      break;
    }
    if (m > 0 && nnz > 0)
      k_spgemm_symbolic<true><<<grid, 256, 0, st>>>(
          m, a.pos, a.crd, b.pos, b.crd, nullptr, cpos, ccrd, status);
    if ((rc = finish("taco_hip_spgemm_assemble"))) {
      taco_hip_unified_free(ccrd);
      taco_hip_unified_free(cvals);
      break;
    }
    publish(C, cpos, ccrd, cvals, nnz);
    return 0;
  } while (0);
  taco_hip_unified_free(cpos);
  return rc;
}

// Workspace slots of the one-sort assemble, and of compute's rows.
constexpr int kSlotCandOff = 8, kSlotScratch = 9, kSlotLongMeta = 10, kSlotLongKeys = 11,
              kSlotSortTemp = 12, kSlotComputeRows = 13;
// Workgroups per CU of k_spgemm_numeric_short's resident grid.
constexpr int kShortBlocksPerCu = 8;

int device_cus() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0, n = 256;
    if (hipGetDevice(&dev) == hipSuccess)
      (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
    cus = n > 0 ? n : 256;
  }
  return cus;
}

// Resident grid of the short-row kernels (4 waves per workgroup, each
// taking kRowsTogether rows per step), no larger than the rows need.
unsigned short_rows_grid(int32_t m) {
  const int64_t need = ((int64_t)m + kWavesPerBlock * kRowsTogether - 1) /
                       (kWavesPerBlock * kRowsTogether);
  const int64_t resident = (int64_t)kShortBlocksPerCu * device_cus();
  return (unsigned)(need < resident ? (need > 0 ? need : 1) : resident);
}

// Rows listed by the symbolic pass (more than kHashCap distinct columns):
// candidates written out, sorted per row in global memory, deduplicated into
// their scratch regions with their distinct counts.
int assemble_long_rows(const CsrView& a, const CsrView& b, int32_t nlong,
                       const int32_t* long_rows, const int32_t* candoff, int32_t* scratch,
                       int32_t* counts, hipStream_t st) {
  char* meta = (char*)workspace(sizeof(uint32_t) * (2 * (size_t)nlong + 2), kSlotLongMeta);
  if (!meta) return 1;
  int32_t* lens = (int32_t*)meta;
  uint32_t* loff = (uint32_t*)meta + nlong + 1;
  k_spgemm_long_lengths<<<(nlong + 255) / 256, 256, 0, st>>>(nlong, long_rows, candoff, lens);
  TH_LAUNCH_CHECK("spgemm long rows");
  std::vector<int32_t> h_lens((size_t)nlong);
  TH_CHECK(hipMemcpyAsync(h_lens.data(), lens, sizeof(int32_t) * (size_t)nlong,
                          hipMemcpyDeviceToHost, st));
  TH_CHECK(hipStreamSynchronize(st));
  std::vector<uint32_t> h_off((size_t)nlong + 1, 0);
  uint64_t total = 0;
  for (int32_t r = 0; r < nlong; ++r) {
    h_off[(size_t)r] = (uint32_t)total;
    total += (uint64_t)h_lens[(size_t)r];
  }
  TH_REQUIRE(total < 0xFFFFFFFFull, "spgemm: long rows hold too many candidates");
  h_off[(size_t)nlong] = (uint32_t)total;
  TH_CHECK(hipMemcpyAsync(loff, h_off.data(), sizeof(uint32_t) * ((size_t)nlong + 1),
                          hipMemcpyHostToDevice, st));
  uint32_t* keys = (uint32_t*)workspace(sizeof(uint32_t) * 2 * (size_t)(total ? total : 1),
                                        kSlotLongKeys);
  if (!keys) return 1;
  uint32_t* sorted = keys + total;
  const unsigned grid = (unsigned)(((int64_t)nlong + kWavesPerBlock - 1) / kWavesPerBlock);
  k_spgemm_long_fill<<<grid, 256, 0, st>>>(nlong, long_rows, loff, a.pos, a.crd, b.pos, b.crd,
                                           keys);
  TH_LAUNCH_CHECK("spgemm long rows: candidates");
  unsigned bits = 1;
  while (bits < 32 && (1ull << bits) < (uint64_t)(b.n > 1 ? b.n : 2)) ++bits;
  size_t temp_bytes = 0;
  TH_CHECK(rocprim::segmented_radix_sort_keys(nullptr, temp_bytes, keys, sorted,
                                              (unsigned)total, (unsigned)nlong, loff, loff + 1,
                                              0, bits, st));
  void* temp = workspace(temp_bytes ? temp_bytes : 1, kSlotSortTemp);
  if (!temp) return 1;
  TH_CHECK(rocprim::segmented_radix_sort_keys(temp, temp_bytes, keys, sorted, (unsigned)total,
                                              (unsigned)nlong, loff, loff + 1, 0, bits, st));
  k_spgemm_long_dedup<<<grid, 256, 0, st>>>(nlong, long_rows, loff, sorted, candoff, scratch,
                                            counts);
  TH_LAUNCH_CHECK("spgemm long rows: distinct columns");
  return 0;
}

// The one-sort assemble (see the file comment).  *two_pass is set when the
// candidate total exceeds the int32 range; nothing is published then.
int assemble_one_sort(const CsrView& a, const CsrView& b, taco_tensor_t* C, hipStream_t st,
                      bool* two_pass) {
  *two_pass = false;
  const int32_t m = a.m;
  // status[0]: flags (2: nnz(C) beyond int32, 4: scratch too small);
  // status[1]: long rows listed; status[2]: candidate-total flags (2);
  // status[3]: candidates; status[4]: nnz(C); status[5]: rows of
  // more than 64 candidates or A entries.
  char* ws = (char*)workspace(256 + sizeof(int32_t) * 3 * ((size_t)m + 1), 2);
  int32_t* candoff = (int32_t*)workspace(sizeof(int32_t) * ((size_t)m + 1), kSlotCandOff);
  if (!ws || !candoff) return 1;
  int32_t* status = (int32_t*)ws;
  int32_t* counts = (int32_t*)(ws + 256);
  int32_t* long_rows = counts + m + 1;
  int32_t* mid_rows = long_rows + m + 1;
  int32_t* cpos = (int32_t*)taco_hip_unified_alloc(sizeof(int32_t) * ((size_t)m + 1));
  if (!cpos) return 1;
  const unsigned short_grid = short_rows_grid(m);
  int rc = 0;
  do {
    // The status words are cleared by k_spgemm_row_cands (a memset costs a
    // runtime call of its own).
    if (m > 0)
      k_spgemm_row_cands<<<(unsigned)(((int64_t)m * kCandLanes + 255) / 256), 256, 0, st>>>(
          m, a.pos, a.crd, b.pos, counts, status);
    else if (hipMemsetAsync(status, 0, 16 * sizeof(int32_t), st) != hipSuccess) {
      rc = fail("spgemm: memset failed");
      break;
    }
    if ((rc = device_counts_to_pos(m, counts, candoff, status + 2, st, status + 3))) break;
    size_t cap_bytes = workspace_size(kSlotScratch);
    int32_t* scratch = (int32_t*)workspace(cap_bytes ? cap_bytes : 4096, kSlotScratch);
    if (!scratch) {
      rc = 1;
      break;
    }
    cap_bytes = workspace_size(kSlotScratch);
    int32_t host[5] = {0, 0, 0, 0, 0};  // status[0..4]
    for (int attempt = 0; attempt < 2; ++attempt) {
      if (attempt > 0 && hipMemsetAsync(status, 0, 2 * sizeof(int32_t), st) != hipSuccess) {
        rc = fail("spgemm: memset failed");
        break;
      }
      if (m > 0) {
        k_spgemm_symbolic_short<<<short_grid, 256, 0, st>>>(
            m, a.pos, a.crd, (int32_t)a.nnz, b.pos, b.crd, (int32_t)b.nnz, candoff,
            (int64_t)(cap_bytes / sizeof(int32_t)), scratch, counts, mid_rows, status);
        k_spgemm_symbolic_mid<<<mid_grid(m), 256, 0, st>>>(
            mid_rows, a.pos, a.crd, b.pos, b.crd, (int32_t)b.nnz, candoff, scratch, counts,
            long_rows, status);
      }
      if ((rc = device_counts_to_pos(m, counts, cpos, status, st, status + 4))) break;
      if ((rc = read_back_i32(status, 5, host, st))) break;
      if ((host[2] & 2) || !(host[0] & 4)) break;
      // The scratch was too small for the candidate total: grow, run again.
      cap_bytes = sizeof(int32_t) * (size_t)host[3];
      scratch = (int32_t*)workspace(cap_bytes, kSlotScratch);
      if (!scratch) {
        rc = 1;
        break;
      }
    }
    if (rc) break;
    if (host[2] & 2) {
      *two_pass = true;
      break;
    }
    TH_REQUIRE(!(host[0] & 4), "spgemm: scratch sizing failed");
    if (host[1] > 0) {
      if ((rc = assemble_long_rows(a, b, host[1], long_rows, candoff, scratch, counts, st)))
        break;
      if (hipMemsetAsync(status, 0, sizeof(int32_t), st) != hipSuccess) {
        rc = fail("spgemm: memset failed");
        break;
      }
      if ((rc = device_counts_to_pos(m, counts, cpos, status, st, status + 4))) break;
      if ((rc = read_back_i32(status, 5, host, st))) break;
    }
    if (host[0] & 2) {
      rc = fail("spgemm: nnz(C) exceeds the int32 index range");
      break;
    }
    const int32_t nnz = host[4];
    int32_t* ccrd = (int32_t*)taco_hip_unified_alloc(sizeof(int32_t) * (size_t)nnz);
    double* cvals = (double*)taco_hip_unified_alloc(sizeof(double) * (size_t)nnz);
    if (nnz > 0 && (!ccrd || !cvals)) {
      taco_hip_unified_free(ccrd);
      taco_hip_unified_free(cvals);
      rc = 1;
      break;
    }
    if (m > 0 && nnz > 0)
      k_spgemm_compact<<<(unsigned)(((int64_t)m + kCompactRows - 1) / kCompactRows), 256, 0,
                         st>>>(m, candoff, cpos, scratch, ccrd);
    if ((rc = finish("taco_hip_spgemm_assemble"))) {
      taco_hip_unified_free(ccrd);
      taco_hip_unified_free(cvals);
      break;
    }
    publish(C, cpos, ccrd, cvals, nnz);
    return 0;
  } while (0);
  taco_hip_unified_free(cpos);
  return rc;
}

}  // namespace

extern "C" int taco_hip_spgemm_assemble(taco_tensor_t* C, taco_tensor_t* A,
                                        taco_tensor_t* B) {
  CsrView a, b;
  if (int rc = check_spgemm_operands(C, A, B, &a, &b)) return rc;
  hipStream_t st = current_stream();
  bool two_pass = false;
  if (int rc = assemble_one_sort(a, b, C, st, &two_pass)) return rc;
  return two_pass ? assemble_two_pass(a, b, C, st) : 0;
}

extern "C" int taco_hip_spgemm_compute(taco_tensor_t* C, taco_tensor_t* A,
                                       taco_tensor_t* B) {
  CsrView a, b, c;
  if (int rc = check_spgemm_operands(C, A, B, &a, &b)) return rc;
  if (int rc = view_csr(C, "C", &c)) return rc;
  if (a.m == 0 || c.nnz == 0) return finish("taco_hip_spgemm_compute");
  hipStream_t st = current_stream();
  if (a.nnz == 0 || b.nnz == 0) return finish("taco_hip_spgemm_compute");  // no products
  // Workspace: the number of rows of more than 64 candidates, a list for
  // them, and a flag for every row.
  const size_t flag_bytes = ((size_t)a.m + 3) / 4 * 4;
  int32_t* listed = (int32_t*)workspace(
      256 + sizeof(int32_t) * (size_t)a.m + flag_bytes, kSlotComputeRows);
  if (!listed) return 1;
  int32_t* list = listed + 64;
  uint8_t* mid = (uint8_t*)(list + a.m);
  k_spgemm_numeric_short<<<short_rows_grid(a.m), 256, 0, st>>>(
      a.m, a.pos, a.crd, (const double*)a.vals, (int32_t)a.nnz, b.pos, b.crd,
      (const double*)b.vals, (int32_t)b.nnz, c.pos, (double*)c.vals, mid, listed);
  k_spgemm_list_mid<<<(unsigned)(((int64_t)a.m + kListRows - 1) / kListRows), 256, 0, st>>>(
      a.m, (const uint32_t*)mid, list, listed);
  k_spgemm_numeric_mid<<<mid_grid(a.m), 256, 0, st>>>(
      list, listed, a.pos, a.crd, (const double*)a.vals, b.pos, b.crd, (const double*)b.vals,
      (int32_t)b.nnz, c.pos, c.crd, (double*)c.vals);
  return finish("taco_hip_spgemm_compute");
}

extern "C" int taco_hip_device_exclusive_scan(const int32_t* counts, int32_t m,
                                              int32_t* pos) {
  hipStream_t st = current_stream();
  int32_t* status = (int32_t*)workspace(sizeof(int32_t), 7);
  if (!status) return 1;
  TH_CHECK(hipMemsetAsync(status, 0, sizeof(int32_t), st));
  if (int rc = device_counts_to_pos(m, counts, pos, status, st)) return rc;
  int32_t host = 0;
  TH_CHECK(hipMemcpyAsync(&host, status, sizeof(int32_t), hipMemcpyDeviceToHost, st));
  TH_CHECK(hipStreamSynchronize(st));
  TH_REQUIRE(host == 0, "exclusive scan: total exceeds the int32 index range");
  return 0;
}

// Hand-written HIP SpMV kernels, y(i) = A(i,j) * x(j), A in CSR.
//
// Four schedules, each the wave64 form of a schedule family taco emits or
// that the power-law workload needs:
//   THREAD_PER_ROW  taco's default GPU schedule, split(i,256) -> GPUBlock /
//                   GPUThread (reference src/index_notation/
//                   transformations.cpp:1585-1596): the generated body
//                   `for (jA = pos[i]; jA < pos[i+1]; jA++) y += A*x[crd]`.
//   GROUP_PER_ROW   scheduleSpMVRowsGPU (test/tests-scheduling-eval.cpp:
//                   211-223): a lane group strides one row's entries and the
//                   group reduces (GPUWarpReduction) — here a shuffle tree
//                   within the 64-lane wave instead of lane 0's serial loop
//                   (codegen_cuda.cpp:875-890).
//   NNZ_SPLIT       scheduleSpMVGPU / scheduleSpMVSplitPosGPU (tests-
//                   scheduling-eval.cpp:193-209, 233-247): fuse(i,j) -> pos ->
//                   split into fixed entry chunks per thread, row found by
//                   binary search (taco_binarySearchBefore, codegen_cuda.cpp:
//                   89-109), atomics at row changes, wave-aggregated when the
//                   whole wave is in one row (atomicAddWarp, codegen_cuda.cpp:
//                   142-159, here over 64 lanes).
//   MERGE_PATH      merge-path decomposition of (row ends, entries): equal
//                   work per thread regardless of row lengths; within a
//                   workgroup the partial rows are combined by a segmented
//                   scan; rows crossing workgroups are fixed up in order from
//                   a carry array by a second kernel.  No atomics, so results
//                   are deterministic run to run.

#include <climits>
#include <mutex>

#include "common.h"
#include "device.h"

namespace taco_hip {
namespace {

template <typename T>
__global__ __launch_bounds__(1024) void k_spmv_thread_per_row(
    int32_t m, const int32_t* __restrict__ pos, const int32_t* __restrict__ crd,
    const T* __restrict__ vals, const T* __restrict__ x, T* __restrict__ y) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  T acc = 0;
  const int32_t end = pos[i + 1];
  for (int32_t p = pos[i]; p < end; ++p) acc += vals[p] * x[crd[p]];
  y[i] = acc;
}

template <typename T, int G>
__global__ __launch_bounds__(1024) void k_spmv_group_per_row(
    int32_t m, int32_t rows_per_group, const int32_t* __restrict__ pos,
    const int32_t* __restrict__ crd, const T* __restrict__ vals,
    const T* __restrict__ x, T* __restrict__ y) {
  const int lane = threadIdx.x & (G - 1);
  const int64_t group = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / G;
  const int64_t first = group * rows_per_group;
  for (int32_t rr = 0; rr < rows_per_group; ++rr) {
    const int64_t i = first + rr;
    if (i >= m) break;  // uniform across the group
    T acc = 0;
    const int32_t end = pos[i + 1];
    for (int32_t p = pos[i] + lane; p < end; p += G)
      acc += stream_load(vals + p) * x[stream_load(crd + p)];
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, G);
    if (lane == 0) y[i] = acc;
  }
}

// Largest r in [0, m) with pos[r] <= z (the row holding entry z < nnz).
__device__ __forceinline__ int32_t row_of_entry(const int32_t* pos, int32_t m,
                                                int64_t z) {
  int32_t lo = 0, hi = m;  // pos[lo] <= z < pos[hi]
  while (hi - lo > 1) {
    int32_t mid = lo + (hi - lo) / 2;
    if ((int64_t)pos[mid] <= z)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

template <typename T, int K>
__global__ __launch_bounds__(1024) void k_spmv_nnz_split(
    int32_t m, int64_t nnz, const int32_t* __restrict__ pos,
    const int32_t* __restrict__ crd, const T* __restrict__ vals,
    const T* __restrict__ x, T* __restrict__ y, bool coarse) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t z0 = t * K;
  int32_t r = 0;
  T acc = 0;
  const bool active = z0 < nnz;
  if (active) {
    const int64_t z1 = z0 + K < nnz ? z0 + K : nnz;
    r = row_of_entry(pos, m, z0);
    int64_t rend = pos[r + 1];
    for (int64_t z = z0; z < z1; ++z) {
      while (z >= rend) {  // skips empty rows too
        if (acc != T(0)) atomic_add(y + r, acc, coarse);
        acc = 0;
        ++r;
        rend = pos[r + 1];
      }
      acc += stream_load(vals + z) * x[stream_load(crd + z)];
    }
  }
  // Wave-aggregated flush: one atomic when every active lane ends in the
  // same row, otherwise one per lane.
  const uint64_t act = __ballot(active);
  const int leader = act ? __ffsll((unsigned long long)act) - 1 : 0;
  const int32_t r_lead = __shfl(r, leader, kWave);
  const bool same = !active || r == r_lead;
  if (__ballot(same) == ~0ull) {
    T s = wave_sum(active ? acc : T(0));
    if ((int)__lane_id() == leader && act) atomic_add(y + r_lead, s, coarse);
  } else if (active) {
    atomic_add(y + r, acc, coarse);
  }
}

// Merge-path SpMV: one workgroup of 256 threads per IPW = 256*K merge items.
template <typename T, int K>
__global__ __launch_bounds__(256) void k_spmv_merge(
    int32_t m, int64_t nnz, const int32_t* __restrict__ pos,
    const int32_t* __restrict__ crd, const T* __restrict__ vals,
    const T* __restrict__ x, T* __restrict__ y, int32_t* __restrict__ carry_row,
    T* __restrict__ carry_val) {
  constexpr int B = 256;
  constexpr int IPW = B * K;
  constexpr int NW = B / kWave;
  __shared__ T s_prod[IPW];
  __shared__ int32_t s_row_end[IPW + 1];
  __shared__ int64_t s_coord[2];
  __shared__ int32_t s_wlast[NW], s_wfirst[NW];
  __shared__ T s_wval[NW];

  const int tid = threadIdx.x;
  const int wave = tid / kWave;
  const int lane = tid % kWave;
  const int64_t total = (int64_t)m + nnz;
  const int64_t d0 = (int64_t)blockIdx.x * IPW;
  const int64_t d1 = d0 + IPW < total ? d0 + IPW : total;

  // Tile coordinates: wave 0 finds the start split, wave 1 the end split.
  if (wave < 2) {
    const int64_t r = wave_merge_search(pos, m, nnz, wave == 0 ? d0 : d1);
    if (lane == 0) s_coord[wave] = r;
  }
  __syncthreads();
  const int64_t r0 = s_coord[0], r1 = s_coord[1];
  const int64_t z0 = d0 - r0;
  const int nrows = (int)(r1 - r0);       // row ends inside the tile
  const int nz = (int)((d1 - r1) - z0);   // entries inside the tile

  // Stage the tile's row ends (plus the end of the row in progress at the
  // tile end) and the products A_z * x[crd_z], coalesced.
  for (int q = tid; q <= nrows; q += B) {
    const int64_t rr = r0 + 1 + q;
    s_row_end[q] = rr <= m ? pos[rr] : INT_MAX;
  }
  {
    int32_t c[K];
    T v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int q = tid + k * B;
      c[k] = 0;
      v[k] = 0;
      if (q < nz) {
        c[k] = stream_load(crd + z0 + q);
        v[k] = stream_load(vals + z0 + q);
      }
    }
    T xv[K];
#pragma unroll
    for (int k = 0; k < K; ++k) xv[k] = (tid + k * B < nz) ? x[c[k]] : T(0);
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (tid + k * B < nz) s_prod[tid + k * B] = v[k] * xv[k];
  }
  __syncthreads();

  // This thread's start on the tile-local merge path.
  const int dl = tid * K;
  const int tile_items = nrows + nz;
  int rl, zl;
  if (dl >= tile_items) {
    rl = nrows;
    zl = nz;
  } else {
    int lo = dl - nz > 0 ? dl - nz : 0;
    int hi = dl < nrows ? dl : nrows;
    while (lo < hi) {
      const int p = (lo + hi) >> 1;
      if ((int64_t)s_row_end[p] <= z0 + dl - p - 1)
        lo = p + 1;
      else
        hi = p;
    }
    rl = lo;
    zl = dl - lo;
  }

  // Consume K merge items.  Completed rows after the first are final within
  // this thread; the first completed row still lacks the partial sums of the
  // threads before it, added after the scan.
  T acc = 0;
  bool have_first = false;
  int first_rl = 0;
  T first_val = 0;
  const int items = tile_items - dl < K ? (tile_items - dl > 0 ? tile_items - dl : 0) : K;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (k < items) {
      if (z0 + zl < (int64_t)s_row_end[rl]) {
        acc += s_prod[zl];
        ++zl;
      } else {
        if (!have_first) {
          have_first = true;
          first_rl = rl;
          first_val = acc;
        } else {
          y[r0 + rl] = acc;
        }
        acc = 0;
        ++rl;
      }
    }
  }

  // Segmented inclusive scan of the carries (row in progress, partial sum)
  // over the workgroup, keyed by row.
  T inc = wave_segmented_inclusive_sum(acc, rl);
  if (lane == kWave - 1) {
    s_wlast[wave] = rl;
    s_wval[wave] = inc;
  }
  if (lane == 0) s_wfirst[wave] = rl;
  __syncthreads();
  int cin_row = -1;
  T cin = 0;
  if (wave > 0) {
    cin_row = s_wlast[wave - 1];
    cin = s_wval[wave - 1];
    for (int w2 = wave - 2; w2 >= 0; --w2) {
      if (s_wfirst[w2 + 1] == cin_row && s_wlast[w2] == cin_row)
        cin += s_wval[w2];
      else
        break;
    }
    if (rl == cin_row) inc += cin;
  }
  T prev_inc = __shfl_up(inc, 1, kWave);
  int prev_row = __shfl_up(rl, 1, kWave);
  if (lane == 0) {
    prev_inc = cin;
    prev_row = cin_row;
  }
  if (have_first) {
    T v = first_val;
    if (prev_row == first_rl) v += prev_inc;
    y[r0 + first_rl] = v;
  }
  if (tid == B - 1) {
    carry_row[blockIdx.x] = (int32_t)(r0 + rl);
    carry_val[blockIdx.x] = inc;
  }
}

// Adds each row's cross-workgroup partial sums, in a fixed order.  A wave to
// 64 slots: the runs of equal rows are added in the lanes, and the wave that
// holds a run's first slot also adds what follows in the next 64 slots, and
// so on, a slot a lane.  The wave waits for memory twice, whatever the runs
// within its slots (a lane that looked along its run waited once a slot): a
// 50,000-row power-law matrix with a run of 13 slots, f64, 13.6 -> 11.9 us a
// call, 200,000 rows 30.2 -> 27.9.
template <typename T>
__global__ __launch_bounds__(256) void k_spmv_merge_fixup(
    int32_t nblocks, int32_t m, const int32_t* __restrict__ carry_row,
    const T* __restrict__ carry_val, T* __restrict__ y) {
  const int32_t b = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x % kWave;
  const int32_t first = b - lane;
  if (first >= nblocks) return;
  const int32_t r = b < nblocks ? carry_row[b] : -1;
  T s = b < nblocks ? carry_val[b] : T(0);
  // The rows before the wave's first slot and after its last.
  const int32_t outside = first > 0 ? carry_row[first - 1] : -1;
  const int32_t after = first + kWave < nblocks ? carry_row[first + kWave] : -1;
  int32_t before = __shfl_up(r, 1, kWave);
  if (lane == 0) before = outside;
  const bool head = r >= 0 && r < m && before != r;
  const T old = head ? y[r] : T(0);
  // s: the sum of the lane's run from the lane on.  Most waves hold none of
  // two slots.
  if (__ballot(r >= 0 && lane > 0 && before == r)) {
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const T u = __shfl_down(s, off, kWave);
      const int32_t ru = __shfl_down(r, off, kWave);
      if (lane + off < kWave && ru == r) s += u;
    }
  }
  const int32_t last = __builtin_amdgcn_readlane(r, kWave - 1);
  const bool open = head && r == last && after == last;
  if (__ballot(open)) {
    T more = 0;
    for (int32_t c = first + kWave + lane;; c += kWave) {
      // Slots of a run are consecutive: lanes past its end add nothing.
      const bool in_run = c < nblocks && carry_row[c] == last;
      more += in_run ? carry_val[c] : T(0);
      if (__ballot(!in_run)) break;
    }
    more = wave_sum(more);
    if (open) s += more;
  }
  if (head) y[r] = old + s;
}

// The merge path's form for few entries (small_spmv): one launch, no search
// and no carries.  G lanes take a row; rows of more than kSmallOwn entries a
// lane are left for the workgroup's teams of 16 lanes (up to kSmallTeamRow
// entries), its waves (up to kSmallWaveRow) or all its threads, so that many
// of them are summed side by side.  Sums are taken in a fixed order, without
// atomics, like the merge path's.
//
// Such calls cost launches and chains of dependent loads, not bandwidth: a
// merge-path call launches twice (3.5 us each back to back) and searches its
// tile's corners before it loads an entry.
//
// Neighbouring rows go to different workgroups (row i to workgroup i %
// gridDim.x): long rows that lie together, as the border or a dense block of
// an operator, are spread over the CUs, of which each gathers one line of x
// a cycle at most.  Short regular rows pay for the lines they share (16,000
// rows of 4, f64, 5.9 us; 4.4 with runs of eight rows to a workgroup, which
// would take 25 for nine neighbouring rows of 5000 and not 8.4).  The number of
// workgroups is odd, so that long rows at a power of two's distance are spread
// as well; small grids are widened to kSmallSpread (1000 rows of 10 in 33
// workgroups 2.4 us of kernel time, in 5 3.5).  `stride` is the grid's size: a
// kernel that reads gridDim needs arguments from the runtime, 0.3 us a launch.
constexpr int kSmallOwn = 16;
constexpr int kSmallThreads = 1024;
constexpr int kSmallAhead = 16;
constexpr int kSmallTeam = 16;
constexpr int32_t kSmallTeamRow = kSmallTeam * kSmallAhead;
constexpr int32_t kSmallWaveRow = 2 * kWave * kSmallAhead;
// Workgroups, rows allowing.
constexpr int kSmallSpread = 32;

// Sum of the products of entries [q0, q1), every TEAM-th from the lane's,
// AHEAD of them loaded at a time.
template <typename T, int TEAM, int AHEAD>
__device__ __forceinline__ T small_row_part(int32_t q0, int32_t q1, int lane,
                                            const int32_t* __restrict__ crd,
                                            const T* __restrict__ vals,
                                            const T* __restrict__ x) {
  T s = 0;
  for (int32_t p = q0 + lane; p < q1; p += AHEAD * TEAM) {
    T v[AHEAD], xv[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      // Entries past the end repeat the lane's first one and add nothing.
      const int32_t q = p + u * TEAM < q1 ? p + u * TEAM : p;
      v[u] = vals[q];
      xv[u] = x[crd[q]];
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (p + u * TEAM < q1) s += v[u] * xv[u];
  }
  return s;
}
// Repeated entries cost loads too: a row of 34 entries takes 4 a lane of its
// team, not 16.
template <typename T, int TEAM>
__device__ __forceinline__ T small_row_sum(int32_t q0, int32_t q1, int lane,
                                           const int32_t* __restrict__ crd,
                                           const T* __restrict__ vals,
                                           const T* __restrict__ x) {
  return q1 - q0 <= 4 * TEAM   ? small_row_part<T, TEAM, 4>(q0, q1, lane, crd, vals, x)
         : q1 - q0 <= 8 * TEAM ? small_row_part<T, TEAM, 8>(q0, q1, lane, crd, vals, x)
                               : small_row_part<T, TEAM, kSmallAhead>(q0, q1, lane, crd, vals, x);
}

template <typename T, int G>
__global__ __launch_bounds__(kSmallThreads) void k_spmv_small(
    int32_t m, int32_t stride, const int32_t* __restrict__ pos,
    const int32_t* __restrict__ crd, const T* __restrict__ vals, const T* __restrict__ x,
    T* __restrict__ y) {
  constexpr int kRows = kSmallThreads / G;
  constexpr int kTeams = kSmallThreads / kSmallTeam, kWaves = kSmallThreads / kWave;
  constexpr int kAhead = 4;
  __shared__ int32_t s_team[kRows], s_wave[kRows], s_all[kRows];
  __shared__ T s_sum[kWaves];
  __shared__ int s_count[3];
  const int tid = threadIdx.x, sub = tid % G, slot = tid / G;
  const int64_t row0 = blockIdx.x;
  const int64_t i = row0 + (int64_t)slot * stride;
  const int32_t p0 = i < m ? pos[i] : 0, p1 = i < m ? pos[i + 1] : 0;
  const bool is_long = p1 - p0 > kSmallOwn * G;
  if (tid < 3) s_count[tid] = 0;
  __syncthreads();
  if (sub == 0 && is_long) {
    if (p1 - p0 <= kSmallTeamRow)
      s_team[atomicAdd(&s_count[0], 1)] = slot;
    else if (p1 - p0 <= kSmallWaveRow)
      s_wave[atomicAdd(&s_count[1], 1)] = slot;
    else
      s_all[atomicAdd(&s_count[2], 1)] = slot;
  }
  T acc = 0;
  for (int32_t p = is_long ? p1 : p0 + sub; p < p1; p += kAhead * G) {
    T v[kAhead], xv[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      // Entries past the end repeat the lane's first one and add nothing.
      const int32_t q = p + u * G < p1 ? p + u * G : p;
      v[u] = vals[q];
      xv[u] = x[crd[q]];
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      if (p + u * G < p1) acc += v[u] * xv[u];
  }
#pragma unroll
  for (int off = G / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, G);
  if (sub == 0 && i < m && !is_long) y[i] = acc;
  __syncthreads();
  // Each long row's sum does not depend on the order of the lists.  Waves
  // take rows from the last wave on, teams from the first.
  for (int k = tid / kSmallTeam; k < s_count[0]; k += kTeams) {
    const int64_t row = row0 + (int64_t)s_team[k] * stride;
    T s = small_row_sum<T, kSmallTeam>(pos[row], pos[row + 1], tid % kSmallTeam, crd, vals, x);
#pragma unroll
    for (int off = kSmallTeam / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, kSmallTeam);
    if (tid % kSmallTeam == 0) y[row] = s;
  }
  for (int k = kWaves - 1 - tid / kWave; k < s_count[1]; k += kWaves) {
    const int64_t row = row0 + (int64_t)s_wave[k] * stride;
    T s = small_row_sum<T, kWave>(pos[row], pos[row + 1], tid % kWave, crd, vals, x);
    s = wave_sum(s);
    if (tid % kWave == 0) y[row] = s;
  }
  for (int k = 0; k < s_count[2]; ++k) {
    const int64_t row = row0 + (int64_t)s_all[k] * stride;
    T s = small_row_sum<T, kSmallThreads>(pos[row], pos[row + 1], tid, crd, vals, x);
    s = wave_sum(s);
    if (tid % kWave == 0) s_sum[tid / kWave] = s;
    __syncthreads();
    if (tid == 0) {
      T all = 0;
      for (int w = 0; w < kWaves; ++w) all += s_sum[w];
      y[row] = all;
    }
    __syncthreads();
  }
}

// Where this form is taken; times are f64, this form against the merge path.
//   Few entries: 1000 rows of 10 3.5 against 7.8 us, 8192 of 8 4.7 : 8.4.
//     Long rows that lie together: 512 of 64 among 10,500 of 3 5.5 : 8.3, 30
//     of 2000 4.1 : 7.4, a power law of 4000 rows 6.2 : 8.0 (with the whole
//     workgroup taking one long row after another 804, 98 and 21 us).  The
//     line at 65,536 entries is not where the two meet: 131,072 in rows of 8
//     take 5.3 : 8.5.
//   No row that one workgroup takes too long for: a row holds at most n
//     entries (one each of its columns).  Rows of 16,384 entries 7.0 : 7.9
//     (four of them) and 8.5 : 9.0 (one among 12,000 of 2), of 24,000 13.2 :
//     9.7; in f32 24,000 take 8.6 : 9.5.
//   Not too many rows, which lie apart in pos and y here: 250,000 rows 9.0 :
//     9.6, 500,000 16.2 : 11.2.
constexpr int64_t kSmallEntries = 1 << 16;
constexpr int64_t kSmallRows = 1 << 18;
template <typename T>
bool small_spmv(const CsrView& a) {
  const int64_t longest = a.nnz < a.n ? a.nnz : a.n;
  return a.nnz <= kSmallEntries && a.m <= kSmallRows &&
         longest <= (sizeof(T) == 8 ? 16384 : 24576);
}

// Lanes a row: about three entries of an average row to a lane.
template <typename T>
void launch_spmv_small(const CsrView& a, const T* x, T* y, hipStream_t st) {
  int g = 2;
  while (g < 64 && (int64_t)g * 3 * a.m < a.nnz) g <<= 1;
  const int64_t need = ((int64_t)a.m * g + kSmallThreads - 1) / kSmallThreads;
  const int64_t spread = a.m < kSmallSpread ? a.m : kSmallSpread;
  const unsigned grid = (unsigned)((need > spread ? need : spread) | 1);
#define TH_SMALL(G)                                                            \
  case G:                                                                      \
    k_spmv_small<T, G><<<grid, kSmallThreads, 0, st>>>(                        \
        a.m, (int32_t)grid, a.pos, a.crd, (const T*)a.vals, x, y);             \
    break;
  switch (g) {
    TH_SMALL(2) TH_SMALL(4) TH_SMALL(8) TH_SMALL(16) TH_SMALL(32) TH_SMALL(64)
  }
#undef TH_SMALL
}

// ext_scratch / ext_bytes: caller-provided scratch for the merge path's
// carries (the no-allocation entry point); nullptr: the library workspace.
template <typename T>
int run_spmv(const CsrView& a, const T* x, T* y, const taco_hip_schedule& s,
             void* ext_scratch = nullptr, size_t ext_bytes = 0) {
  hipStream_t st = current_stream();
  if (a.m == 0) return 0;
  const int algo = s.algo;
  if (algo == TACO_HIP_THREAD_PER_ROW) {
    int bs = s.block_size > 0 ? s.block_size : 256;
    TH_REQUIRE(bs % kWave == 0 && bs <= 1024, "spmv: bad block size %d", bs);
    unsigned grid = (unsigned)((a.m + bs - 1) / bs);
    k_spmv_thread_per_row<T><<<grid, bs, 0, st>>>(
        a.m, a.pos, a.crd, (const T*)a.vals, x, y);
    return 0;
  }
  if (algo == TACO_HIP_GROUP_PER_ROW) {
    int bs = s.block_size > 0 ? s.block_size : 256;
    int g = s.group_size > 0 ? s.group_size : 8;
    int rpg = s.rows_per_group > 0 ? s.rows_per_group : 1;
    TH_REQUIRE(bs % kWave == 0 && bs <= 1024, "spmv: bad block size %d", bs);
    int64_t groups = ((int64_t)a.m + rpg - 1) / rpg;
    int64_t threads = groups * g;
    unsigned grid = (unsigned)((threads + bs - 1) / bs);
#define TH_GPR(G)                                                          \
  case G:                                                                  \
    k_spmv_group_per_row<T, G><<<grid, bs, 0, st>>>(                       \
        a.m, rpg, a.pos, a.crd, (const T*)a.vals, x, y);                   \
    return 0;
    switch (g) {
      TH_GPR(1) TH_GPR(2) TH_GPR(4) TH_GPR(8) TH_GPR(16) TH_GPR(32) TH_GPR(64)
      default:
        return fail("spmv: group_size %d not a power of two <= 64", g);
    }
#undef TH_GPR
  }
  if (algo == TACO_HIP_NNZ_SPLIT) {
    int bs = s.block_size > 0 ? s.block_size : 256;
    int k = s.items_per_thread > 0 ? s.items_per_thread : 8;
    TH_REQUIRE(bs % kWave == 0 && bs <= 1024, "spmv: bad block size %d", bs);
    if (int rc = zero_fill(y, sizeof(T) * (size_t)a.m, st)) return rc;
    if (a.nnz == 0) return 0;
    int64_t threads = (a.nnz + k - 1) / k;
    unsigned grid = (unsigned)((threads + bs - 1) / bs);
    const bool coarse = coarse_grained(y);
#define TH_NS(K)                                                           \
  case K:                                                                  \
    k_spmv_nnz_split<T, K><<<grid, bs, 0, st>>>(a.m, a.nnz, a.pos, a.crd,  \
                                                (const T*)a.vals, x, y,    \
                                                coarse);                   \
    return 0;
    switch (k) {
      TH_NS(1) TH_NS(2) TH_NS(4) TH_NS(8) TH_NS(16) TH_NS(32)
      default:
        return fail("spmv: items_per_thread %d unsupported for NNZ_SPLIT", k);
    }
#undef TH_NS
  }
  if (algo == TACO_HIP_MERGE_PATH) {
    int k = s.items_per_thread > 0 ? s.items_per_thread : 8;
    TH_REQUIRE(s.block_size == 0 || s.block_size == 256,
               "spmv: MERGE_PATH uses 256-thread workgroups");
    TH_REQUIRE(k == 2 || k == 4 || k == 6 || k == 8 || k == 12 || k == 16,
               "spmv: items_per_thread %d unsupported for MERGE_PATH", k);
    if (small_spmv<T>(a)) {
      launch_spmv_small<T>(a, x, y, st);
      return 0;
    }
    const int64_t total = (int64_t)a.m + a.nnz;
    const int64_t ipw = 256 * (int64_t)k;
    const int64_t nblocks = (total + ipw - 1) / ipw;
    TH_REQUIRE(nblocks < INT32_MAX, "spmv: problem too large");
    const size_t need = (size_t)nblocks * (sizeof(int32_t) + sizeof(T)) + 64;
    void* ws = ext_scratch;
    if (ws) {
      TH_REQUIRE(need <= ext_bytes,
                 "spmv (no-allocation form): the merge path needs %zu bytes of scratch "
                 "for %lld rows + entries at %d items per thread; the limit is %zu bytes",
                 need, (long long)total, k, ext_bytes);
    } else {
      ws = workspace(need, 0);
      if (!ws) return 1;
    }
    int32_t* crow = (int32_t*)ws;
    T* cval = (T*)((char*)ws + ((size_t)nblocks * sizeof(int32_t) + 15) / 16 * 16);
#define TH_MP(K)                                                           \
  case K:                                                                  \
    k_spmv_merge<T, K><<<(unsigned)nblocks, 256, 0, st>>>(                 \
        a.m, a.nnz, a.pos, a.crd, (const T*)a.vals, x, y, crow, cval);     \
    break;
    switch (k) {  // one of these, as required above
      TH_MP(2) TH_MP(4) TH_MP(6) TH_MP(8) TH_MP(12) TH_MP(16)
    }
#undef TH_MP
    TH_LAUNCH_CHECK("k_spmv_merge");
    unsigned g2 = (unsigned)((nblocks + 255) / 256);
    k_spmv_merge_fixup<T><<<g2, 256, 0, st>>>((int32_t)nblocks, a.m, crow,
                                               cval, y);
    return 0;
  }
  return fail("spmv: schedule algo %d not available for SpMV", algo);
}

__global__ __launch_bounds__(256) void k_zero_fill(uint32_t* __restrict__ p, int64_t words) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += stride)
    p[i] = 0u;
}

}  // namespace

int zero_fill(void* p, size_t bytes, hipStream_t st) {
  TH_REQUIRE(bytes % 4 == 0 && ((uintptr_t)p % 4) == 0, "zero fill: %zu bytes at %p", bytes, p);
  const int64_t words = (int64_t)(bytes / 4);
  if (words == 0) return 0;
  const int64_t blocks = (words + 255) / 256;
  k_zero_fill<<<(unsigned)(blocks < 8192 ? blocks : 8192), 256, 0, st>>>((uint32_t*)p, words);
  TH_LAUNCH_CHECK("k_zero_fill");
  return 0;
}

}  // namespace taco_hip

using namespace taco_hip;

namespace {

// Scratch of the no-allocation entry point: the merge path's per-workgroup
// carries (row, partial sum), written by every workgroup before the fix-up
// kernel reads them, so nothing needs clearing between calls.  Each device
// holds its own copy until the process ends; host code uses the address
// hipGetSymbolAddress returns for the current device, never the symbol.
constexpr size_t kNoAllocScratchBytes = size_t(1) << 20;
__device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kScratchDevices] = {};

// The current device's scratch address, resolved once per device.
int noalloc_scratch(void** out) {
  int dev = 0;
  TH_CHECK(hipGetDevice(&dev));
  TH_REQUIRE(dev >= 0 && dev < kScratchDevices, "spmv (no-allocation form): device %d", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    TH_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    TH_REQUIRE(p != nullptr, "spmv (no-allocation form): no scratch address");
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return 0;
}

int spmv_entry(taco_tensor_t* y, taco_tensor_t* A, taco_tensor_t* x,
               const taco_hip_schedule* sched, bool no_alloc) {
  CsrView a;
  DenseView xv, yv;
  if (int rc = view_csr(A, "A", &a)) return rc;
  if (int rc = view_dense(x, "x", 1, &xv)) return rc;
  if (int rc = view_dense(y, "y", 1, &yv)) return rc;
  TH_REQUIRE(xv.dims[0] == a.n, "spmv: x has %d entries, A has %d columns",
             xv.dims[0], a.n);
  TH_REQUIRE(yv.dims[0] == a.m, "spmv: y has %d entries, A has %d rows",
             yv.dims[0], a.m);
  TH_REQUIRE(a.vt == xv.vt && a.vt == yv.vt,
             "spmv: A, x and y must share one value type");
  taco_hip_schedule s;
  if (sched)
    s = *sched;
  else
    taco_hip_default_schedule(0, a.m, a.nnz, 1, &s);
  void* ext = nullptr;
  if (no_alloc)
    if (int rc = noalloc_scratch(&ext)) return rc;
  const size_t ext_bytes = no_alloc ? kNoAllocScratchBytes : 0;
  int rc;
  if (a.vt == VType::F64)
    rc = run_spmv<double>(a, (const double*)xv.vals, (double*)yv.vals, s, ext, ext_bytes);
  else if (a.vt == VType::F32)
    rc = run_spmv<float>(a, (const float*)xv.vals, (float*)yv.vals, s, ext, ext_bytes);
  else
    return fail("spmv: value type must be f64 or f32");
  if (rc) return rc;
  return finish(no_alloc ? "taco_hip_spmv_compute_noalloc" : "taco_hip_spmv_compute");
}

}  // namespace

extern "C" int taco_hip_spmv_compute(taco_tensor_t* y, taco_tensor_t* A,
                                     taco_tensor_t* x,
                                     const taco_hip_schedule* sched) {
  return spmv_entry(y, A, x, sched, false);
}

extern "C" int taco_hip_spmv_compute_noalloc(taco_tensor_t* y, taco_tensor_t* A,
                                             taco_tensor_t* x,
                                             const taco_hip_schedule* sched) {
  return spmv_entry(y, A, x, sched, true);
}

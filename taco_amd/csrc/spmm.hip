// Hand-written HIP SpMM kernels, C(i,k) = A(i,j) * B(j,k): A in CSR, B and C
// dense row-major.  Value forms: f64, f32, and bf16 A/B with f32 C.
//
// Schedules (wave64 forms of the reference's GPU SpMM schedules):
//   THREAD_PER_ROW  taco's default split(i,256) -> GPUBlock/GPUThread
//                   (reference transformations.cpp:1585-1596): one thread
//                   owns a row of C and runs the generated i-j-k loop nest.
//   GROUP_PER_ROW   scheduleSpMMRowsGPU (tests-scheduling-eval.cpp:345-355):
//                   a lane group owns rows, lanes split k.
//   NNZ_SPLIT       scheduleSpMMGPU (tests-scheduling-eval.cpp:249-268):
//                   fuse(i,j) -> pos -> fixed entry chunks per lane group,
//                   lanes split k, atomics at row changes.
//   MERGE_PATH      merge-path over (row ends, entries) per lane group with
//                   lanes on k; a group's unfinished last row is written to a
//                   carry slot and added in order by a fix-up kernel.
//   MFMA            bf16 only; see spmm_mfma.hip.

#include <climits>

#include "common.h"
#include "device.h"

namespace taco_hip {

// bf16 stored as raw 16-bit patterns; widening to f32 is exact.
struct bf16_t {
  uint16_t bits;
};
__device__ __forceinline__ float widen(bf16_t v) {
  return __uint_as_float((uint32_t)v.bits << 16);
}
__device__ __forceinline__ float widen(float v) { return v; }
__device__ __forceinline__ bf16_t stream_load(const bf16_t* p) {
  return bf16_t{__builtin_nontemporal_load(&p->bits)};
}
__device__ __forceinline__ double widen(double v) { return v; }

namespace {

template <typename TA, typename TC>
__global__ __launch_bounds__(1024) void k_spmm_thread_per_row(
    int32_t m, int32_t K, const int32_t* __restrict__ pos,
    const int32_t* __restrict__ crd, const TA* __restrict__ vals,
    const TA* __restrict__ B, TC* __restrict__ C) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  TC* crow = C + i * K;
  for (int32_t k = 0; k < K; ++k) crow[k] = 0;
  for (int32_t p = pos[i]; p < pos[i + 1]; ++p) {
    const TC a = widen(vals[p]);
    const TA* brow = B + (int64_t)crd[p] * K;
    for (int32_t k = 0; k < K; ++k) crow[k] += a * widen(brow[k]);
  }
}

// G lanes per row team, CPL columns per lane (K <= G * CPL).
template <typename TA, typename TC, int G, int CPL>
__global__ __launch_bounds__(256) void k_spmm_group_per_row(
    int32_t m, int32_t K, int32_t rows_per_group,
    const int32_t* __restrict__ pos, const int32_t* __restrict__ crd,
    const TA* __restrict__ vals, const TA* __restrict__ B,
    TC* __restrict__ C) {
  const int lane = threadIdx.x & (G - 1);
  const int64_t team = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / G;
  for (int32_t rr = 0; rr < rows_per_group; ++rr) {
    const int64_t i = team * rows_per_group + rr;
    if (i >= m) break;
    TC acc[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) acc[c] = 0;
    const int32_t end = pos[i + 1];
    int32_t p = pos[i];
    for (; p + 4 <= end; p += 4) {
      int32_t j[4];
      TC a[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        j[u] = stream_load(crd + p + u);
        a[u] = widen(stream_load(vals + p + u));
      }
      TC b[4][CPL];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          const int k = lane + c * G;
          b[u][c] = k < K ? widen(B[(int64_t)j[u] * K + k]) : TC(0);
        }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int c = 0; c < CPL; ++c) acc[c] += a[u] * b[u][c];
    }
    for (; p < end; ++p) {
      const int32_t j = stream_load(crd + p);
      const TC a = widen(stream_load(vals + p));
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        const int k = lane + c * G;
        if (k < K) acc[c] += a * widen(B[(int64_t)j * K + k]);
      }
    }
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const int k = lane + c * G;
      if (k < K) C[i * K + k] = acc[c];
    }
  }
}

template <typename TA, typename TC, int G, int CPL>
__global__ __launch_bounds__(256) void k_spmm_nnz_split(
    int32_t m, int64_t nnz, int32_t K, int32_t nnz_per_team,
    const int32_t* __restrict__ pos, const int32_t* __restrict__ crd,
    const TA* __restrict__ vals, const TA* __restrict__ B,
    TC* __restrict__ C, bool coarse) {
  const int lane = threadIdx.x & (G - 1);
  const int64_t team = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / G;
  const int64_t z0 = team * nnz_per_team;
  if (z0 >= nnz) return;
  const int64_t z1 = z0 + nnz_per_team < nnz ? z0 + nnz_per_team : nnz;
  // Row holding entry z0 (taco_binarySearchBefore).
  int32_t lo = 0, hi = m;
  while (hi - lo > 1) {
    int32_t mid = lo + (hi - lo) / 2;
    if ((int64_t)pos[mid] <= z0) lo = mid; else hi = mid;
  }
  int32_t r = lo;
  int64_t rend = pos[r + 1];
  TC acc[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) acc[c] = 0;
  for (int64_t z = z0; z < z1; ++z) {
    if (z >= rend) {
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        const int k = lane + c * G;
        if (k < K) atomic_add(C + (int64_t)r * K + k, acc[c], coarse);
        acc[c] = 0;
      }
      do {
        ++r;
        rend = pos[r + 1];
      } while (z >= rend);
    }
    const int32_t j = stream_load(crd + z);
    const TC a = widen(stream_load(vals + z));
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const int k = lane + c * G;
      if (k < K) acc[c] += a * widen(B[(int64_t)j * K + k]);
    }
  }
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    const int k = lane + c * G;
    if (k < K) atomic_add(C + (int64_t)r * K + k, acc[c], coarse);
  }
}

// Value of lane `idx` (wave-uniform), in a scalar register.
template <typename T>
__device__ __forceinline__ T wave_bcast(T v, int idx) {
  if constexpr (sizeof(T) == 8) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, idx);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), idx);
    return __builtin_bit_cast(T, ((uint64_t)hi << 32) | lo);
  } else {
    return __builtin_bit_cast(T, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), idx));
  }
}

// W adjacent values, aligned as one of them.
template <typename T, int W>
struct Adjacent;
#define TH_ADJACENT(T, W)                                                        \
  template <>                                                                    \
  struct Adjacent<T, W> {                                                        \
    typedef T vec __attribute__((ext_vector_type(W), aligned(sizeof(T))));       \
  };
TH_ADJACENT(double, 1) TH_ADJACENT(double, 2) TH_ADJACENT(double, 4)
TH_ADJACENT(float, 1) TH_ADJACENT(float, 2) TH_ADJACENT(float, 4)
TH_ADJACENT(uint16_t, 1) TH_ADJACENT(uint16_t, 2) TH_ADJACENT(uint16_t, 4)
#undef TH_ADJACENT
template <int W>
__device__ __forceinline__ void load_wide(const double* p, double (&out)[W]) {
  const typename Adjacent<double, W>::vec v = *(const typename Adjacent<double, W>::vec*)p;
#pragma unroll
  for (int c = 0; c < W; ++c) out[c] = v[c];
}
template <int W>
__device__ __forceinline__ void load_wide(const float* p, float (&out)[W]) {
  const typename Adjacent<float, W>::vec v = *(const typename Adjacent<float, W>::vec*)p;
#pragma unroll
  for (int c = 0; c < W; ++c) out[c] = v[c];
}
template <int W>
__device__ __forceinline__ void load_wide(const bf16_t* p, float (&out)[W]) {
  const typename Adjacent<uint16_t, W>::vec v = *(const typename Adjacent<uint16_t, W>::vec*)p;
#pragma unroll
  for (int c = 0; c < W; ++c) out[c] = widen(bf16_t{v[c]});
}

// One wave per team.  L = ceil(K / CPL) lanes cover the K columns, each
// owning CPL adjacent ones: its first column is kl * CPL, or K - CPL where
// that would pass the end, so that every lane loads CPL columns of a B row in
// one go (16 bytes for four f32 or two f64 columns); the last two lanes may
// overlap and then hold the same sums.  The wave's S = 64 / L groups of L
// lanes take consecutive entries, so that one load instruction gathers S B
// rows; a finished row's sums are added across the groups.  Wide loads and
// full waves are what counts where B's rows come from the caches: the L1's
// data path works by the lane, whether it is of use or not.  (ONE: a wave to
// a B row, whose address and value then sit in scalar registers.)
//
// Entries are taken in blocks, U steps of S of them (S * U <= 64), whatever
// rows they belong to: a block's B rows are gathered together, then added step by
// step with the row ends in between.  The next chunk's columns and values
// load while the current one is worked on, and 64 row ends are held in the
// lanes, so no step waits for a chain of dependent loads; the walk itself is
// the same for the whole wave and runs on the scalar unit.
//
// 400,009 banded rows of 24 entries, K = 33, f32: 294 us with one row at a
// time (pos, then its entries, then B rows, each waited for; a row's last
// entries one by one; one B row to a load), 179 us now: the L1 fetches 1.7
// lines of B from L2 for an entry, 1.9 GB at the 18 TB/s that L2 delivers
// being 104 us of it.  1M-row power-law matrix, K = 64, f64: 1295 -> 1210 us,
// 64 M lines of B, at the 53 G random lines a second that the card delivers.
template <typename TA, typename TC, int CPL, int U, bool ONE>
__global__ __launch_bounds__(256) void k_spmm_merge(
    int32_t m, int64_t nnz, int32_t K, int32_t items_per_team,
    const int32_t* __restrict__ pos, const int32_t* __restrict__ crd,
    const TA* __restrict__ vals, const TA* __restrict__ B,
    TC* __restrict__ C, int64_t nteams, int32_t* __restrict__ carry_row,
    TC* __restrict__ carry_val) {
  typedef typename Adjacent<TC, CPL>::vec Out;
  const int lane = threadIdx.x % kWave;
  const int L = (K + CPL - 1) / CPL;
  // 4 groups for 10 to 16 lanes, though 10 to 12 leave room for 5 or 6: the
  // sums of a row take fewer moves, and a chunk is a whole 64 entries.
  const int S = ONE                 ? 1
                : L > 9 && L <= 16  ? 4
                : kWave / L < kWave / U ? kWave / L
                                    : kWave / U;
  const int chunk = kWave / (S * U) * (S * U);
  const int sub = ONE ? 0 : lane / L, kl = ONE ? lane : lane % L;
  const bool owns = sub < S && kl < L;  // lanes left over repeat others' loads
  const int64_t team = (int64_t)blockIdx.x * (256 / kWave) +
                       __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  if (team >= nteams) return;
  const int64_t total = (int64_t)m + nnz;
  const int64_t d0 = team * items_per_team;
  int32_t left = (int32_t)(total - d0 < items_per_team ? total - d0 : items_per_team);
  int32_t r = __builtin_amdgcn_readfirstlane((int)wave_merge_search(pos, m, nnz, d0));
  int32_t z = (int32_t)(d0 - r);
  // kStrided: a lane's columns are lane, lane + 64, ... instead, those past
  // the end repeating column K - 1.
  constexpr bool kStrided = ONE && sizeof(TC) == 8;
  const int32_t k0 = kStrided ? 0 : kl * CPL < K - CPL ? kl * CPL : K - CPL;
  const bool stores = sub == 0 && owns;
  int32_t ks[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) ks[c] = lane + c * kWave < K ? lane + c * kWave : K - 1;
  const auto store_row = [&](TC* row, Out sum, bool stream) {
    if constexpr (kStrided) {
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        if (lane + c * kWave >= K) continue;
        if (stream)
          __builtin_nontemporal_store((TC)sum[c], row + lane + c * kWave);
        else
          row[lane + c * kWave] = sum[c];
      }
    } else if (stores) {
      if (stream)
        __builtin_nontemporal_store(sum, (Out*)(row + k0));
      else
        *(Out*)(row + k0) = sum;
    }
  };
  TC acc[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) acc[c] = 0;
  // The row's sums, added across the lane groups, in group 0.
  const auto row_sum = [&]() {
    if constexpr (!ONE) {
      for (int g = S > 8 ? 8 : S > 4 ? 4 : S > 2 ? 2 : S > 1 ? 1 : 0; g > 0; g >>= 1) {
        const bool have = sub + g < S;
        const int from = have ? lane + g * L : lane;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
          const TC v = __shfl(acc[c], from, kWave);
          acc[c] = have ? acc[c] + v : acc[c];
        }
      }
    }
    Out sum;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      sum[c] = acc[c];
      acc[c] = 0;
    }
    return sum;
  };
  // Ends of the rows first .. first + 63; row m's never comes.
  const auto row_ends = [&](int32_t first) {
    const int64_t q = (int64_t)first + 1 + lane;
    return q <= m ? pos[q] : INT_MAX;
  };
  int at = 0;
  int32_t ends = row_ends(r);
  int32_t rend = __builtin_amdgcn_readlane(ends, 0);
  int32_t zrow = z;  // the team's first entry of row r
  // Entries past nnz > 0 are loaded as the last one and never added.
  const auto entry = [&](int32_t first) {
    const int64_t q = (int64_t)first + lane;
    return q < nnz ? q : nnz - 1;
  };
  int32_t zc = z;
  int32_t jn = stream_load(crd + entry(zc));
  TA an = stream_load(vals + entry(zc));
  while (left > 0) {
    const int32_t jl = jn;
    const TC al = widen(an);
    zc = zc < INT_MAX - kWave ? zc + chunk : zc;
    jn = stream_load(crd + entry(zc));
    an = stream_load(vals + entry(zc));
    for (int e0 = 0; e0 < chunk && left > 0; e0 += S * U) {
      TC a[U], b[U][CPL];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        int32_t j;
        if constexpr (ONE) {
          j = wave_bcast(jl, e0 + u);
          a[u] = wave_bcast(al, e0 + u);
        } else {
          j = __shfl(jl, e0 + u * S + sub, kWave);
          a[u] = __shfl(al, e0 + u * S + sub, kWave);
        }
        if constexpr (kStrided) {
#pragma unroll
          for (int c = 0; c < CPL; ++c) b[u][c] = widen(B[(int64_t)j * K + ks[c]]);
        } else {
          load_wide<CPL>(B + (int64_t)j * K + k0, b[u]);
        }
      }
      if (left >= S * U && rend - z >= S * U) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int c = 0; c < CPL; ++c) acc[c] += a[u] * b[u][c];
        z += S * U;
        left -= S * U;
        continue;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        int done = 0;  // entries of this step already added
        do {
          while (left > 0 && z == rend) {
            // Row end item: row r completes in this team (its earlier
            // entries, if any, arrive through the carries of preceding teams).
            const Out sum = row_sum();
            // non-temporal: C is written once, B rows keep the caches
            store_row(C + (int64_t)r * K, sum, true);
            ++r;
            --left;
            zrow = z;
            if (++at == kWave) {
              at = 0;
              ends = row_ends(r);
            }
            rend = __builtin_amdgcn_readlane(ends, at);
          }
          int take = S - done < rend - z ? S - done : rend - z;
          take = take < left ? take : left;
          // Only the entries' own lanes add: a B row outside may hold
          // infinities or NaN.
          if (ONE ? take > 0 : sub >= done && sub < done + take) {
#pragma unroll
            for (int c = 0; c < CPL; ++c) acc[c] += a[u] * b[u][c];
          }
          z += take;
          left -= take;
          done += take;
        } while (left > 0 && done < S);
      }
    }
  }
  const bool has_carry = z > zrow && r < m;
  if (lane == 0) carry_row[team] = has_carry ? r : -1;
  if (has_carry) {
    const Out sum = row_sum();
    store_row(carry_val + team * K, sum, false);
  }
}

// A wave per carry slot; the first slot of each run of equal rows adds the
// run.  The rows of 63 slots and the first carry load at once, then C's row:
// a wave waits for memory twice, which is what this kernel's time is made
// of.  Runs of up to kFixupOwn slots are added by that wave in team order;
// longer ones (a row of 1e5 entries leaves some 400) are cut into 4
// consecutive pieces, one for each wave of the workgroup, whose sums are
// then added in order: the order is fixed, so results do not change from
// run to run.  Walking run and carries one after another in one wave, the
// longest row of a 1M-row power-law matrix at K = 64, f64, kept this kernel
// busy for 115 us (now 31).
constexpr int kFixupWaves = 4;
constexpr int kFixupOwn = 16;
template <typename TC>
__device__ __forceinline__ TC add_carries(const TC* __restrict__ carry_val, int64_t q, int64_t e,
                                          int32_t K, int32_t k, TC s) {
  for (; q + 16 <= e; q += 16) {
    TC v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = carry_val[(q + u) * K + k];
#pragma unroll
    for (int u = 0; u < 16; ++u) s += v[u];
  }
  for (; q < e; ++q) s += carry_val[q * K + k];
  return s;
}
template <typename TC>
__global__ __launch_bounds__(kFixupWaves * kWave) void k_spmm_merge_fixup(
    int64_t nteams, int32_t K, const int32_t* __restrict__ carry_row,
    const TC* __restrict__ carry_val, TC* __restrict__ C) {
  __shared__ int32_t s_len[kFixupWaves];
  __shared__ TC s_sum[kFixupWaves][kWave];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int lane = threadIdx.x % kWave;
  const int64_t t0 = (int64_t)blockIdx.x * kFixupWaves;
  const int64_t t = t0 + wave;
  // Lane l holds the row of slot t - 1 + l; -2 outside the slots.
  const int64_t q = t - 1 + lane;
  const int32_t row = q >= 0 && q < nteams ? carry_row[q] : -2;
  const TC first = t < nteams && lane < K ? carry_val[t * K + lane] : TC(0);
  const int32_t before = __builtin_amdgcn_readlane(row, 0);
  const int32_t r = __builtin_amdgcn_readlane(row, 1);
  int64_t e = t;  // the run is t .. e - 1
  if (r >= 0 && before != r) {
    uint64_t other = __ballot(row != r) >> 1;  // bit i: slot t + i is of another row
    if (other) {
      e = t + __ffsll((unsigned long long)other) - 1;
    } else {
      for (e = t + kWave - 1;; e += kWave) {
        const int64_t p = e + lane;
        other = __ballot(p >= nteams || carry_row[p < nteams ? p : t] != r);
        if (other) {
          e += __ffsll((unsigned long long)other) - 1;
          break;
        }
      }
    }
    if (e - t <= kFixupOwn)
      for (int32_t k = lane; k < K; k += kWave) {
        const TC s = k == lane ? first : carry_val[t * K + k];
        C[(int64_t)r * K + k] += add_carries(carry_val, t + 1, e, K, k, s);
      }
  }
  // At most INT32_MAX teams.
  if (lane == 0) s_len[wave] = (int32_t)(e - t);
  __syncthreads();
  for (int w = 0; w < kFixupWaves; ++w) {
    const int32_t len = s_len[w];  // the same for the whole workgroup
    if (len <= kFixupOwn) continue;
    const int64_t q0 = t0 + w, q1 = q0 + len;
    const int64_t piece = (len + kFixupWaves - 1) / kFixupWaves;
    const int64_t a = q0 + wave * piece < q1 ? q0 + wave * piece : q1;
    const int64_t b = a + piece < q1 ? a + piece : q1;
    for (int32_t kb = 0; kb < K; kb += kWave) {
      const int32_t k = kb + lane;
      s_sum[wave][lane] = k < K ? add_carries(carry_val, a, b, K, k, TC(0)) : TC(0);
      __syncthreads();
      if (wave == w && k < K) {
        TC s = 0;
        for (int v = 0; v < kFixupWaves; ++v) s += s_sum[v][lane];
        C[(int64_t)r * K + k] += s;
      }
      __syncthreads();
    }
  }
}

// Adjacent columns a lane of the merge kernel owns: 16 bytes of f32 or f64
// (one column below that width), except f64 rows of 33 to 64 columns, which
// take a wave to a B row.  Two columns a lane, two or three B rows to a load,
// are no better throughout (one : two columns, f64): 300,000 power-law rows
// of 16, K = 33 287 : 305 us, 48 298 : 304, 64 392 : 401; 300,000 banded rows
// of 20 231 : 198, 259 : 241, 346 : 339; 100,000 uniform rows of 16 100 : 98,
// 105 : 104, 136 : 138.  Wider f64 rows take strided columns (kStrided:
// 326,797 uniform rows of 30, K = 102: 1272 us against 1307 with adjacent
// ones; 200,000 banded rows, K = 128: 406 against 430).
template <typename TC>
int merge_cols(int32_t K) {
  const int wide = 16 / (int)sizeof(TC);
  if (sizeof(TC) == 8 && K > 32 && K <= 64) return 1;
  return K < wide ? 1 : K <= 64 * wide ? wide : 4;
}

template <typename TA, typename TC>
int run_spmm(const CsrView& a, int32_t K, const TA* B, TC* C,
             const taco_hip_schedule& s) {
  hipStream_t st = current_stream();
  if (a.m == 0 || K == 0) return 0;
  const int algo = s.algo;
  if (algo == TACO_HIP_THREAD_PER_ROW) {
    int bs = s.block_size > 0 ? s.block_size : 256;
    TH_REQUIRE(bs % kWave == 0 && bs <= 1024, "spmm: bad block size %d", bs);
    unsigned grid = (unsigned)((a.m + bs - 1) / bs);
    k_spmm_thread_per_row<TA, TC><<<grid, bs, 0, st>>>(
        a.m, K, a.pos, a.crd, (const TA*)a.vals, B, C);
    return 0;
  }
  // Lane-team shape: G lanes along k, CPL columns per lane.
  int G = s.group_size > 0 ? s.group_size : (K >= 64 ? 64 : 1);
  if (s.group_size <= 0)
    while (G < K && G < 64) G <<= 1;
  TH_REQUIRE(G == 8 || G == 16 || G == 32 || G == 64,
             "spmm: group_size %d must be 8, 16, 32 or 64", G);
  const int cpl = (K + G - 1) / G;
  TH_REQUIRE(cpl <= 4, "spmm: K=%d too wide for %d lanes (max 4 per lane)",
             K, G);
  const int CPL = cpl <= 1 ? 1 : cpl <= 2 ? 2 : 4;
  const int bs = 256;
  const int teams_per_block = bs / G;

#define TH_SHAPES(X)                                                       \
  X(8, 1) X(8, 2) X(8, 4) X(16, 1) X(16, 2) X(16, 4) X(32, 1) X(32, 2)     \
  X(32, 4) X(64, 1) X(64, 2) X(64, 4)

  if (algo == TACO_HIP_GROUP_PER_ROW) {
    int rpg = s.rows_per_group > 0 ? s.rows_per_group : 1;
    int64_t teams = ((int64_t)a.m + rpg - 1) / rpg;
    unsigned grid = (unsigned)((teams + teams_per_block - 1) / teams_per_block);
#define TH_X(g, c)                                                          \
  if (G == g && CPL == c) {                                                 \
    k_spmm_group_per_row<TA, TC, g, c><<<grid, bs, 0, st>>>(                \
        a.m, K, rpg, a.pos, a.crd, (const TA*)a.vals, B, C);                \
    return 0;                                                               \
  }
    TH_SHAPES(TH_X)
#undef TH_X
    return fail("spmm: no kernel for G=%d CPL=%d", G, CPL);
  }
  if (algo == TACO_HIP_NNZ_SPLIT) {
    int npt = s.items_per_thread > 0 ? s.items_per_thread : 8;
    if (int rc = zero_fill(C, sizeof(TC) * (size_t)a.m * K, st)) return rc;
    if (a.nnz == 0) return 0;
    int64_t teams = (a.nnz + npt - 1) / npt;
    unsigned grid = (unsigned)((teams + teams_per_block - 1) / teams_per_block);
#define TH_X(g, c)                                                          \
  if (G == g && CPL == c) {                                                 \
    k_spmm_nnz_split<TA, TC, g, c><<<grid, bs, 0, st>>>(                    \
        a.m, a.nnz, K, npt, a.pos, a.crd, (const TA*)a.vals, B, C,          \
        coarse_grained(C));                                                 \
    return 0;                                                               \
  }
    TH_SHAPES(TH_X)
#undef TH_X
    return fail("spmm: no kernel for G=%d CPL=%d", G, CPL);
  }
  if (algo == TACO_HIP_MERGE_PATH) {
    if (a.nnz == 0) return zero_fill(C, sizeof(TC) * (size_t)a.m * K, st);
    int ipt = s.items_per_thread > 0 ? s.items_per_thread : 256;
    // Below the default a wave takes the items of the 64 / G teams of G lanes
    // that fit in it: its lane groups walk the rows together, and with 16
    // items of K = 4 columns it had little but searches and carries to do
    // (200,000 uniform rows of 16, f64: 219 us, now 71; 32 items 127, now 67;
    // 256 items 67).
    if (ipt < 256) ipt = ipt * (kWave / G) < 256 ? ipt * (kWave / G) : 256;
    const int cols = merge_cols<TC>(K);
    const bool one = (K + cols - 1) / cols > 32;
    const int64_t total = (int64_t)a.m + a.nnz;
    // f64 rows of 17 to 32 columns in fewer waves than are resident (8192):
    // 192 items each, f64, K = 24, 192 against 256: 100,000 uniform rows of
    // 16 67.9 : 76.6 us, 100,000 banded of 20 58.1 : 61.7; in more waves than
    // that, 150,000 uniform rows, 104.6 : 100.9.  (f32 rows of 16 columns
    // 41.7 : 37.5.)
    if (sizeof(TC) == 8 && K > 16 && !one && ipt > 192 && total < (int64_t)ipt * 8192) ipt = 192;
    const int64_t nteams = (total + ipt - 1) / ipt;
    const size_t row_bytes = ((size_t)nteams * sizeof(int32_t) + 255) / 256 * 256;
    void* ws = workspace(row_bytes + (size_t)nteams * K * sizeof(TC), 1);
    if (!ws) return 1;
    int32_t* crow = (int32_t*)ws;
    TC* cval = (TC*)((char*)ws + row_bytes);
    unsigned grid = (unsigned)((nteams * kWave + bs - 1) / bs);
    // Narrow rows: 16 groups of 4 lanes, 4 steps each.
    const int steps = (K + cols - 1) / cols <= 4 ? 4 : 8;
#define TH_MERGE(c, u, o)                                                   \
  if (cols == c && steps == u && one == o)                                  \
    k_spmm_merge<TA, TC, c, u, o><<<grid, bs, 0, st>>>(                     \
        a.m, a.nnz, K, ipt, a.pos, a.crd, (const TA*)a.vals, B, C, nteams,  \
        crow, cval);
    TH_MERGE(1, 4, false) TH_MERGE(1, 8, false) TH_MERGE(1, 8, true)
    TH_MERGE(2, 4, false) TH_MERGE(2, 8, false) TH_MERGE(2, 8, true)
    TH_MERGE(4, 4, false) TH_MERGE(4, 8, false) TH_MERGE(4, 8, true)
#undef TH_MERGE
    TH_LAUNCH_CHECK("k_spmm_merge");
    unsigned g2 = (unsigned)((nteams + kFixupWaves - 1) / kFixupWaves);
    k_spmm_merge_fixup<TC><<<g2, kFixupWaves * kWave, 0, st>>>(nteams, K, crow, cval, C);
    return 0;
  }
#undef TH_SHAPES
  return fail("spmm: schedule algo %d not available here", algo);
}

}  // namespace

int spmm_mfma_bf16(const CsrView& a, int32_t K, const void* B, float* C,
                   const taco_hip_schedule& s);

}  // namespace taco_hip

using namespace taco_hip;

extern "C" int taco_hip_spmm_compute(taco_tensor_t* C, taco_tensor_t* A,
                                     taco_tensor_t* B,
                                     const taco_hip_schedule* sched) {
  CsrView a;
  DenseView bv, cv;
  if (int rc = view_csr(A, "A", &a)) return rc;
  if (int rc = view_dense(B, "B", 2, &bv)) return rc;
  if (int rc = view_dense(C, "C", 2, &cv)) return rc;
  TH_REQUIRE(bv.dims[0] == a.n, "spmm: B has %d rows, A has %d columns",
             bv.dims[0], a.n);
  TH_REQUIRE(cv.dims[0] == a.m && cv.dims[1] == bv.dims[1],
             "spmm: C is %dx%d, expected %dx%d", cv.dims[0], cv.dims[1], a.m,
             bv.dims[1]);
  const int32_t K = bv.dims[1];
  taco_hip_schedule s;
  if (sched)
    s = *sched;
  else
    taco_hip_default_schedule(1, a.m, a.nnz, K, &s);
  int rc;
  if (a.vt == VType::F64 && bv.vt == VType::F64 && cv.vt == VType::F64) {
    TH_REQUIRE(s.algo != TACO_HIP_MFMA, "spmm: MFMA schedule needs bf16 A/B");
    rc = run_spmm<double, double>(a, K, (const double*)bv.vals,
                                  (double*)cv.vals, s);
  } else if (a.vt == VType::F32 && bv.vt == VType::F32 &&
             cv.vt == VType::F32) {
    TH_REQUIRE(s.algo != TACO_HIP_MFMA, "spmm: MFMA schedule needs bf16 A/B");
    rc = run_spmm<float, float>(a, K, (const float*)bv.vals, (float*)cv.vals,
                                s);
  } else if (a.vt == VType::BF16 && bv.vt == VType::BF16 &&
             cv.vt == VType::F32) {
    if (s.algo == TACO_HIP_MFMA)
      rc = spmm_mfma_bf16(a, K, bv.vals, (float*)cv.vals, s);
    else
      rc = run_spmm<bf16_t, float>(a, K, (const bf16_t*)bv.vals,
                                   (float*)cv.vals, s);
  } else {
    return fail("spmm: supported value forms are f64, f32, and bf16 A/B "
                "with f32 C");
  }
  if (rc) return rc;
  return finish("taco_hip_spmm_compute");
}

// Block-sparse (BSR, 3x3 fp32 blocks) assembly of the Newton system: the
// triplet -> BSR conversion the contact Hessian goes through, a value-only
// refill over a kept pattern, and the sum of two BSR matrices
// (warp.sparse.bsr_from_triplets / bsr_axpy at dynamic_contacts.py:290-297,
// affine_body_dynamics.py:500-503, augmented_lagrangian.py:631-632).
//
// Triplet -> BSR in row buckets instead of a global key sort:
//   count    a workgroup takes 1024 triplets: a triplet is dropped (row or
//            column out of range, or all nine values zero) or counted in an
//            LDS table of the workgroup's rows; then one atomic a distinct
//            row takes the workgroup's range of that row's bucket;
//   scan     bucket starts = exclusive scan of the row counts;
//   scatter  (column, triplet) into the row's bucket;
//   sort     one wave per row of up to 512 entries: a bitonic network in
//            registers by (column, triplet); longer rows one workgroup each,
//            merged in LDS (up to 8192 entries) or in place in memory. The
//            row's distinct columns and where their runs start replace the
//            head of its bucket;
//   scan     row offsets = exclusive scan of the distinct counts;
//   pattern  the columns and run starts moved to their place in the matrix;
//   sum      nine lanes a block, one an entry of it, add the block's triplets
//            in ascending order from +0 (all that a refill repeats).
// Every step reads or writes each triplet a bounded number of times; the
// result does not depend on the order the atomics hand out slots.
#include <cstdio>

#include "../../include/ipc_warp_amd.h"
#include "cull.hpp"
#include "ipc_kernels.hpp"
#include "scan.hpp"

using namespace ipcd;

struct ipc_bsr {
  DevBuf cnt;      // int [n_rows + 1]: per-row kept triplets, then distinct columns
  DevBuf start;    // int [n_rows + 1]: bucket start of each row
  DevBuf slot;     // int [n_triplets]: slot in the row's bucket (-1 if dropped); once sorted, the kept
                   // triplets by row, then column, then triplet
  DevBuf bucket;   // u64 [n_triplets]: column << 32 | triplet, by row; once sorted, each row's
                   // column << 32 | first sorted entry, per distinct column
  DevBuf big;      // int [1 + big_cap]: count of the rows longer than kWaveRow, and which
  DevBuf seg;      // int [capacity + 1]: first sorted entry of each block
  DevBuf part;     // scan partial sums
  DevBuf nnz;      // int [1]: blocks of the kept pattern
  int* host = nullptr;  // pinned readback of the block count
  int n_rows = 0, n_triplets = 0, max_blocks = 0;
  bool planned = false;
};

namespace {

constexpr int kB = 256;
constexpr int kWaves = kB / 64;
constexpr int kWaveRow = 512;   // entries of a row that one wave sorts in registers

int bsr_fail(int code, const char* what) {
  set_error(what);
  return code;
}

int bsr_hip(hipError_t e, const char* where) {
  if (e == hipSuccess) return IPC_OK;
  char buf[512];
  std::snprintf(buf, sizeof(buf), "%s: %s", where, hipGetErrorString(e));
  set_error(buf);
  return -int(e);
}

inline int nblk(long long n, int per) { return int((n + per - 1) / per); }

// ---------------------------------------------------- triplets -> BSR ---
__device__ inline bool block_nonzero(const float* v) {
  bool nz = false;
#pragma unroll
  for (int k = 0; k < 9; ++k) nz |= !(v[k] == 0.0f);  // NaN counts as nonzero
  return nz;
}

// A workgroup's rows in LDS: open addressing, at most one row a triplet.
constexpr int kCountPer = 4;
constexpr int kCountTile = kB * kCountPer;
constexpr int kTable = 2 * kCountTile;

__global__ __launch_bounds__(kB) void bsr_clear_kernel(int* cnt, int n, int* big) {
  for (int i = blockIdx.x * kB + threadIdx.x; i < n; i += gridDim.x * kB) cnt[i] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) big[0] = 0;
}

// Counts each row's kept triplets and gives each a slot in its row's bucket.
// Neighbouring lanes of one row take consecutive slots together (the contact
// Hessian writes the four blocks of a pair's block row next to each other),
// and the workgroup's lanes of one row share one device atomic: those run at
// some 25 G/s, and one for each run of lanes (3.4 million on the rod twist's
// 14.6 million triplets; 0.36 million now) took longer than reading the
// values (280 us, 146 us now).
__global__ __launch_bounds__(kB) void bsr_count_kernel(const int* __restrict__ rows, const int* __restrict__ cols,
                                                       const float* __restrict__ vals, int m, int nr, int nc, int* cnt,
                                                       int* __restrict__ slot) {
  __shared__ int key[kTable], num[kTable];
  for (int i = threadIdx.x; i < kTable; i += kB) {
    key[i] = -1;
    num[i] = 0;
  }
  const int lane = threadIdx.x & 63;
  const long long t0 = (long long)blockIdx.x * kCountTile + threadIdx.x;
  int row[kCountPer], at[kCountPer], pos[kCountPer];
#pragma unroll
  for (int k = 0; k < kCountPer; ++k) {
    const long long t = t0 + k * kB;
    row[k] = -1;
    if (t < m) {
      float v[9];
      __builtin_memcpy(v, vals + 9 * t, sizeof(v));
      const int r = rows[t], c = cols[t];
      if (unsigned(r) < unsigned(nr) && unsigned(c) < unsigned(nc) && block_nonzero(v)) row[k] = r;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kCountPer; ++k) {
    const bool keep = row[k] >= 0;
    const int prev = __shfl_up(row[k], 1);
    const bool head = keep && (lane == 0 || prev != row[k]);
    const unsigned long long hm = __ballot(head), km = __ballot(keep);
    // this lane's run starts at the last head at or below it and ends before
    // the next head or dropped lane
    const unsigned long long upto = lane == 63 ? ~0ull : (2ull << lane) - 1;
    const int h = keep ? 63 - __clzll(hm & upto) : lane;
    const unsigned long long brk = (hm | ~km) & ~((h == 63 ? ~0ull : (2ull << h) - 1));
    const int end = brk ? __ffsll(static_cast<long long>(brk)) - 1 : 64;
    int e = 0, p = 0;
    if (head) {
      e = int((unsigned(row[k]) * 2654435761u) >> 21) & (kTable - 1);
      for (;;) {
        const int was = atomicCAS(key + e, -1, row[k]);
        if (was == -1 || was == row[k]) break;
        e = (e + 1) & (kTable - 1);
      }
      p = atomicAdd(num + e, end - h);
    }
    at[k] = __shfl(e, h);
    pos[k] = __shfl(p, h) + (lane - h);
  }
  __syncthreads();
#pragma unroll
  for (int i = threadIdx.x; i < kTable; i += kB)
    if (key[i] >= 0) num[i] = atomicAdd(cnt + key[i], num[i]);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kCountPer; ++k) {
    const long long t = t0 + k * kB;
    if (t < m) slot[t] = row[k] >= 0 ? num[at[k]] + pos[k] : -1;
  }
}
static_assert(kTable == 2048, "the hash takes 11 bits");

__global__ void bsr_scatter_kernel(const int* rows, const int* cols, const int* slot, const int* start, int m,
                                   unsigned long long* bucket) {
  const int t = blockIdx.x * kB + threadIdx.x;
  if (t >= m) return;
  const int s = slot[t];
  if (s >= 0) bucket[start[rows[t]] + s] = (static_cast<unsigned long long>(unsigned(cols[t])) << 32) | unsigned(t);
}

__device__ inline int key_col(unsigned long long k) { return int(k >> 32); }
__device__ inline int key_triplet(unsigned long long k) { return int(unsigned(k)); }

// v of lane ^ X.
template <int X>
__device__ __forceinline__ unsigned lane_xor(unsigned v) {
  const int i = int(v);
  if (X == 1) return unsigned(__builtin_amdgcn_mov_dpp(i, 0xB1, 0xf, 0xf, true));   // quad_perm 1 0 3 2
  if (X == 2) return unsigned(__builtin_amdgcn_mov_dpp(i, 0x4E, 0xf, 0xf, true));   // quad_perm 2 3 0 1
  if (X == 3) return unsigned(__builtin_amdgcn_mov_dpp(i, 0x1B, 0xf, 0xf, true));   // quad_perm 3 2 1 0
  if (X == 4) return lane_xor<3>(lane_xor<7>(v));
  if (X == 7) return unsigned(__builtin_amdgcn_mov_dpp(i, 0x141, 0xf, 0xf, true));  // row_half_mirror
  if (X == 8) return unsigned(__builtin_amdgcn_mov_dpp(i, 0x128, 0xf, 0xf, true));  // row_ror:8
  if (X == 15) return unsigned(__builtin_amdgcn_mov_dpp(i, 0x140, 0xf, 0xf, true)); // row_mirror
  if (X == 16) return unsigned(__builtin_amdgcn_ds_swizzle(i, 0x401f));             // xor 16 within 32 lanes
  if (X == 31) return lane_xor<15>(lane_xor<16>(v));
  return unsigned(__shfl_xor(i, X, 64));
}

// One cross-lane compare step: lane l against lane l ^ X; the lane without
// the mask's top bit keeps the smaller key. REV: the partner's register
// K - 1 - k instead of k.
template <int K, int X, bool REV>
__device__ __forceinline__ void cross_step(unsigned long long (&key)[K], int lane) {
  constexpr int kTop = X >= 32 ? 32 : X >= 16 ? 16 : X >= 8 ? 8 : X >= 4 ? 4 : X >= 2 ? 2 : 1;
  const bool low = (lane & kTop) == 0;
  unsigned long long other[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const unsigned long long v = key[REV ? K - 1 - k : k];
    other[k] = (static_cast<unsigned long long>(lane_xor<X>(unsigned(v >> 32))) << 32) | lane_xor<X>(unsigned(v));
  }
#pragma unroll
  for (int k = 0; k < K; ++k) key[k] = (other[k] < key[k]) == low ? other[k] : key[k];
}

// One in-lane compare step of distance J (or mirrored within 2 J).
template <int K, int J, bool REV>
__device__ __forceinline__ void lane_step(unsigned long long (&key)[K]) {
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int o = REV ? k ^ (2 * J - 1) : k ^ J;
    if (o <= k) continue;
    const unsigned long long a = key[k], b = key[o];
    const bool sw = b < a;
    key[k] = sw ? b : a;
    key[o] = sw ? a : b;
  }
}

template <int K, int J>
__device__ __forceinline__ void half_steps(unsigned long long (&key)[K], int lane) {
  if constexpr (J >= K) cross_step<K, J / K, false>(key, lane);
  else lane_step<K, J, false>(key);
  if constexpr (J > 1) half_steps<K, J / 2>(key, lane);
}

template <int K, int S>
__device__ __forceinline__ void sort_size(unsigned long long (&key)[K], int lane) {
  if constexpr (S > K) cross_step<K, S / K - 1, true>(key, lane);
  else lane_step<K, S / 2, true>(key);
  if constexpr (S > 2) half_steps<K, S / 4>(key, lane);
  if constexpr (S < 64 * K) sort_size<K, 2 * S>(key, lane);
}

// The wave's 64 K distinct keys, entry lane K + k in key[k], sorted: a
// bitonic network whose merges start mirrored, so that every step puts the
// smaller key first. K = 4 takes some 700 instructions; ranking each key
// against every other took ten times as many at a row's usual 150 entries.
template <int K>
__device__ __forceinline__ void wave_sort(unsigned long long (&key)[K], int lane) {
  sort_size<K, 2>(key, lane);
}

// A row of at most 64 K entries: sorted, its triplets to tri, its distinct
// columns with their first entries to the head of its bucket. Returns their
// number.
template <int K>
__device__ __forceinline__ int sort_row(unsigned long long* bucket, int* tri, int b, int L, int lane) {
  unsigned long long key[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = K * lane + k;
    key[k] = i < L ? bucket[b + i] : ~0ull;
  }
  wave_sort<K>(key, lane);
  const int last = __shfl_up(key_col(key[K - 1]), 1, 64);
  int before = 0;  // heads of the lanes below
  bool head[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = K * lane + k;
    const int prev = k > 0 ? key_col(key[k > 0 ? k - 1 : 0]) : last;
    head[k] = i < L && (i == 0 || key_col(key[k]) != prev);
    if (i < L) tri[b + i] = key_triplet(key[k]);
  }
  int total = 0;
  const unsigned long long below = (1ull << lane) - 1;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const unsigned long long m = __ballot(head[k]);
    before += __popcll(m & below);
    total += __popcll(m);
  }
#pragma unroll
  for (int k = 0; k < K; ++k)
    if (head[k]) bucket[b + before++] = (key[k] & ~0xffffffffull) | unsigned(b + K * lane + k);
  return total;
}

// One wave per row. Rows longer than kWaveRow are listed for
// bsr_sort_long_kernel, where a workgroup and 64 KB of LDS take one row: with
// rows of 257 to 512 entries there, a build of 15,563 rows of 257 took 407 us
// (119 so; 284 with the keys ranked against a row staged in LDS).
__global__ __launch_bounds__(kB) void bsr_sort_rows_kernel(const int* __restrict__ start, int nr,
                                                           unsigned long long* bucket, int* tri, int* rnnz, int* big) {
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int r = blockIdx.x * kWaves + w; r < nr; r += gridDim.x * kWaves) {
    const int b = start[r], L = start[r + 1] - b;
    int heads = 0;
    if (L == 0) {
    } else if (L <= 64) {
      heads = sort_row<1>(bucket, tri, b, L, lane);
    } else if (L <= 128) {
      heads = sort_row<2>(bucket, tri, b, L, lane);
    } else if (L <= 256) {
      heads = sort_row<4>(bucket, tri, b, L, lane);
    } else if (L <= kWaveRow) {
      heads = sort_row<8>(bucket, tri, b, L, lane);
    } else {
      if (lane == 0) big[1 + atomicAdd(big, 1)] = r;  // at most n_triplets / (kWaveRow + 1) rows
      continue;
    }
    if (lane == 0) rnnz[r] = heads;
  }
}

// ---- long rows: a workgroup each
constexpr int kLongB = 512;
constexpr int kLongWaves = kLongB / 64;
constexpr int kLongLds = 8192;              // entries sorted in LDS
constexpr int kLongPer = kLongLds / kLongB;
constexpr int kLongGrid = 512;

// n <= kLongLds keys of src sorted into the workgroup's LDS: 256 at a time
// by a wave in registers, then merges in which each key finds its place by a
// binary search of the neighbouring run.
__device__ void lds_sort(unsigned long long* s, const unsigned long long* src, int n) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int c = 256 * w; c < n; c += 256 * kLongWaves) {
    unsigned long long key[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = c + 4 * lane + k;
      key[k] = i < n ? src[i] : ~0ull;
    }
    wave_sort<4>(key, lane);
#pragma unroll
    for (int k = 0; k < 4; ++k) s[c + 4 * lane + k] = key[k];
  }
  __syncthreads();
  for (int run = 256; run < n; run *= 2) {
    unsigned long long key[kLongPer];
    int to[kLongPer];
#pragma unroll
    for (int k = 0; k < kLongPer; ++k) {
      const int i = threadIdx.x + k * kLongB;
      to[k] = -1;
      if (i >= n) continue;
      key[k] = s[i];
      const int mine = i / run * run, pair = i / (2 * run) * (2 * run);
      const int sib = mine == pair ? pair + run : pair;
      int lo = sib < n ? sib : n, hi = sib + run < n ? sib + run : n;
      const int from = lo;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        const bool less = s[mid] < key[k];
        lo = less ? mid + 1 : lo;
        hi = less ? hi : mid;
      }
      to[k] = pair + (i - mine) + (lo - from);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kLongPer; ++k)
      if (to[k] >= 0) s[to[k]] = key[k];
    __syncthreads();
  }
}

// The order of a row longer than kLongLds, in place in memory: chunks of
// kLongLds sorted in LDS, then bitonic merges (mirrored first, so that every
// step puts the smaller key first and the entries missing past L need no
// padding), whose steps below a chunk's length run in LDS.
__device__ void memory_sort(unsigned long long* s, unsigned long long* key, int L) {
  for (int c = 0; c < L; c += kLongLds) {
    const int n = L - c < kLongLds ? L - c : kLongLds;
    lds_sort(s, key + c, n);
    for (int i = threadIdx.x; i < n; i += kLongB) key[c + i] = s[i];
    __syncthreads();
  }
  for (long long size = 2ll * kLongLds; size < 2ll * L; size *= 2) {
    for (long long j = size / 2; j >= kLongLds; j /= 2) {
      const bool mirror = j == size / 2;
      for (int i = threadIdx.x; i < L; i += kLongB) {
        if (i & j) continue;  // the lower of each pair
        const long long o = mirror ? (i ^ (size - 1)) : (i ^ j);
        if (o >= L) continue;
        const unsigned long long a = key[i], b = key[o];
        if (b < a) {
          key[i] = b;
          key[o] = a;
        }
      }
      __syncthreads();
    }
    for (int c = 0; c < L; c += kLongLds) {
      const int n = L - c < kLongLds ? L - c : kLongLds;
      for (int i = threadIdx.x; i < n; i += kLongB) s[i] = key[c + i];
      __syncthreads();
      for (int j = kLongLds / 2; j > 0; j /= 2) {
        for (int i = threadIdx.x; i < n; i += kLongB) {
          const int o = i ^ j;
          if (o < i || o >= n) continue;
          const unsigned long long a = s[i], b = s[o];
          if (b < a) {
            s[i] = b;
            s[o] = a;
          }
        }
        __syncthreads();
      }
      for (int i = threadIdx.x; i < n; i += kLongB) key[c + i] = s[i];
      __syncthreads();
    }
  }
}

__global__ __launch_bounds__(kLongB) void bsr_sort_long_kernel(const int* __restrict__ start, const int* big,
                                                               unsigned long long* bucket, int* tri, int* rnnz) {
  __shared__ unsigned long long s[kLongLds];
  __shared__ int wsum[kLongWaves];
  __shared__ int edge;  // the last column of the tile before
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int rows = big[0];
  for (int q = blockIdx.x; q < rows; q += gridDim.x) {
    const int r = big[1 + q], b = start[r], L = start[r + 1] - b;
    unsigned long long* key = bucket + b;
    const bool in_lds = L <= kLongLds;
    if (in_lds) lds_sort(s, key, L);
    else memory_sort(s, key, L);
    // heads in order; in memory they overwrite entries already read
    int heads = 0;
    for (int t = 0; t < L; t += kLongB) {
      const int i = t + threadIdx.x;
      const unsigned long long k = i < L ? (in_lds ? s[i] : key[i]) : ~0ull;
      const int c = key_col(k);
      int prev = __shfl_up(c, 1, 64);
      if (lane == 0 && i > 0 && i < L && threadIdx.x > 0) prev = key_col(in_lds ? s[i - 1] : key[i - 1]);
      if (threadIdx.x == 0 && t > 0) prev = edge;
      const bool head = i < L && (i == 0 || c != prev);
      const unsigned long long m = __ballot(head);
      if (lane == 0) wsum[w] = __popcll(m);
      __syncthreads();  // the tile has been read
      if (threadIdx.x == kLongB - 1) edge = c;
      int at = heads, sum = 0;
#pragma unroll
      for (int u = 0; u < kLongWaves; ++u) {
        at += u < w ? wsum[u] : 0;
        sum += wsum[u];
      }
      if (i < L) tri[b + i] = key_triplet(k);
      if (head) key[at + __popcll(m & ((1ull << lane) - 1))] = (k & ~0xffffffffull) | unsigned(b + i);
      heads += sum;
      __syncthreads();
    }
    if (threadIdx.x == 0) rnnz[r] = heads;
  }
}

// Sixteen lanes a row move its columns and run starts to their place; the
// last row also closes the run list.
constexpr int kPatternLanes = 16;
constexpr int kPatternRows = kB / kPatternLanes;
__global__ __launch_bounds__(kB) void bsr_pattern_kernel(const int* __restrict__ start,
                                                         const int* __restrict__ offsets, int nr,
                                                         const unsigned long long* __restrict__ bucket, int cap,
                                                         int* __restrict__ columns, int* __restrict__ seg,
                                                         int* nnz_out) {
  const int total = offsets[nr];
  if (blockIdx.x == 0 && threadIdx.x == 0) *nnz_out = total <= cap ? total : -1;
  if (total > cap) return;
  const int r = blockIdx.x * kPatternRows + threadIdx.x / kPatternLanes;
  if (r >= nr) return;
  const int b = start[r], o = offsets[r], n = offsets[r + 1] - o;
  for (int i = threadIdx.x % kPatternLanes; i < n; i += kPatternLanes) {
    const unsigned long long u = bucket[b + i];
    columns[o + i] = key_col(u);
    seg[o + i] = int(unsigned(u));
  }
  if (r == nr - 1 && threadIdx.x % kPatternLanes == 0) seg[total] = start[nr];
}

// Block values, a block's triplets added in ascending order from +0. Two ways,
// by the mean length of the runs (read on the device):
//   short  a wave takes 64 consecutive blocks, gathers their triplets' values
//          into LDS a window at a time and adds a block a lane;
//   long   nine lanes a block, one for each value, seven blocks a wave: a
//          block's next nine triplets are read by its lanes together, then
//          their values nine loads at a time.
// With one lane a block 64 lanes wait for the longest of 64 runs (4 million
// triplets, 16 a block: 49 us, 30 with nine); nine lanes a block take ten times
// the instructions for a run of one (4 million: 142 us, 69 with one lane), and
// lose at a mean run of 5.1 still (a tet mesh's 1.44 million blocks: 105 us,
// 90). At eight they are ahead (34 and 32 us). Below 2^17 blocks the waves of
// 64 are too few. (Nine lanes walking nine blocks as one range, so that none
// waits for a longer one, took 189 us where nine a block take 130: the block
// ends cost more than the waiting.)
constexpr int kSumBlocks = 7;
constexpr int kSumWin = 128;          // entries of a window
constexpr int kSumShort = 6;          // mean run from which nine lanes take a block
constexpr int kSumFew = 1 << 17;

__device__ __forceinline__ void sum_lane_a_block(int n, const int* __restrict__ seg, const int* __restrict__ tri,
                                                 const float* __restrict__ vals, float* __restrict__ values, float* s) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (long long o0 = (long long)(blockIdx.x * kWaves + w) * 64; o0 < n; o0 += (long long)gridDim.x * kWaves * 64) {
    const long long o = o0 + lane;
    const bool active = o < n;
    const int mb = active ? seg[o] : 0, me = active ? seg[o + 1] : 0;
    const int e0 = seg[o0], e1 = seg[o0 + 64 < n ? o0 + 64 : n];
    float acc[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int w0 = e0; w0 < e1; w0 += kSumWin) {
      const int cnt = e1 - w0 < kSumWin ? e1 - w0 : kSumWin;
      for (int k = lane; k < cnt; k += 64) {
        float v[9];
        __builtin_memcpy(v, vals + 9ll * tri[w0 + k], sizeof(v));
#pragma unroll
        for (int j = 0; j < 9; ++j) s[k * 9 + j] = v[j];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      const int lo = mb > w0 ? mb : w0, hi = me < w0 + cnt ? me : w0 + cnt;
      for (int q = lo; q < hi; ++q) {
#pragma unroll
        for (int j = 0; j < 9; ++j) acc[j] += s[(q - w0) * 9 + j];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (active) __builtin_memcpy(values + 9 * o, acc, sizeof(acc));
  }
}

// kept_p: the kept triplets, seg[*nnz_p] too, but read beside the block count
// instead of after it; so are the first run ends, below the most blocks there
// can be (seg holds max_blocks + 1).
__global__ __launch_bounds__(kB) void bsr_sum_kernel(const int* nnz_p, const int* kept_p, int max_blocks,
                                                     const int* __restrict__ seg,
                                                     const int* __restrict__ tri, const float* __restrict__ vals,
                                                     float* __restrict__ values) {
  __shared__ float window[kWaves][kSumWin * 9];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = lane / 9, e = lane - 9 * g;
  long long o = (long long)(blockIdx.x * kWaves + w) * kSumBlocks + g;
  int q = 0, end = 0;
  if (o < max_blocks) {
    q = seg[o];
    end = seg[o + 1];
  }
  const int n = *nnz_p, kept = *kept_p;
  if (n >= kSumFew && kept < (long long)kSumShort * n) {
    sum_lane_a_block(n, seg, tri, vals, values, window[w]);
    return;
  }
  if (g == kSumBlocks) return;  // the wave's last lane
  while (o < n) {
    float acc = 0.0f;
    int t = q + e < end ? tri[q + e] : 0;
    while (q < end) {
      const int left = end - q;
      const int next = q + 9 + e < end ? tri[q + 9 + e] : 0;
      float v[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) {
        const long long at = __shfl(t, 9 * g + k, 64);
        v[k] = k < left ? vals[9 * at + e] : 0.0f;
      }
#pragma unroll
      for (int k = 0; k < 9; ++k) acc = k < left ? acc + v[k] : acc;
      t = next;
      q += 9;
    }
    values[9 * o + e] = acc;
    o += (long long)gridDim.x * kWaves * kSumBlocks;
    if (o < n) {
      q = seg[o];
      end = seg[o + 1];
    }
  }
}

hipError_t launch_sum(const ipc_bsr* w, int n_rows, int max_blocks, const float* vals, float* values, hipStream_t s) {
  const int need = nblk(max_blocks, kWaves * kSumBlocks);
  const int g = need < 1 ? 1 : (need < 8192 ? need : 8192);  // strides over the blocks there are
  hipLaunchKernelGGL(bsr_sum_kernel, dim3(g), dim3(kB), 0, s, w->nnz.as<int>(), w->start.as<int>() + n_rows,
                     max_blocks, w->seg.as<int>(), w->slot.as<int>(), vals, values);
  return hipGetLastError();
}

// ------------------------------------------------------------ axpy ---
// Row r of z = alpha x + beta y over the union of the two rows' columns
// (both sorted and distinct per row); a block missing from one side counts
// as zero there.
__global__ void bsr_union_count_kernel(int nr, const int* xo, const int* xc, const int* yo, const int* yc, int* cnt) {
  const int r = blockIdx.x * kB + threadIdx.x;
  if (r > nr) return;
  if (r == nr) {
    cnt[r] = 0;
    return;
  }
  int i = xo[r], j = yo[r];
  const int ie = xo[r + 1], je = yo[r + 1];
  int n = 0;
  while (i < ie && j < je) {
    const int a = xc[i], c = yc[j];
    ++n;
    i += a <= c;
    j += c <= a;
  }
  cnt[r] = n + (ie - i) + (je - j);
}

// Eight lanes per row: the group's first lane merges the two column lists,
// up to kUnionChunk union entries at a time, into LDS (source block of each
// side or -1, column); then the group writes those entries' columns and
// values with consecutive lanes on consecutive floats, so that a row's
// output is written as one contiguous stream. (One lane per row writing its
// own blocks 36 bytes at a time left partial cache lines across the wave:
// the fill moved ten times its algorithmic bytes.)
constexpr int kRowGroup = 8;
constexpr int kUnionChunk = 64;
constexpr int kGroups = kB / kRowGroup;

__global__ __launch_bounds__(kB) void bsr_union_fill_kernel(int nr, const int* xo, const int* xc, const float* xv,
                                                            float alpha, const int* yo, const int* yc, const float* yv,
                                                            float beta, const int* zo, int* zc, float* zv, int cap,
                                                            int* nnz_out) {
  __shared__ int sx[kGroups][kUnionChunk], sy[kGroups][kUnionChunk], sc[kGroups][kUnionChunk];
  const int total = zo[nr];
  if (blockIdx.x == 0 && threadIdx.x == 0 && nnz_out) *nnz_out = total;
  if (total > cap) return;
  const int g = threadIdx.x / kRowGroup, l = threadIdx.x % kRowGroup;
  const int r = blockIdx.x * kGroups + g;
  if (r >= nr) return;  // the whole group
  const int leader = (threadIdx.x & 63) & ~(kRowGroup - 1);
  int i = xo[r], j = yo[r], o = zo[r];
  const int ie = xo[r + 1], je = yo[r + 1];
  for (;;) {
    int m = 0;
    if (l == 0) {
      while (m < kUnionChunk && (i < ie || j < je)) {
        const int a = i < ie ? xc[i] : 0x7fffffff, c = j < je ? yc[j] : 0x7fffffff;
        const bool tx = a <= c, ty = c <= a;
        sx[g][m] = tx ? i : -1;
        sy[g][m] = ty ? j : -1;
        sc[g][m] = tx ? a : c;
        ++m;
        i += tx;
        j += ty;
      }
    }
    m = __shfl(m, leader, 64);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int k = l; k < m; k += kRowGroup) zc[o + k] = sc[g][k];
    for (int f = l; f < 9 * m; f += kRowGroup) {
      const int k = f / 9, e = f - 9 * k;
      const int ix = sx[g][k], iy = sy[g][k];
      const float xs = ix >= 0 ? xv[9ll * ix + e] : 0.0f;
      const float ys = iy >= 0 ? yv[9ll * iy + e] : 0.0f;
      zv[9ll * o + f] = alpha * xs + beta * ys;
    }
    o += m;
    const int more = __shfl(int(i < ie || j < je), leader, 64);
    if (!more) break;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the entries are read before the next chunk
  }
}

}  // namespace

// ============================================================== C ABI ===
extern "C" {

int ipc_bsr_create(ipc_bsr** out) {
  if (!out) return bsr_fail(IPC_EINVAL, "bsr_create: null output");
  ipc_bsr* w = new (std::nothrow) ipc_bsr();
  if (!w) return bsr_fail(IPC_EINVAL, "bsr_create: out of host memory");
  hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&w->host), sizeof(int));
  if (e != hipSuccess) {
    delete w;
    return bsr_hip(e, "bsr_create");
  }
  *out = w;
  return IPC_OK;
}

int ipc_bsr_destroy(ipc_bsr* w) {
  if (!w) return IPC_OK;
  for (DevBuf* d : {&w->cnt, &w->start, &w->slot, &w->bucket, &w->seg, &w->part, &w->nnz, &w->big})
    d->release();
  if (w->host) hipHostFree(w->host);
  delete w;
  return IPC_OK;
}

int ipc_bsr_from_triplets(ipc_bsr* w, int n_rows, int n_cols, const int* rows, const int* cols, const float* vals,
                          int n_triplets, int* offsets, int* columns, float* values, int capacity, void* stream) {
  if (!w) return bsr_fail(IPC_EINVAL, "bsr_from_triplets: null workspace");
  if (n_rows < 0 || n_cols < 0 || n_triplets < 0 || capacity < 0)
    return bsr_fail(IPC_EINVAL, "bsr_from_triplets: negative size");
  if (!offsets) return bsr_fail(IPC_EINVAL, "bsr_from_triplets: null offsets");
  if (n_triplets > 0 && (!rows || !cols || !vals)) return bsr_fail(IPC_EINVAL, "bsr_from_triplets: null triplets");
  if (capacity > 0 && (!columns || !values)) return bsr_fail(IPC_EINVAL, "bsr_from_triplets: null columns/values");
  hipStream_t s = static_cast<hipStream_t>(stream);
  w->planned = false;
  const int m = n_triplets, nr = n_rows;
  hipError_t e = hipSuccess;
  for (DevBuf* d : {&w->cnt, &w->start}) {
    if (e == hipSuccess) e = d->ensure(sizeof(int) * (size_t(nr) + 1));
  }
  if (e == hipSuccess) e = w->slot.ensure(sizeof(int) * size_t(m > 0 ? m : 1));
  if (e == hipSuccess) e = w->bucket.ensure(sizeof(unsigned long long) * size_t(m > 0 ? m : 1));
  const int big_cap = m / (kWaveRow + 1);
  if (e == hipSuccess) e = w->big.ensure(sizeof(int) * (size_t(big_cap) + 1));
  if (e == hipSuccess) e = w->seg.ensure(sizeof(int) * (size_t(capacity) + 1));
  if (e == hipSuccess) e = w->nnz.ensure(sizeof(int));
  if (e != hipSuccess) return bsr_hip(e, "bsr_from_triplets: workspace");
  int* cnt = w->cnt.as<int>();
  int* start = w->start.as<int>();
  int* big = w->big.as<int>();
  int* tri = w->slot.as<int>();
  unsigned long long* bucket = w->bucket.as<unsigned long long>();
  const int cg = nblk((long long)nr + 1, kB);
  hipLaunchKernelGGL(bsr_clear_kernel, dim3(cg < 1024 ? cg : 1024), dim3(kB), 0, s, cnt, nr + 1, big);
  if (m > 0)
    hipLaunchKernelGGL(bsr_count_kernel, dim3(nblk(m, kCountTile)), dim3(kB), 0, s, rows, cols, vals, m, nr, n_cols,
                       cnt, w->slot.as<int>());
  e = hipGetLastError();
  if (e == hipSuccess) e = exclusive_scan(cnt, nr + 1, start, w->part, s);
  if (e == hipSuccess && m > 0)
    hipLaunchKernelGGL(bsr_scatter_kernel, dim3(nblk(m, kB)), dim3(kB), 0, s, rows, cols, w->slot.as<int>(), start, m,
                       bucket);
  if (e == hipSuccess) e = hipGetLastError();
  if (e == hipSuccess && nr > 0) {
    // cnt[nr] stays 0: the rows' distinct counts go to cnt[0..nr)
    const int rg = nblk(nr, kWaves) < 65536 ? nblk(nr, kWaves) : 65536;
    hipLaunchKernelGGL(bsr_sort_rows_kernel, dim3(rg), dim3(kB), 0, s, start, nr, bucket, tri, cnt, big);
    if (big_cap > 0)
      hipLaunchKernelGGL(bsr_sort_long_kernel, dim3(big_cap < kLongGrid ? big_cap : kLongGrid), dim3(kLongB), 0, s,
                         start, big, bucket, tri, cnt);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = exclusive_scan(cnt, nr + 1, offsets, w->part, s);
  if (e == hipSuccess) {
    if (nr > 0) {
      hipLaunchKernelGGL(bsr_pattern_kernel, dim3(nblk(nr, kPatternRows)), dim3(kB), 0, s, start, offsets, nr, bucket,
                         capacity, columns, w->seg.as<int>(), w->nnz.as<int>());
      e = hipGetLastError();
      if (e == hipSuccess && m > 0) e = launch_sum(w, nr, capacity < m ? capacity : m, vals, values, s);
    } else {
      e = fill_i32(w->nnz.as<int>(), 1, 0, s);
      if (e == hipSuccess) e = fill_i32(w->seg.as<int>(), 1, 0, s);
    }
  }
  if (e == hipSuccess) e = hipGetLastError();
  if (e != hipSuccess) return bsr_hip(e, "bsr_from_triplets");
  w->n_rows = nr;
  w->n_triplets = m;
  w->max_blocks = capacity < m ? capacity : m;
  if (capacity >= m) {
    w->planned = true;
    return IPC_OK;
  }
  // the pattern may not fit: read the block count back
  e = hipMemcpyAsync(w->host, offsets + nr, sizeof(int), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return bsr_hip(e, "bsr_from_triplets: block count readback");
  if (*w->host > capacity) return *w->host;
  w->planned = true;
  return IPC_OK;
}

int ipc_bsr_refill(ipc_bsr* w, const float* vals, int n_triplets, float* values, void* stream) {
  if (!w) return bsr_fail(IPC_EINVAL, "bsr_refill: null workspace");
  if (!w->planned) return bsr_fail(IPC_EINVAL, "bsr_refill: no pattern (ipc_bsr_from_triplets has not succeeded)");
  if (n_triplets != w->n_triplets) return bsr_fail(IPC_EINVAL, "bsr_refill: triplet count differs from the pattern's");
  if (n_triplets == 0) return IPC_OK;
  if (!vals || !values) return bsr_fail(IPC_EINVAL, "bsr_refill: null pointer");
  hipError_t e = launch_sum(w, w->n_rows, w->max_blocks, vals, values, static_cast<hipStream_t>(stream));
  return bsr_hip(e, "bsr_refill");
}

int ipc_bsr_axpy(ipc_bsr* w, int n_rows, const int* x_offsets, const int* x_columns, const float* x_values, int x_nnz,
                 float alpha, const int* y_offsets, const int* y_columns, const float* y_values, int y_nnz, float beta,
                 int* z_offsets, int* z_columns, float* z_values, int capacity, void* stream) {
  if (!w) return bsr_fail(IPC_EINVAL, "bsr_axpy: null workspace");
  if (n_rows < 0 || x_nnz < 0 || y_nnz < 0 || capacity < 0) return bsr_fail(IPC_EINVAL, "bsr_axpy: negative size");
  if (!x_offsets || !y_offsets || !z_offsets) return bsr_fail(IPC_EINVAL, "bsr_axpy: null offsets");
  if ((x_nnz > 0 && (!x_columns || !x_values)) || (y_nnz > 0 && (!y_columns || !y_values)) ||
      (capacity > 0 && (!z_columns || !z_values)))
    return bsr_fail(IPC_EINVAL, "bsr_axpy: null columns/values");
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipError_t e = w->cnt.ensure(sizeof(int) * (size_t(n_rows) + 1));
  if (e != hipSuccess) return bsr_hip(e, "bsr_axpy: workspace");
  // the row counts share the triplet path's count buffer; a kept pattern
  // (sorted entries, runs, block count) stays valid
  int* cnt = w->cnt.as<int>();
  hipLaunchKernelGGL(bsr_union_count_kernel, dim3(nblk(n_rows + 1, kB)), dim3(kB), 0, s, n_rows, x_offsets, x_columns,
                     y_offsets, y_columns, cnt);
  e = hipGetLastError();
  if (e == hipSuccess) e = exclusive_scan(cnt, n_rows + 1, z_offsets, w->part, s);
  if (e == hipSuccess && n_rows > 0)
    hipLaunchKernelGGL(bsr_union_fill_kernel, dim3(nblk(n_rows, kGroups)), dim3(kB), 0, s, n_rows, x_offsets, x_columns,
                       x_values, alpha, y_offsets, y_columns, y_values, beta, z_offsets, z_columns, z_values, capacity,
                       nullptr);
  if (e == hipSuccess) e = hipGetLastError();
  if (e != hipSuccess) return bsr_hip(e, "bsr_axpy");
  if (static_cast<long long>(x_nnz) + y_nnz <= capacity) return IPC_OK;
  e = hipMemcpyAsync(w->host, z_offsets + n_rows, sizeof(int), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return bsr_hip(e, "bsr_axpy: block count readback");
  return *w->host > capacity ? *w->host : IPC_OK;
}

}  // extern "C"

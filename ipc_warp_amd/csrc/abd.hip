// Affine-body contact reduction (affine_body_dynamics.py:144-190): vertex
// contact Hessian blocks and forces carried onto the affine degrees of
// freedom q_b = [p, a0, a1, a2] of each body, with x_i = p + r_i.x a0 +
// r_i.y a1 + r_i.z a2 for the rest-frame coordinates r_i. A vertex triplet
// (v_i, v_j, H) adds c_a(v_i) c_c(v_j) H to the 3x3 block (4 b_i + a,
// 4 b_j + c) for a, c in 0..3, with c_0 = 1 and c_k = r_k-1; a block touching
// a fixed body is zero.
//
// The reference writes those 16 blocks per vertex triplet as new triplets
// and sorts them into BSR; with ~1e7 vertex triplets onto a handful of
// bodies that is ~1.6e8 triplets falling into a few rows. Here the blocks
// are summed where they are produced:
//   mark     one bit per (body, body) pair that receives a nonzero block,
//            each workgroup setting the distinct pairs of its triplets once;
//   pattern  the pairs as a BSR over bodies (rows sorted) and its DOF-level
//            BSR: body pair (A, B) owns the 16 blocks (4A + a, 4B + c);
//   reduce   each workgroup walks a contiguous run of vertex triplets, its
//            kept ones queued densely in order; its four waves go through
//            the queue together, wave a summing the blocks (a, 0..3) in fp64
//            registers while a lane's body pair stays the same; on a change
//            the wave adds the lanes' sums per body pair into one of up to
//            64 fp64 accumulator copies (workgroup index modulo the copy
//            count) with one atomic per value;
//   finish   values = scale * (sum of the copies) rounded to fp32.
// The forces reduce the same way per vertex (one body per vertex).
#include <cstdio>

#include "../../include/ipc_warp_amd.h"
#include "cull.hpp"
#include "ipc_kernels.hpp"
#include "scan.hpp"

using namespace ipcd;

struct ipc_abd {
  DevBuf bits;     // uint32 [n_b][words]: body pairs with a nonzero block
  DevBuf pcnt;     // int [n_b + 1]
  DevBuf poff;     // int [n_b + 1]: body-level offsets
  DevBuf pcol;     // int [pairs]: body-level columns
  DevBuf part;     // scan partials
  DevBuf acc;      // double [16 * pairs * 9]
  DevBuf facc;     // double [4 * n_b * 3]
  int* host = nullptr;
};

namespace {

constexpr int kB = 256;
constexpr int kWaves = kB / 64;
constexpr int kMaxBodies = 8192;

int abd_fail(int code, const char* what) {
  set_error(what);
  return code;
}

int abd_hip(hipError_t e, const char* where) {
  if (e == hipSuccess) return IPC_OK;
  char buf[512];
  std::snprintf(buf, sizeof(buf), "%s: %s", where, hipGetErrorString(e));
  set_error(buf);
  return -int(e);
}

inline int nblk(long long n, int per) { return int((n + per - 1) / per); }
inline int words_of(int nb) { return (nb + 31) >> 5; }

__global__ void fill_u32_kernel(unsigned* p, long long n) {
  for (long long i = blockIdx.x * (long long)kB + threadIdx.x; i < n; i += (long long)gridDim.x * kB) p[i] = 0u;
}

__global__ void fill_f64_kernel(double* p, long long n) {
  for (long long i = blockIdx.x * (long long)kB + threadIdx.x; i < n; i += (long long)gridDim.x * kB) p[i] = 0.0;
}

hipError_t zero_u32(unsigned* p, long long n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int g = nblk(n, kB) < 2048 ? nblk(n, kB) : 2048;
  hipLaunchKernelGGL(fill_u32_kernel, dim3(g), dim3(kB), 0, s, p, n);
  return hipGetLastError();
}

hipError_t zero_f64(double* p, long long n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int g = nblk(n, kB) < 2048 ? nblk(n, kB) : 2048;
  hipLaunchKernelGGL(fill_f64_kernel, dim3(g), dim3(kB), 0, s, p, n);
  return hipGetLastError();
}

// The body pair of a vertex triplet in range with both bodies free.
__device__ inline bool free_pair(int r, int c, int nv, int nb, const int* __restrict__ body,
                                 const int* __restrict__ fixed, int& bi, int& bj) {
  if (unsigned(r) >= unsigned(nv) || unsigned(c) >= unsigned(nv)) return false;
  bi = body[r];
  bj = body[c];
  return unsigned(bi) < unsigned(nb) && unsigned(bj) < unsigned(nb) && !fixed[bi] && !fixed[bj];
}

__device__ inline bool any_nonzero(const float* __restrict__ v) {
  float h[9];
  __builtin_memcpy(h, v, sizeof(h));
  bool nz = false;
#pragma unroll
  for (int k = 0; k < 9; ++k) nz |= !(h[k] == 0.0f);
  return nz;
}

constexpr int kMarkPer = 32;     // triplets per thread of the mark kernel
constexpr int kMarkSet = 256;    // LDS set of body pairs per workgroup
constexpr int kMarkProbes = 16;

// Bits of the body pairs receiving a nonzero block. Each workgroup collects
// the distinct pairs of its kB * kMarkPer triplets in an LDS set and sets
// each bit once; a pair that finds the set full sets its bit itself. A
// triplet whose pair is in the set already needs no look at its values: a
// list of few body pairs is then read without them (screw and nut, 9.95
// million triplets: 189 us with them, 50 without).
__global__ __launch_bounds__(kB) void mark_kernel(const int* __restrict__ rows, const int* __restrict__ cols,
                                                  const float* __restrict__ vals, int m, int nv, int nb,
                                                  const int* __restrict__ body, const int* __restrict__ fixed,
                                                  int words, unsigned* bits) {
  __shared__ unsigned set[kMarkSet];
  for (int i = threadIdx.x; i < kMarkSet; i += kB) set[i] = 0xffffffffu;
  __syncthreads();
  const long long base = (long long)blockIdx.x * kB * kMarkPer + threadIdx.x;
  constexpr int kAhead = 4;
  for (int k0 = 0; k0 < kMarkPer; k0 += kAhead) {
    int r[kAhead], c[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const long long t = base + (long long)(k0 + k) * kB;
      r[k] = t < m ? rows[t] : -1;
      c[k] = t < m ? cols[t] : -1;
    }
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      int bi, bj;
      if (!free_pair(r[k], c[k], nv, nb, body, fixed, bi, bj)) continue;
      const unsigned key = unsigned(bi) * unsigned(nb) + unsigned(bj);
      const unsigned h = (key * 2654435761u) >> 24;  // 8 bits: kMarkSet slots
      bool known = false;
      for (int probe = 0; probe < kMarkProbes && !known; ++probe) {
        const unsigned old = __hip_atomic_load(&set[(h + probe) & (kMarkSet - 1)], __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
        if (old == 0xffffffffu) break;
        known = old == key;
      }
      if (known || !any_nonzero(vals + 9 * (base + (long long)(k0 + k) * kB))) continue;
      bool placed = false;
      for (int probe = 0; probe < kMarkProbes && !placed; ++probe) {
        const unsigned old = atomicCAS(&set[(h + probe) & (kMarkSet - 1)], 0xffffffffu, key);
        placed = old == 0xffffffffu || old == key;
      }
      if (!placed) atomicOr(bits + (long long)bi * words + (bj >> 5), 1u << (bj & 31));
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kMarkSet; i += kB) {
    const unsigned key = set[i];
    if (key == 0xffffffffu) continue;
    const int bi = int(key / unsigned(nb)), bj = int(key % unsigned(nb));
    atomicOr(bits + (long long)bi * words + (bj >> 5), 1u << (bj & 31));
  }
}

__global__ void row_count_kernel(const unsigned* bits, int nb, int words, int* cnt) {
  const int r = blockIdx.x * kB + threadIdx.x;
  if (r > nb) return;
  int n = 0;
  if (r < nb)
    for (int k = 0; k < words; ++k) n += __popc(bits[(long long)r * words + k]);
  cnt[r] = n;
}

__global__ void row_fill_kernel(const unsigned* bits, int nb, int words, const int* off, int* col) {
  const int r = blockIdx.x * kB + threadIdx.x;
  if (r >= nb) return;
  int o = off[r];
  for (int k = 0; k < words; ++k) {
    unsigned w = bits[(long long)r * words + k];
    while (w) {
      const int j = __ffs(int(w)) - 1;
      col[o++] = 32 * k + j;
      w &= w - 1;
    }
  }
}

// DOF-level pattern: row 4A + a holds, for each body B of body row A in
// order, the blocks (4A + a, 4B + c), c = 0..3.
__global__ void dof_pattern_kernel(int nb, const int* poff, const int* pcol, int* offsets, int* columns) {
  const int R = blockIdx.x * kB + threadIdx.x;
  if (R > 4 * nb) return;
  if (R == 4 * nb) {
    offsets[R] = 16 * poff[nb];
    return;
  }
  const int A = R >> 2, a = R & 3;
  const int p0 = poff[A], len = poff[A + 1] - p0;
  const int o = 16 * p0 + 4 * a * len;
  offsets[R] = o;
  for (int j = 0; j < len; ++j) {
    const int B = pcol[p0 + j];
    if (columns) {
#pragma unroll
      for (int c = 0; c < 4; ++c) columns[o + 4 * j + c] = 4 * B + c;
    }
  }
}

// index of block (4A + a, 4B + c) in the DOF-level arrays
__device__ inline long long dof_block(const int* poff, const int* pcol, int A, int B, int a, int c) {
  const int p0 = poff[A], len = poff[A + 1] - p0;
  int lo = 0, hi = len - 1;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (pcol[p0 + mid] < B) lo = mid + 1;
    else hi = mid;
  }
  return 16ll * p0 + 4ll * a * len + 4 * lo + c;
}

constexpr int kPad = 65;    // LDS row pitch of the flush table (conflict-free both ways)
constexpr int kChunk = 12;  // values per LDS pass of a flush (3 passes of a wave's 36)
constexpr int kFlushKeys = 64 / kChunk;  // body pairs, or bodies, of a flush's batch

// Hands every pending lane sum of a wave over, N values each, up to kFlushKeys
// keys (body pairs, or bodies) at a time: per pass of kChunk values every lane
// writes its sums to LDS, then lane 12 p + k adds value k over the lanes of the
// batch's key p and issues the fp64 atomic, at to(key) + k. A single key (a list
// of few bodies) has four lanes a value add sixteen lanes each. A list of many
// body pairs flushes every few triplets: one pair at a time it waited for LDS (3
// million triplets of 1000 bodies 2170 us a call, 770 so).
template <int N, typename To>
__device__ __forceinline__ void flush_sums(int& cur_a, int cur_b, double* acc, int lane, double* sh, To to) {
  constexpr int kAhead = N == kChunk ? 8 : 4;  // reads in flight; the block sums leave no registers for more
  while (true) {
    // the batch's keys; lane 12 p + k keeps key p
    unsigned long long left = __ballot(cur_a >= 0), taken = 0ull, mask = 0ull;
    if (!left) break;
    const int mine = lane / kChunk, k = lane - kChunk * mine;
    int A = -1, B = -1, keys = 0;
#pragma unroll 1
    for (; keys < kFlushKeys && left; ++keys) {
      const int leader = __ffsll(static_cast<long long>(left)) - 1;
      const int pa = __builtin_amdgcn_readlane(cur_a, leader), pb = __builtin_amdgcn_readlane(cur_b, leader);
      const unsigned long long m = __ballot(cur_a == pa && cur_b == pb);
      if (mine == keys) {
        A = pa;
        B = pb;
        mask = m;
      }
      left &= ~m;
      taken |= m;
    }
    const bool add = mine < keys;
    double* out = nullptr;
    if (keys == 1) out = to(__shfl(A, 0), __shfl(B, 0));
    else if (add) out = to(A, B);
    const bool in = (taken >> lane) & 1;
#pragma unroll
    for (int c = 0; c < N / kChunk; ++c) {
#pragma unroll
      for (int i = 0; i < kChunk; ++i) sh[i * kPad + lane] = in ? acc[c * kChunk + i] : 0.0;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (keys == 1) {
        const int v = lane & 15, part = lane >> 4;
        double sum = 0.0;
        if (v < kChunk) {
          const double* p = sh + v * kPad + 16 * part;
          double u[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
          for (int j = 0; j < 16; ++j) u[j & 3] += p[j];
          sum = (u[0] + u[1]) + (u[2] + u[3]);
        }
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        if (lane < kChunk) atomicAdd(out + c * kChunk + lane, sum);
      } else if (add) {
        const double* p = sh + k * kPad;
        double sum = 0.0;
        for (unsigned long long m = mask; m;) {
          double u[kAhead];
#pragma unroll
          for (int j = 0; j < kAhead; ++j) {
            u[j] = m ? p[__ffsll(static_cast<long long>(m)) - 1] : 0.0;
            m &= m - 1;  // 0 stays 0
          }
#pragma unroll
          for (int j = 0; j < kAhead; j += 4) sum += (u[j] + u[j + 1]) + (u[j + 2] + u[j + 3]);
        }
        atomicAdd(out + c * kChunk + k, sum);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (in) {
      cur_a = -1;
#pragma unroll
      for (int i = 0; i < N; ++i) acc[i] = 0.0;
    }
  }
}

// What bounds it: the triplets are read once, but a triplet waits for its
// vertices, their bodies and its values in turn, and three in four of a
// contact list with a fixed body are dropped. With one lane a triplet and all
// 144 sums in its registers two waves a SIMD did not hide that (289 us for
// 9.95 million triplets); here the kept ones are first queued, and a wave
// holds 36 sums, so that four waves a SIMD run. The sums are fp64, since a
// lane adds up many triplets: fp32 ones lost more the longer the list (and
// took 58 us instead of 65 for 4 million triplets of two bodies).
constexpr int kQueuePer = 4;
constexpr int kQueueTile = kB * kQueuePer;
__global__ __launch_bounds__(kB) __attribute__((amdgpu_waves_per_eu(4))) void reduce_hessian_kernel(const int* __restrict__ rows,
                                                            const int* __restrict__ cols,
                                                            const float* __restrict__ vals, int m, int per_block,
                                                            int nv, int nb, const int* __restrict__ body,
                                                            const int* __restrict__ fixed,
                                                            const float* __restrict__ rest,
                                                            const int* __restrict__ poff,
                                                            const int* __restrict__ pcol, double* acc_reps, int reps,
                                                            long long rep_stride) {
  __shared__ int queue[2][kQueueTile];
  __shared__ int num[2][kQueuePer * kWaves];
  __shared__ double sh[kWaves][kChunk * kPad];
  const int lane = threadIdx.x & 63;
  const int a = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave, and its block row
  // workgroups spread their atomics over `reps` copies of the accumulator, so
  // a body pair shared by all is not one chain of atomics per value
  double* out = acc_reps + (blockIdx.x % reps) * rep_stride;
  // the four blocks (a, 0..3) of a body pair are neighbours
  const auto blocks_of = [&](int A, int B) { return out + 9 * dof_block(poff, pcol, A, B, a, 0); };
  const long long w0 = (long long)blockIdx.x * per_block;
  const long long w1 = w0 + per_block < m ? w0 + per_block : m;
  double acc[36];
#pragma unroll
  for (int k = 0; k < 36; ++k) acc[k] = 0.0;
  int cur_a = -1, cur_b = -1;
  int buf = 0;
  for (long long tile = w0; tile < w1; tile += kQueueTile, buf ^= 1) {
    bool keep[kQueuePer];
    int before[kQueuePer];
#pragma unroll
    for (int k = 0; k < kQueuePer; ++k) {
      const long long t = tile + k * kB + threadIdx.x;
      int bi, bj;
      keep[k] = t < w1 && free_pair(rows[t], cols[t], nv, nb, body, fixed, bi, bj) && any_nonzero(vals + 9 * t);
    }
#pragma unroll
    for (int k = 0; k < kQueuePer; ++k) {
      const unsigned long long b = __ballot(keep[k]);
      before[k] = __popcll(b & ((1ull << lane) - 1));
      if (lane == 0) num[buf][k * kWaves + a] = __popcll(b);
    }
    __syncthreads();
    int total = 0;
#pragma unroll
    for (int j = 0; j < kQueuePer * kWaves; ++j) {
      const int c = num[buf][j];
      if (j % kWaves == a) before[j / kWaves] += total;
      total += c;
    }
#pragma unroll
    for (int k = 0; k < kQueuePer; ++k)
      if (keep[k]) queue[buf][before[k]] = int(tile + k * kB + threadIdx.x);
    __syncthreads();
    for (int q = 0; q < total; q += 64) {
      const bool kept = q + lane < total;
      const long long t = kept ? queue[buf][q + lane] : 0;
      int r = 0, c = 0, bi = -1, bj = -1;
      if (kept) {
        r = rows[t];
        c = cols[t];
        bi = body[r];
        bj = body[c];
      }
      // a lane moving to another body pair first hands its sums to the wave (the
      // values are read after that: they would not stay in registers across it)
      if (__ballot(kept && cur_a >= 0 && (bi != cur_a || bj != cur_b)))
        flush_sums<36>(cur_a, cur_b, acc, lane, sh[a], blocks_of);
      float h[9], ca = 1.0f, cc[4];
      if (kept) {
        __builtin_memcpy(h, vals + 9 * t, sizeof(h));
        if (a > 0) ca = rest[3ll * r + a - 1];
        cc[0] = 1.0f;
        __builtin_memcpy(cc + 1, rest + 3ll * c, 12);
      }
      if (kept) {
        cur_a = bi;
        cur_b = bj;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const double w = double(ca) * double(cc[b]);
#pragma unroll
          for (int k = 0; k < 9; ++k) acc[b * 9 + k] = fma(w, double(h[k]), acc[b * 9 + k]);
        }
      }
    }
  }
  flush_sums<36>(cur_a, cur_b, acc, lane, sh[a], blocks_of);
}

// Triplets of a workgroup's contiguous run: about 2048 workgroups (twice what
// the device holds at once), in whole tiles of the queue or, for a list too
// short for those, whole waves. A list of many body pairs changes pair every
// few triplets and hands its sums over each time, so a short one has to be
// spread: 40 bodies, 1600 triplets 264 us with runs of a tile and 23 so
// (100,000: 85 and 42); two bodies 8.7 and 5.9 (300,000: 12.6 and 14.2).
// (Flushed a pair at a time; 12, 22, 6 and 15 us now.)
long long run_of(long long n) {
  constexpr long long kWgs = 2048;
  const long long per = (n + kWgs - 1) / kWgs;
  const long long unit = per < kQueueTile ? 64 : kQueueTile;
  return (per + unit - 1) / unit * unit;
}

// One wave a value, a lane a copy: for few values, whose copies one lane
// would wait for in turn.
__global__ void finish_few_kernel(const double* acc, int n, int reps, double scale, float* values) {
  const int i = (blockIdx.x * kB + threadIdx.x) >> 6, lane = threadIdx.x & 63;
  if (i >= n) return;
  double v = lane < reps ? acc[(long long)lane * n + i] : 0.0;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  if (lane == 0) values[i] = static_cast<float>(scale * v);
}

__global__ void finish_values_kernel(const double* acc, long long n, int reps, double scale, float* values) {
  for (long long i = blockIdx.x * (long long)kB + threadIdx.x; i < n; i += (long long)gridDim.x * kB) {
    double v = 0.0;
    for (int r = 0; r < reps; ++r) v += acc[r * n + i];
    values[i] = static_cast<float>(scale * v);
  }
}

// Forces: vertex i of a free body adds (f, r.x f, r.y f, r.z f) to its
// body's four rows. A wave walks 64 `run` vertices, a lane adding up in fp64
// while its body stays the same; on a change the wave hands its lanes' sums
// over, body by body.
__global__ __launch_bounds__(kB) void reduce_force_kernel(const float* __restrict__ force,
                                                          const float* __restrict__ rest,
                                                          const int* __restrict__ body,
                                                          const int* __restrict__ fixed, int nv, int nb, int run,
                                                          double* out) {
  __shared__ double sh[kWaves][kChunk * kPad];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const long long first = (long long)(blockIdx.x * kWaves + w) * 64 * run + lane;
  int cur = -1;
  double v[kChunk];
#pragma unroll
  for (int k = 0; k < kChunk; ++k) v[k] = 0.0;
  const auto sums_of = [&](int b, int) { return out + 12ll * b; };
  for (int q = 0; q < run; ++q) {
    const long long i = first + 64 * q;
    int b = -1;
    if (i < nv) {
      b = body[i];
      if (unsigned(b) >= unsigned(nb) || fixed[b]) b = -1;
    }
    if (__ballot(b >= 0 && cur >= 0 && b != cur)) flush_sums<kChunk>(cur, 0, v, lane, sh[w], sums_of);
    if (b >= 0) {
      cur = b;
      const double f[3] = {force[3 * i], force[3 * i + 1], force[3 * i + 2]};
      const double c[4] = {1.0, rest[3 * i], rest[3 * i + 1], rest[3 * i + 2]};
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int k = 0; k < 3; ++k) v[3 * a + k] = fma(c[a], f[k], v[3 * a + k]);
    }
  }
  flush_sums<kChunk>(cur, 0, v, lane, sh[w], sums_of);
}
static_assert(kChunk == 12, "a body's sums are one pass of a flush");

// Runs of 64 vertices of a wave of reduce_force_kernel. Atomics on one address
// take some 10 ns in turn, and a body's sums take one from each wave: at most
// some 256 (118k vertices of two bodies, 64 a wave: 26 us, 11 with four runs).
// Small bodies end a lane's run early: 64 spheres of 42 vertices took 38 us with
// eight runs a wave, 5 with one.
int force_run(int nv, int nb) {
  const long long per = (nv / nb + 64ll * 256 - 1) / (64ll * 256);
  return int(per < 1 ? 1 : (per > 8 ? 8 : per));
}

__global__ void finish_force_kernel(const double* acc, int n, float* out) {
  const int i = blockIdx.x * kB + threadIdx.x;
  if (i < n) out[i] += static_cast<float>(acc[i]);
}

}  // namespace

extern "C" {

int ipc_abd_create(ipc_abd** out) {
  if (!out) return abd_fail(IPC_EINVAL, "abd_create: null output");
  ipc_abd* w = new (std::nothrow) ipc_abd();
  if (!w) return abd_fail(IPC_EINVAL, "abd_create: out of host memory");
  hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&w->host), sizeof(int));
  if (e != hipSuccess) {
    delete w;
    return abd_hip(e, "abd_create");
  }
  *out = w;
  return IPC_OK;
}

int ipc_abd_destroy(ipc_abd* w) {
  if (!w) return IPC_OK;
  for (DevBuf* d : {&w->bits, &w->pcnt, &w->poff, &w->pcol, &w->part, &w->acc, &w->facc}) d->release();
  if (w->host) hipHostFree(w->host);
  delete w;
  return IPC_OK;
}

int ipc_abd_reduce_contacts(ipc_abd* w, int n_bodies, const int* body, const float* rest, const int* fixed,
                            int n_vertices, const int* rows, const int* cols, const float* vals, int n_triplets,
                            const float* force, double scale, int* offsets, int* columns, float* values, int capacity,
                            float* reduced_force, void* stream) {
  if (!w) return abd_fail(IPC_EINVAL, "abd_reduce_contacts: null workspace");
  if (n_bodies <= 0 || n_bodies > kMaxBodies)
    return abd_fail(IPC_EINVAL, "abd_reduce_contacts: n_bodies must be in [1, 8192]");
  if (n_vertices < 0 || n_triplets < 0 || capacity < 0) return abd_fail(IPC_EINVAL, "abd_reduce_contacts: negative size");
  if (!body || !rest || !fixed || !offsets) return abd_fail(IPC_EINVAL, "abd_reduce_contacts: null pointer");
  if (n_triplets > 0 && (!rows || !cols || !vals)) return abd_fail(IPC_EINVAL, "abd_reduce_contacts: null triplets");
  if (capacity > 0 && (!columns || !values)) return abd_fail(IPC_EINVAL, "abd_reduce_contacts: null columns/values");
  if (force && !reduced_force) return abd_fail(IPC_EINVAL, "abd_reduce_contacts: force given without reduced_force");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int nb = n_bodies, words = words_of(nb);
  hipError_t e = w->bits.ensure(sizeof(unsigned) * size_t(nb) * words);
  if (e == hipSuccess) e = w->pcnt.ensure(sizeof(int) * (size_t(nb) + 1));
  if (e == hipSuccess) e = w->poff.ensure(sizeof(int) * (size_t(nb) + 1));
  if (e != hipSuccess) return abd_hip(e, "abd_reduce_contacts: workspace");
  e = zero_u32(w->bits.as<unsigned>(), (long long)nb * words, s);
  if (e == hipSuccess && n_triplets > 0)
    hipLaunchKernelGGL(mark_kernel, dim3(nblk(n_triplets, kB * kMarkPer)), dim3(kB), 0, s, rows, cols, vals, n_triplets,
                       n_vertices, nb, body, fixed, words, w->bits.as<unsigned>());
  if (e == hipSuccess) e = hipGetLastError();
  if (e == hipSuccess)
    hipLaunchKernelGGL(row_count_kernel, dim3(nblk(nb + 1, kB)), dim3(kB), 0, s, w->bits.as<unsigned>(), nb, words,
                       w->pcnt.as<int>());
  if (e == hipSuccess) e = hipGetLastError();
  if (e == hipSuccess) e = exclusive_scan(w->pcnt.as<int>(), nb + 1, w->poff.as<int>(), w->part, s);
  if (e == hipSuccess) e = hipMemcpyAsync(w->host, w->poff.as<int>() + nb, sizeof(int), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return abd_hip(e, "abd_reduce_contacts: body pattern");
  const int pairs = *w->host;
  const long long blocks = 16ll * pairs;
  if (blocks > 0x7fffffffll) return abd_fail(IPC_EINVAL, "abd_reduce_contacts: pattern too large");
  // accumulator replicas: up to 64, within 64 MiB
  long long reps = (64ll << 20) / (72 * (blocks > 0 ? blocks : 1));
  reps = reps < 1 ? 1 : (reps > 64 ? 64 : reps);
  e = w->pcol.ensure(sizeof(int) * size_t(pairs > 0 ? pairs : 1));
  if (e == hipSuccess) e = w->acc.ensure(sizeof(double) * size_t(blocks > 0 ? blocks : 1) * 9 * size_t(reps));
  if (e == hipSuccess) e = w->facc.ensure(sizeof(double) * size_t(nb) * 12);
  if (e != hipSuccess) return abd_hip(e, "abd_reduce_contacts: accumulators");
  hipLaunchKernelGGL(row_fill_kernel, dim3(nblk(nb, kB)), dim3(kB), 0, s, w->bits.as<unsigned>(), nb, words,
                     w->poff.as<int>(), w->pcol.as<int>());
  e = hipGetLastError();
  if (e == hipSuccess)
    hipLaunchKernelGGL(dof_pattern_kernel, dim3(nblk(4 * nb + 1, kB)), dim3(kB), 0, s, nb, w->poff.as<int>(),
                       w->pcol.as<int>(), offsets, blocks <= capacity ? columns : nullptr);
  if (e == hipSuccess) e = hipGetLastError();
  if (e != hipSuccess) return abd_hip(e, "abd_reduce_contacts: pattern");
  if (blocks > capacity) return int(blocks);
  if (force) {
    e = zero_f64(w->facc.as<double>(), 12ll * nb, s);
    if (e == hipSuccess && n_vertices > 0)
    {
      const int run = force_run(n_vertices, nb);
      hipLaunchKernelGGL(reduce_force_kernel, dim3(nblk(n_vertices, kB * run)), dim3(kB), 0, s, force, rest, body,
                         fixed, n_vertices, nb, run, w->facc.as<double>());
    }
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess)
      hipLaunchKernelGGL(finish_force_kernel, dim3(nblk(12 * nb, kB)), dim3(kB), 0, s, w->facc.as<double>(), 12 * nb,
                         reduced_force);
    if (e == hipSuccess) e = hipGetLastError();
    if (e != hipSuccess) return abd_hip(e, "abd_reduce_contacts: force");
  }
  if (blocks == 0) return IPC_OK;
  e = zero_f64(w->acc.as<double>(), 9 * blocks * reps, s);
  if (e == hipSuccess && n_triplets > 0) {
    const long long per = run_of(n_triplets);
    hipLaunchKernelGGL(reduce_hessian_kernel, dim3(unsigned((n_triplets + per - 1) / per)), dim3(kB), 0, s, rows, cols,
                       vals, n_triplets, int(per), n_vertices, nb, body, fixed, rest, w->poff.as<int>(),
                       w->pcol.as<int>(), w->acc.as<double>(), int(reps), 9 * blocks);
    e = hipGetLastError();
  }
  if (e == hipSuccess) {
    const long long n = 9 * blocks;
    // up to 65536 values a wave each still fits the device at once
    if (n <= 65536)
      hipLaunchKernelGGL(finish_few_kernel, dim3(nblk(n, kWaves)), dim3(kB), 0, s, w->acc.as<double>(), int(n),
                         int(reps), scale, values);
    else
      hipLaunchKernelGGL(finish_values_kernel, dim3(nblk(n, kB) < 4096 ? nblk(n, kB) : 4096), dim3(kB), 0, s,
                         w->acc.as<double>(), n, int(reps), scale, values);
    e = hipGetLastError();
  }
  return abd_hip(e, "abd_reduce_contacts: reduce");
}

}  // extern "C"

// A wave's per-vertex sums of forces in LDS, on their way into a [V][3]
// array: neighbouring tets and contacts share vertices, and device atomics
// run at some 28 G cache lines/s (an instruction touches each of its lines
// once).
#pragma once

#include <hip/hip_runtime.h>

namespace ipcd {

// A wave's 64 N forces, N vertices a lane, with twice as many hash slots.
template <typename R, int N>
struct ForceSums {
  static constexpr int kSlots = 128 * N;
  static_assert((N & (N - 1)) == 0, "the hash masks");
  alignas(16) int key[kSlots];
  alignas(16) int at[kSlots];  // counts, then where a vertex's forces start
  int vert[64 * N];
  R f[3][64 * N];
};

// Whether a wave's active records (one a lane, four vertices each) share
// enough vertices for add_forces: an eighth of them name one that the record
// before names too. Lists come with neighbours side by side, or they share
// little that a wave could sum: a shuffled list of 262,144 contacts took 68 us
// summed and 60 added one by one, 455,625 shuffled tets 164 and 150. On a rod
// twist 88 % of the EE contacts do, 80 % of the PT contacts and 67 % of the
// tets; nearly none in a shuffled list.
__device__ __forceinline__ bool neighbours_share(const int4 v, bool active) {
  const int lane = threadIdx.x & 63;
  const int4 u = make_int4(__shfl_up(v.x, 1, 64), __shfl_up(v.y, 1, 64), __shfl_up(v.z, 1, 64), __shfl_up(v.w, 1, 64));
  const unsigned long long on = __ballot(active);
  const auto in = [&](int a) { return a == u.x || a == u.y || a == u.z || a == u.w; };
  const bool shares = active && lane > 0 && ((on >> (lane - 1)) & 1) && (in(v.x) || in(v.y) || in(v.z) || in(v.w));
  return 8 * __popcll(__ballot(shares)) >= __popcll(on);
}

// The other way: `records` records' twelve components each in f, their four
// vertices each in v, component j by lane j % 64, so that an instruction adds
// consecutive components of consecutive records and touches a few lines where
// their vertices are adjacent. A zero is not added.
template <typename R>
__device__ __forceinline__ void add_forces_one_by_one(const R* f, const int* v, int records, R* b) {
  for (int j = threadIdx.x & 63; j < 12 * records; j += 64) {
    const R x = f[j];
    if (x != R(0)) {
      const int slot = j / 12, comp = j - 12 * slot, vert = comp / 3;
      unsafeAtomicAdd(b + 3 * (long long)v[slot * 4 + vert] + (comp - 3 * vert), x);
    }
  }
}

// Adds f (three components a vertex) of the lanes with `active` into b, one
// atomic per distinct vertex and component of the wave. The forces are
// sorted by vertex (a hash slot per vertex, counted and scanned) and summed
// over runs of lanes. Float atomics in LDS on the slots themselves take
// about 190 clocks a wave instruction: with twelve of them a contact Hessian
// of 911k records of a rod twist took 193 us, and 169 so. Sixteen
// consecutive vertices share a group of slots, rotated by the group's hash
// (so that vertices 16 apart do not all meet), and a taken slot leads to the
// same place of the next group: the result walks runs of neighbouring
// vertices, several to a line. Called by all 64 lanes of a wave.
template <typename R, int N>
__device__ __forceinline__ void add_forces(ForceSums<R, N>& T, const int (&v)[N], const R (&f)[3 * N], bool active,
                                           R* b) {
  constexpr int slots = ForceSums<R, N>::kSlots;
  const int lane = threadIdx.x & 63;
  for (int i = lane; i < slots / 4; i += 64) {
    reinterpret_cast<int4*>(T.key)[i] = make_int4(-1, -1, -1, -1);
    reinterpret_cast<int4*>(T.at)[i] = make_int4(0, 0, 0, 0);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  int s[N], rank[N];
  bool on[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    on[k] = active && (f[3 * k] != R(0) || f[3 * k + 1] != R(0) || f[3 * k + 2] != R(0));
    const unsigned h = (unsigned(v[k]) >> 4) * 2654435761u;
    s[k] = int((h >> 12) & unsigned(slots - 16)) + int((unsigned(v[k]) + (h >> 28)) & 15u);
    if (on[k]) {
      for (;;) {
        const int was = atomicCAS(&T.key[s[k]], -1, v[k]);
        if (was == -1 || was == v[k]) break;
        s[k] += 16;
        if (s[k] >= slots) s[k] -= slots - 1;  // past the last group: the next place (every slot is tried but 0)
      }
      rank[k] = atomicAdd(&T.at[s[k]], 1);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  int c[2 * N], sum = 0, most = 0;
  __builtin_memcpy(c, T.at + 2 * N * lane, sizeof(c));
#pragma unroll
  for (int k = 0; k < 2 * N; ++k) {
    const int n = c[k];
    c[k] = sum;
    sum += n;
    most = max(most, n);
  }
  int end = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(end, d, 64);
    end += lane >= d ? u : 0;
  }
#pragma unroll
  for (int k = 0; k < 2 * N; ++k) c[k] += end - sum;
  __builtin_memcpy(T.at + 2 * N * lane, c, sizeof(c));
  const int total = __shfl(end, 63, 64);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int k = 0; k < N; ++k)
    if (on[k]) {
      const int p = T.at[s[k]] + rank[k];
      T.vert[p] = v[k];
#pragma unroll
      for (int a = 0; a < 3; ++a) T.f[a][p] = f[3 * k + a];
    }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  // A vertex's forces lie side by side: 64 at a time, lane l adds up those of
  // its vertex at and before l; the last one holds the sum and moves it to
  // the front. As many doublings as the longest run needs.
  int distinct = 0;
#pragma unroll 1
  for (int j = 0; j < total; j += 64) {
    const bool in = j + lane < total;
    const int vv = in ? T.vert[j + lane] : -1;
    R x[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) x[a] = in ? T.f[a][j + lane] : R(0);
#pragma unroll 1
    for (int d = 1; d < 64 && __any(most > d); d <<= 1) {
      const int before = __shfl_up(vv, d, 64);
      const bool same = before == vv && lane >= d;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const R u = __shfl_up(x[a], d, 64);
        x[a] += same ? u : R(0);
      }
    }
    const int next = __shfl_down(vv, 1, 64);  // by every lane: one that stays out hands its neighbour a zero
    const bool last = in && (lane == 63 || next != vv);
    const unsigned long long lasts = __ballot(last);
    if (last) {
      const int p = distinct + __popcll(lasts & ((1ull << lane) - 1));
      T.vert[p] = vv;
#pragma unroll
      for (int a = 0; a < 3; ++a) T.f[a][p] = x[a];
    }
    distinct += __popcll(lasts);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
  for (int i = lane; i < 3 * distinct; i += 64) {
    const int m = i / 3, a = i - 3 * m;
    const R x = T.f[a][m];
    if (x != R(0)) unsafeAtomicAdd(b + 3 * (long long)T.vert[m] + a, x);
  }
}

}  // namespace ipcd

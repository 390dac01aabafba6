// A workgroup's sums of per-vertex forces in LDS, on their way into a
// [V][3] array: neighbouring tets and contacts share vertices, and device
// atomics run at some 25 G/s however few bytes they carry.
#pragma once

#include <hip/hip_runtime.h>

namespace ipcd {

// Open addressing by vertex; at most SLOTS / 2 distinct vertices are added.
template <typename R, int SLOTS>
struct ForceTable {
  static_assert((SLOTS & (SLOTS - 1)) == 0, "the hash masks");
  int key[SLOTS];
  R f[3 * SLOTS];
};

// Called by the whole workgroup; a barrier must follow before the first add.
template <typename R, int SLOTS>
__device__ __forceinline__ void force_clear(ForceTable<R, SLOTS>& T) {
  for (int i = threadIdx.x; i < SLOTS; i += blockDim.x) T.key[i] = -1;
  for (int i = threadIdx.x; i < 3 * SLOTS; i += blockDim.x) T.f[i] = R(0);
}

template <typename R, int SLOTS>
__device__ __forceinline__ void force_add(ForceTable<R, SLOTS>& T, int v, R x, R y, R z) {
  if (x == R(0) && y == R(0) && z == R(0)) return;
  int s = int((unsigned(v) * 2654435761u) >> 16) & (SLOTS - 1);
  for (;;) {
    const int was = atomicCAS(&T.key[s], -1, v);
    if (was == -1 || was == v) break;
    s = (s + 1) & (SLOTS - 1);
  }
  unsafeAtomicAdd(&T.f[3 * s], x);
  unsafeAtomicAdd(&T.f[3 * s + 1], y);
  unsafeAtomicAdd(&T.f[3 * s + 2], z);
}

// Called by the whole workgroup after a barrier behind the last add.
template <typename R, int SLOTS>
__device__ __forceinline__ void force_flush(const ForceTable<R, SLOTS>& T, R* b) {
  for (int i = threadIdx.x; i < 3 * SLOTS; i += blockDim.x) {
    const int s = i / 3, v = T.key[s];
    const R x = T.f[i];
    if (v >= 0 && x != R(0)) unsafeAtomicAdd(b + 3 * (long long)v + (i - 3 * s), x);
  }
}

}  // namespace ipcd

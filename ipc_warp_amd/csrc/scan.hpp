// Device-wide int helpers shared by the assembly and active-set code: a fill
// kernel and an exclusive prefix sum in tiles of 4096 (256 lanes x 16), then
// the tile offsets added. Internal linkage: every
// translation unit that includes this keeps its own copy of the kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "cull.hpp"

namespace ipcd {
namespace {

constexpr int kScanB = 256;
constexpr int kScanPer = 16;
constexpr int kScanTile = kScanB * kScanPer;

__global__ void fill_i32_kernel(int* p, int n, int v) {
  for (int i = blockIdx.x * kScanB + threadIdx.x; i < n; i += gridDim.x * kScanB) p[i] = v;
}

hipError_t fill_i32(int* p, int n, int v, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int blocks = (n + kScanB - 1) / kScanB;
  const int g = blocks < 1024 ? blocks : 1024;
  hipLaunchKernelGGL(fill_i32_kernel, dim3(g), dim3(kScanB), 0, s, p, n, v);
  return hipGetLastError();
}

// Exclusive prefix of v over the workgroup's 256 lanes; sh holds 4 ints.
__device__ int block_exclusive(int v, int* sh, int& total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(x, d, 64);
    x += lane >= d ? u : 0;
  }
  __syncthreads();  // sh may still be read from the call before
  if (lane == 63) sh[w] = x;
  __syncthreads();
  const int s0 = sh[0], s1 = sh[1], s2 = sh[2], s3 = sh[3];
  total = s0 + s1 + s2 + s3;
  return x - v + (w > 0 ? s0 : 0) + (w > 1 ? s1 : 0) + (w > 2 ? s2 : 0);
}

__global__ __launch_bounds__(kScanB) void scan_tiles_kernel(const int* in, int n, int* out, int* tile_sum) {
  __shared__ int sh[4];
  const long long base = (long long)blockIdx.x * kScanTile + threadIdx.x * kScanPer;
  int v[kScanPer];
  int acc = 0;
  if (base + kScanPer <= n) {
    __builtin_memcpy(v, in + base, sizeof(v));
  } else {
#pragma unroll
    for (int k = 0; k < kScanPer; ++k) v[k] = base + k < n ? in[base + k] : 0;
  }
#pragma unroll
  for (int k = 0; k < kScanPer; ++k) acc += v[k];
  int total;
  int run = block_exclusive(acc, sh, total);
#pragma unroll
  for (int k = 0; k < kScanPer; ++k) {
    const int x = v[k];
    v[k] = run;
    run += x;
  }
  if (base + kScanPer <= n) {
    __builtin_memcpy(out + base, v, sizeof(v));
  } else {
#pragma unroll
    for (int k = 0; k < kScanPer; ++k)
      if (base + k < n) out[base + k] = v[k];
  }
  if (threadIdx.x == 0) tile_sum[blockIdx.x] = total;
}

// Adds to each tile past the first what the tiles before it sum to; every
// workgroup adds those sums itself (there are few), which saves the launch
// of a scan of theirs. The tile is read whole before any of it is written:
// read and written a value at a time, the sixteen accesses of a lane waited
// for each other (262k ints, 64 tiles: 6.5 us, 4.5 now).
__global__ __launch_bounds__(kScanB) void scan_add_kernel(int* out, int n, const int* tile_sum) {
  __shared__ int sh[4];
  const int tile = blockIdx.x + 1;
  const long long base = (long long)tile * kScanTile + threadIdx.x;
  int v[kScanPer];
#pragma unroll
  for (int k = 0; k < kScanPer; ++k) v[k] = base + k * kScanB < n ? out[base + k * kScanB] : 0;
  int part = 0;
  for (int i = threadIdx.x; i < tile; i += kScanB) part += tile_sum[i];
  int add;
  block_exclusive(part, sh, add);
#pragma unroll
  for (int k = 0; k < kScanPer; ++k)
    if (base + k * kScanB < n) out[base + k * kScanB] = v[k] + add;
}

// out[0..n) = exclusive prefix sums of in[0..n); in and out distinct. `part`
// holds one int per tile.
hipError_t exclusive_scan(const int* in, int n, int* out, DevBuf& part, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int nt = int(((long long)n + kScanTile - 1) / kScanTile);
  hipError_t e = part.ensure(sizeof(int) * size_t(nt));
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(scan_tiles_kernel, dim3(nt), dim3(kScanB), 0, s, in, n, out, part.as<int>());
  if (nt > 1) hipLaunchKernelGGL(scan_add_kernel, dim3(nt - 1), dim3(kScanB), 0, s, out, n, part.as<int>());
  return hipGetLastError();
}

}  // namespace
}  // namespace ipcd

// Block-sparse products and conjugate gradients over the BSR matrices of
// bsr.hip (3x3 fp32 blocks): the linear solve of the Newton system
// (warp.optim.linear.cg at time_integrator_base.py:500-507 and
// affine_body_dynamics.py:580-592).
//
// y = alpha A x + beta y: eight lanes per block row, each lane every eighth
// block of the row, the three sums reduced across the eight lanes.
//
// CG keeps every scalar on the device, and an iteration is two launches:
//   apply   beta from the sums the last update left, p = z + beta p formed
//           where the product gathers it (p has two buffers, so that no
//           workgroup reads what another has overwritten), q = A p, partial
//           sums of p.q;
//   update  alpha from those, x, r and z updated, partial sums of r.z and r.r.
// Every workgroup adds the partial sums it needs itself, all in the same
// fixed order, so no launch is spent on scalars, no host round trip happens
// between convergence checks and the result does not depend on scheduling.
// (Five launches an iteration, replayed as a graph that had to be captured
// anew for each set of buffers, took 27 us for 68,921 rows, 11 of them in
// the product; two take 17.)
#include <cmath>
#include <cstdio>

#include "../../include/ipc_warp_amd.h"
#include "cull.hpp"
#include "ipc_kernels.hpp"

using namespace ipcd;

struct ipc_cg {
  DevBuf r, q, dinv;      // float [3 n_rows]
  DevBuf zp0, zp1;        // float [6 n_rows]: z and p of a row side by side, two buffers in turn
  DevBuf part;            // double [kApplyGrid + 3 kUpdateGrid]: partial sums of p.q | r.z | r.r | b.b
  DevBuf scal;            // double [2]: r.z of the last two iterations
  double* host = nullptr; // pinned, written by the sums kernel: r.r, b.b
};

namespace {

constexpr int kB = 256;
constexpr int kGroup = 8;           // lanes per block row in the products
constexpr int kRowsPerBlock = kB / kGroup;
// CG's launches take 512 lanes a workgroup: as many waves in flight as with
// 256, and half the partial sums for every workgroup of the next launch to
// add. More workgroups than this go over their rows in strides.
constexpr int kCgB = 512;
constexpr int kCgRows = kCgB / kGroup;
constexpr int kApplyGrid = 4096, kUpdateGrid = 2048;

int cg_fail(int code, const char* what) {
  set_error(what);
  return code;
}

int cg_hip(hipError_t e, const char* where) {
  if (e == hipSuccess) return IPC_OK;
  char buf[512];
  std::snprintf(buf, sizeof(buf), "%s: %s", where, hipGetErrorString(e));
  set_error(buf);
  return -int(e);
}

inline int nblk(long long n, int per) { return int((n + per - 1) / per); }

// The workgroup's sum of v, for every lane: lanes by a butterfly, then the
// eight waves in order.
__device__ inline double block_sum(double v, double* sh) {
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m, 64);
  __syncthreads();  // sh may still be read from the sum before
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  return ((sh[0] + sh[1]) + (sh[2] + sh[3])) + ((sh[4] + sh[5]) + (sh[6] + sh[7]));
}

// Sum of np partial sums, the same in every workgroup; four loads at a time
// are in flight.
__device__ inline double part_sum(const double* part, int np, double* sh) {
  double v = 0.0;
  for (int i = threadIdx.x; i < np; i += 4 * kCgB) {
    double u[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) u[k] = i + k * kCgB < np ? part[i + k * kCgB] : 0.0;
    v += (u[0] + u[1]) + (u[2] + u[3]);
  }
  return block_sum(v, sh);
}

// Row r of A x for the calling 8-lane group (all its lanes get the sums).
__device__ inline void row_product(int r, int j, const int* off, const int* col, const float* val, const float* x,
                                   float& a0, float& a1, float& a2) {
  a0 = a1 = a2 = 0.0f;
  const int k1 = off[r + 1];
  for (int k = off[r] + j; k < k1; k += kGroup) {
    const float* v = val + 9ll * k;
    const float* xc = x + 3ll * col[k];
    const float x0 = xc[0], x1 = xc[1], x2 = xc[2];
    a0 += v[0] * x0 + v[1] * x1 + v[2] * x2;
    a1 += v[3] * x0 + v[4] * x1 + v[5] * x2;
    a2 += v[6] * x0 + v[7] * x1 + v[8] * x2;
  }
#pragma unroll
  for (int m = kGroup / 2; m > 0; m >>= 1) {
    a0 += __shfl_xor(a0, m, kGroup);
    a1 += __shfl_xor(a1, m, kGroup);
    a2 += __shfl_xor(a2, m, kGroup);
  }
}

__global__ __launch_bounds__(kB) void bsr_mv_kernel(int nr, const int* off, const int* col, const float* val,
                                                    const float* x, float* y, float alpha, float beta) {
  const int j = threadIdx.x & (kGroup - 1);
  for (int r = (blockIdx.x * kB + threadIdx.x) / kGroup; r < nr; r += gridDim.x * kRowsPerBlock) {
    float a0, a1, a2;
    row_product(r, j, off, col, val, x, a0, a1, a2);
    if (j == 0) {
      float* yr = y + 3ll * r;
      if (beta == 0.0f) {
        yr[0] = alpha * a0;
        yr[1] = alpha * a1;
        yr[2] = alpha * a2;
      } else {
        yr[0] = alpha * a0 + beta * yr[0];
        yr[1] = alpha * a1 + beta * yr[1];
        yr[2] = alpha * a2 + beta * yr[2];
      }
    }
  }
}

// p = z + beta p, rounded to fp32 once.
__device__ inline float direction(float z, float p, double beta) { return float(double(z) + beta * double(p)); }

// Two of a lane's blocks of a row (k and k + kGroup) with what they multiply.
struct BlockPair {
  float v[2][9], zp[2][6];
  bool two;
};
__device__ inline void load_pair(BlockPair& B, int k, int k1, const int* col, const float* val, const float* zp) {
  B.two = k + kGroup < k1;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int kk = u == 0 || !B.two ? k : k + kGroup;
    __builtin_memcpy(B.v[u], val + 9ll * kk, 36);
    __builtin_memcpy(B.zp[u], zp + 6ll * col[kk], 24);
  }
}

// p_new = z + beta p, q = A p_new and the partial sums of p_new.q. r.z of
// this iteration goes to rz[par], where the update and the next iteration
// read it. z and p lie side by side, so that a column is one gather; the
// first blocks are loaded before the sums, whose latency then hides theirs.
__global__ __launch_bounds__(kCgB) void cg_apply_kernel(int nr, const int* __restrict__ off, const int* __restrict__ col,
                                                        const float* __restrict__ val, const float* __restrict__ zp,
                                                        float* __restrict__ zp_new, float* __restrict__ q,
                                                        const double* part_rz, int np, double* rz, int par,
                                                        double* part_pq) {
  __shared__ double sh[kCgB / 64];
  const int j = threadIdx.x & (kGroup - 1);
  int r = (blockIdx.x * kCgB + threadIdx.x) / kGroup;
  int k = 0, k1 = 0;
  BlockPair B;
  float zr[2] = {0.0f, 0.0f};
  auto start_row = [&]() {
    if (r >= nr) return;
    k = off[r] + j;
    k1 = off[r + 1];
    if (k < k1) load_pair(B, k, k1, col, val, zp);
    if (j < 3) {
      zr[0] = zp[6ll * r + j];
      zr[1] = zp[6ll * r + 3 + j];
    }
  };
  start_row();
  const double rz_old = rz[1 - par];
  const double rz_new = part_sum(part_rz, np, sh);
  if (blockIdx.x == 0 && threadIdx.x == 0) rz[par] = rz_new;
  double beta = rz_old != 0.0 ? rz_new / rz_old : 0.0;
  if (!std::isfinite(beta)) beta = 0.0;
  double pq = 0.0;
  while (r < nr) {
    float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
    while (k < k1) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (u == 1 && !B.two) break;
        const float* v = B.v[u];
        const float x0 = direction(B.zp[u][0], B.zp[u][3], beta), x1 = direction(B.zp[u][1], B.zp[u][4], beta),
                    x2 = direction(B.zp[u][2], B.zp[u][5], beta);
        a0 += v[0] * x0 + v[1] * x1 + v[2] * x2;
        a1 += v[3] * x0 + v[4] * x1 + v[5] * x2;
        a2 += v[6] * x0 + v[7] * x1 + v[8] * x2;
      }
      k += 2 * kGroup;
      if (k < k1) load_pair(B, k, k1, col, val, zp);
    }
#pragma unroll
    for (int m = kGroup / 2; m > 0; m >>= 1) {
      a0 += __shfl_xor(a0, m, kGroup);
      a1 += __shfl_xor(a1, m, kGroup);
      a2 += __shfl_xor(a2, m, kGroup);
    }
    if (j < 3) {
      const float a = j == 0 ? a0 : (j == 1 ? a1 : a2);
      const float pi = direction(zr[0], zr[1], beta);
      zp_new[6ll * r + 3 + j] = pi;
      q[3ll * r + j] = a;
      pq += double(pi) * a;
    }
    r += gridDim.x * kCgRows;
    start_row();
  }
  const double s = block_sum(pq, sh);
  if (threadIdx.x == 0) part_pq[blockIdx.x] = s;
}

// x += alpha p, r -= alpha q, z = D^-1 r, one lane a row; partial sums of r.z
// and r.r.
__global__ __launch_bounds__(kCgB) void cg_update_kernel(int nr, float* __restrict__ x, float* __restrict__ r,
                                                         float* zp, const float* __restrict__ q,
                                                         const float* __restrict__ dinv, const double* part_pq, int np,
                                                         const double* rz_cur, double* part_rz, double* part_rr) {
  __shared__ double sh[kCgB / 64];
  int i = blockIdx.x * kCgB + threadIdx.x;
  float xi[3], ri[3], pi[3], qi[3], di[3] = {1.0f, 1.0f, 1.0f};
  auto load = [&]() {
    if (i >= nr) return;
    __builtin_memcpy(xi, x + 3ll * i, 12);
    __builtin_memcpy(ri, r + 3ll * i, 12);
    __builtin_memcpy(pi, zp + 6ll * i + 3, 12);
    __builtin_memcpy(qi, q + 3ll * i, 12);
    if (dinv) __builtin_memcpy(di, dinv + 3ll * i, 12);
  };
  load();
  const double rzc = *rz_cur;
  const double pq = part_sum(part_pq, np, sh);
  const double alpha = (pq > 0.0 && std::isfinite(pq)) ? rzc / pq : 0.0;
  double rz = 0.0, rr = 0.0;
  while (i < nr) {
    float zi[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      xi[c] = float(double(xi[c]) + alpha * double(pi[c]));
      ri[c] = float(double(ri[c]) - alpha * double(qi[c]));
      zi[c] = di[c] * ri[c];
      rz += double(ri[c]) * zi[c];
      rr += double(ri[c]) * ri[c];
    }
    __builtin_memcpy(x + 3ll * i, xi, 12);
    __builtin_memcpy(r + 3ll * i, ri, 12);
    __builtin_memcpy(zp + 6ll * i, zi, 12);
    i += gridDim.x * kCgB;
    load();
  }
  const double a = block_sum(rz, sh), b = block_sum(rr, sh);
  if (threadIdx.x == 0) {
    part_rz[blockIdx.x] = a;
    part_rr[blockIdx.x] = b;
  }
}

// r = b - q (q = A x), z = D^-1 r, p = 0; partial sums of r.z, r.r, b.b.
__global__ __launch_bounds__(kCgB) void cg_init_kernel(int nr, const float* b, const float* q, float* r, float* zp,
                                                       const float* dinv, double* rz_old, double* part_rz,
                                                       double* part_rr, double* part_bb) {
  __shared__ double sh[kCgB / 64];
  double rz = 0.0, rr = 0.0, bb = 0.0;
  for (int i = blockIdx.x * kCgB + threadIdx.x; i < nr; i += gridDim.x * kCgB) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float bi = b[3ll * i + c], ri = bi - q[3ll * i + c];
      const float zi = dinv ? dinv[3ll * i + c] * ri : ri;
      r[3ll * i + c] = ri;
      zp[6ll * i + c] = zi;
      zp[6ll * i + 3 + c] = 0.0f;
      rz += double(ri) * zi;
      rr += double(ri) * ri;
      bb += double(bi) * bi;
    }
  }
  const double a = block_sum(rz, sh), c = block_sum(rr, sh), d = block_sum(bb, sh);
  if (threadIdx.x == 0) {
    part_rz[blockIdx.x] = a;
    part_rr[blockIdx.x] = c;
    part_bb[blockIdx.x] = d;
    if (blockIdx.x == 0) *rz_old = 0.0;  // the first direction is z
  }
}

// r.r (and b.b) for the host, written to its pinned memory.
__global__ __launch_bounds__(kCgB) void cg_sums_kernel(const double* part_rr, const double* part_bb, int np,
                                                     double* host) {
  __shared__ double sh[kCgB / 64];
  const double rr = part_sum(part_rr, np, sh);
  const double bb = part_bb ? part_sum(part_bb, np, sh) : 0.0;
  if (threadIdx.x == 0) {
    host[0] = rr;
    if (part_bb) host[1] = bb;
  }
}

// Jacobi: the inverse diagonal of each row's diagonal block (1 where it is
// missing, zero or not finite).
__global__ void cg_diag_kernel(int nr, const int* off, const int* col, const float* val, float* dinv) {
  const int r = blockIdx.x * kB + threadIdx.x;
  if (r >= nr) return;
  float d[3] = {1.0f, 1.0f, 1.0f};
  for (int k = off[r]; k < off[r + 1]; ++k)
    if (col[k] == r) {
      const float* v = val + 9ll * k;
      d[0] = v[0];
      d[1] = v[4];
      d[2] = v[8];
      break;
    }
#pragma unroll
  for (int c = 0; c < 3; ++c) dinv[3ll * r + c] = (d[c] != 0.0f && std::isfinite(d[c])) ? 1.0f / d[c] : 1.0f;
}

int grid_for(long long items, int per, int most) {
  const int g = nblk(items, per);
  return g < 1 ? 1 : (g < most ? g : most);
}

}  // namespace

extern "C" {

int ipc_bsr_mv(int n_rows, const int* offsets, const int* columns, const float* values, const float* x, float* y,
               float alpha, float beta, void* stream) {
  if (n_rows < 0) return cg_fail(IPC_EINVAL, "bsr_mv: negative n_rows");
  if (n_rows == 0) return IPC_OK;
  if (!offsets || !x || !y) return cg_fail(IPC_EINVAL, "bsr_mv: null pointer");
  const int g = nblk(n_rows, kRowsPerBlock) < 8192 ? nblk(n_rows, kRowsPerBlock) : 8192;
  hipLaunchKernelGGL(bsr_mv_kernel, dim3(g), dim3(kB), 0, static_cast<hipStream_t>(stream), n_rows, offsets, columns,
                     values, x, y, alpha, beta);
  return cg_hip(hipGetLastError(), "bsr_mv");
}

int ipc_cg_create(ipc_cg** out) {
  if (!out) return cg_fail(IPC_EINVAL, "cg_create: null output");
  ipc_cg* w = new (std::nothrow) ipc_cg();
  if (!w) return cg_fail(IPC_EINVAL, "cg_create: out of host memory");
  hipError_t e = hipHostMalloc(reinterpret_cast<void**>(&w->host), 2 * sizeof(double));
  if (e != hipSuccess) {
    delete w;
    return cg_hip(e, "cg_create");
  }
  *out = w;
  return IPC_OK;
}

int ipc_cg_destroy(ipc_cg* w) {
  if (!w) return IPC_OK;
  for (DevBuf* d : {&w->r, &w->q, &w->dinv, &w->zp0, &w->zp1, &w->part, &w->scal}) d->release();
  if (w->host) hipHostFree(w->host);
  delete w;
  return IPC_OK;
}

int ipc_bsr_cg(ipc_cg* w, int n_rows, const int* offsets, const int* columns, const float* values, const float* b,
               float* x, float tol, int maxiter, int check_every, int jacobi, int* iterations, double* residual,
               void* stream) {
  if (!w) return cg_fail(IPC_EINVAL, "bsr_cg: null workspace");
  if (n_rows < 0) return cg_fail(IPC_EINVAL, "bsr_cg: negative n_rows");
  if (!(tol >= 0.0f)) return cg_fail(IPC_EINVAL, "bsr_cg: tol must be >= 0");
  if (iterations) *iterations = 0;
  if (residual) *residual = 0.0;
  if (n_rows == 0) return IPC_OK;
  if (!offsets || !b || !x) return cg_fail(IPC_EINVAL, "bsr_cg: null pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const long long n = 3ll * n_rows;
  hipError_t e = hipSuccess;
  for (DevBuf* d : {&w->r, &w->q}) {
    if (e == hipSuccess) e = d->ensure(sizeof(float) * size_t(n));
  }
  for (DevBuf* d : {&w->zp0, &w->zp1}) {
    if (e == hipSuccess) e = d->ensure(sizeof(float) * 2 * size_t(n));
  }
  if (e == hipSuccess && jacobi) e = w->dinv.ensure(sizeof(float) * size_t(n));
  if (e == hipSuccess) e = w->part.ensure(sizeof(double) * (kApplyGrid + 3 * kUpdateGrid));
  if (e == hipSuccess) e = w->scal.ensure(sizeof(double) * 2);
  if (e != hipSuccess) return cg_hip(e, "bsr_cg: workspace");
  float* r = w->r.as<float>();
  float* zp[2] = {w->zp0.as<float>(), w->zp1.as<float>()};
  float* q = w->q.as<float>();
  const float* dinv = jacobi ? w->dinv.as<float>() : nullptr;
  double* part_pq = w->part.as<double>();
  double* part_rz = part_pq + kApplyGrid;
  double* part_rr = part_rz + kUpdateGrid;
  double* part_bb = part_rr + kUpdateGrid;
  double* rz = w->scal.as<double>();
  const int gr = grid_for(n_rows, kCgRows, kApplyGrid), gv = grid_for(n_rows, kCgB, kUpdateGrid);
  if (jacobi)
    hipLaunchKernelGGL(cg_diag_kernel, dim3(nblk(n_rows, kB)), dim3(kB), 0, s, n_rows, offsets, columns, values,
                       w->dinv.as<float>());
  hipLaunchKernelGGL(bsr_mv_kernel, dim3(grid_for(n_rows, kRowsPerBlock, 8192)), dim3(kB), 0, s, n_rows, offsets,
                     columns, values, x, q, 1.0f, 0.0f);
  hipLaunchKernelGGL(cg_init_kernel, dim3(gv), dim3(kCgB), 0, s, n_rows, b, q, r, zp[0], dinv, rz + 1, part_rz,
                     part_rr, part_bb);
  hipLaunchKernelGGL(cg_sums_kernel, dim3(1), dim3(kCgB), 0, s, part_rr, part_bb, gv, w->host);
  e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return cg_hip(e, "bsr_cg: start");
  const double goal = double(tol) * double(tol) * w->host[1];
  double rr = w->host[0];
  if (residual) *residual = std::sqrt(rr);
  if (rr <= goal) return IPC_OK;
  if (maxiter <= 0) maxiter = 3 * n_rows;
  if (check_every <= 0) check_every = 10;
  // an even count, so that a run of iterations starts with the same buffers
  const int chunk = (check_every + 1) & ~1;
  int done = 0;
  while (done < maxiter) {
    for (int i = 0; i < chunk; ++i) {
      const int par = i & 1;
      hipLaunchKernelGGL(cg_apply_kernel, dim3(gr), dim3(kCgB), 0, s, n_rows, offsets, columns, values, zp[par],
                         zp[1 - par], q, part_rz, gv, rz, par, part_pq);
      hipLaunchKernelGGL(cg_update_kernel, dim3(gv), dim3(kCgB), 0, s, n_rows, x, r, zp[1 - par], q, dinv, part_pq, gr,
                         rz + par, part_rz, part_rr);
    }
    hipLaunchKernelGGL(cg_sums_kernel, dim3(1), dim3(kCgB), 0, s, part_rr, (const double*)nullptr, gv, w->host);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return cg_hip(e, "bsr_cg: iterations");
    done += chunk;
    rr = w->host[0];
    if (iterations) *iterations = done;
    if (residual) *residual = std::sqrt(rr);
    if (rr <= goal || !std::isfinite(rr)) break;
  }
  return IPC_OK;
}

}  // extern "C"

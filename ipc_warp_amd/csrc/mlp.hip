// Learned warm start: the MLP 48 -> 256 -> 256 -> 256 -> 3 (GELU, fp32) that
// predicts a vertex's converged Newton displacement. Forward, backward, loss
// and Adam are hand-written kernels: one launch for the four layers, two for
// the backward pass, every layer product on the fp32 matrix instructions.
//
// Parameters are one flat fp32 array: W1 [256][48], b1 [256], W2 [256][256],
// b2, W3 [256][256], b3, W4 [3][256], b4 [3] (W row-major, out x in).
// Activations of a forward pass with backward in mind ("work") hold
// Z1, H1, Z2, H2, Z3, H3, each [n][256] (pre-activation and GELU output).
#include <cmath>

#include "../../include/ipc_warp_amd.h"
#include "ipc_kernels.hpp"

namespace ipcd {

constexpr int kIn = IPC_MLP_IN, kHid = IPC_MLP_HIDDEN, kOut = IPC_MLP_OUT;
constexpr long long kOffW1 = 0;
constexpr long long kOffB1 = kOffW1 + (long long)kHid * kIn;
constexpr long long kOffW2 = kOffB1 + kHid;
constexpr long long kOffB2 = kOffW2 + (long long)kHid * kHid;
constexpr long long kOffW3 = kOffB2 + kHid;
constexpr long long kOffB3 = kOffW3 + (long long)kHid * kHid;
constexpr long long kOffW4 = kOffB3 + kHid;
constexpr long long kOffB4 = kOffW4 + (long long)kOut * kHid;
constexpr long long kParams = kOffB4 + kOut;
static_assert(kParams == IPC_MLP_PARAMS, "parameter layout");

// Phi(z), the normal distribution function, and E = exp(-z^2 / 2):
//     |z| < 1.25:  Phi(z) = 1/2 + z R(z^2)
//     else:        Phi(-|z|) = E q(|z|),  q(a) = erfcx(a / sqrt 2) / 2 = t P(t),  t = 1 / (1 + 0.3 a)
// with R and P fitted for the least error of Phi on [0, 1.25] (1.1e-9, as
// rounded here) and the least relative error of q on [1.25, 14] (2.8e-8;
// beyond it E underflows). Near zero q changes fast in t, whose rounding alone
// put 4e-8 into Phi: hence the two ranges. About 30 instructions without a
// branch; erff and expf took three times as many, as long as the matrix
// products themselves. In fp32 over normally distributed z gelu's error is
// 2.1e-8 rms (erff: 2.5e-8), its derivative's 2.5e-8 (2.7e-8). In the lower
// tail the relative error grows as z^2 (the rounding of E's exponent): 8e-7 at
// -4, 7e-6 at -13, where 1 + erff has no digit left.
constexpr float kCentre[7] = {7.110484148e-07f, -1.025638176e-05f, 1.173832643e-04f, -1.189327333e-03f,
                              9.974518791e-03f, -6.649057567e-02f, 3.989422917e-01f};
constexpr float kTail[8] = {2.305391431e-02f, -1.159644797e-01f, 1.503848433e-01f, -1.290252805e-02f,
                            1.113785654e-01f, 1.040908322e-01f,  1.202122197e-01f, 1.196582019e-01f};
__device__ __forceinline__ float phi_cdf(float z, float& e) {
  const float a = fabsf(z), s = z * z;
  e = __builtin_amdgcn_exp2f(s * -0.72134752044448170f);
  const float t = __builtin_amdgcn_rcpf(fmaf(0.3f, a, 1.0f));
  float r = kCentre[0], p = kTail[0];
#pragma unroll
  for (int k = 1; k < 7; ++k) r = fmaf(r, s, kCentre[k]);
#pragma unroll
  for (int k = 1; k < 8; ++k) p = fmaf(p, t, kTail[k]);
  const float lo = e * (p * t);
  const float far = z >= 0.f ? 1.0f - lo : lo;
  return a < 1.25f ? fmaf(z, r, 0.5f) : far;
}
__device__ __forceinline__ float gelu(float z) {
  float e;
  return z * phi_cdf(z, e);
}
__device__ __forceinline__ float gelu_grad(float z) {
  // d/dz [z Phi(z)] = Phi(z) + z phi(z)
  float e;
  const float c = phi_cdf(z, e);
  return fmaf(z * 0.39894228040143268f, e, c);
}

// ------------------------------------------------------------- MFMA tiles ----
// Every layer product runs on the fp32 matrix instructions (fp32 inputs and
// accumulators, as the VALU code before them had). Layouts used, for lane l:
//   16x16x4: A row l % 16, k l / 16; B column l % 16, k l / 16; result
//            column l % 16, rows 4 (l / 16) + 0..3
//   32x32x2: A row l % 32, k l / 32; B column l % 32, k l / 32; result
//            column l % 32, register q row 8 (q / 4) + 4 (l / 32) + q % 4
using f4 = __attribute__((ext_vector_type(4))) float;
using f16 = __attribute__((ext_vector_type(16))) float;
using f2 = __attribute__((ext_vector_type(2))) float;

// Wide global accesses at the 4-byte alignment the entry points ask for.
__device__ __forceinline__ f4 ld4(const float* p) { f4 v; __builtin_memcpy(&v, p, 16); return v; }
__device__ __forceinline__ f2 ld2(const float* p) { f2 v; __builtin_memcpy(&v, p, 8); return v; }
__device__ __forceinline__ void st4(float* p, f4 v) { __builtin_memcpy(p, &v, 16); }
__device__ __forceinline__ void st2(float* p, f2 v) { __builtin_memcpy(p, &v, 8); }

// The row kernels keep two or three weight stages in registers: two waves a
// SIMD hold them without a spill.
#define kFewWaves __attribute__((amdgpu_waves_per_eu(2, 2)))
constexpr int kThreads = 512;  // 8 waves, 32 of the 256 columns each
constexpr int kLd = kHid + 4;  // LDS row stride of an activation tile: a column of 16-byte reads meets every bank once
constexpr int kLdIn = kIn + 4;

// A wave's share of 64 k of a weight matrix, in registers: 32 columns of W^T
// (wt_) or W (w_). A layer is four of them; the kernels keep up to three, so
// that the loads of a stage run under the products of the two before it and
// across the barriers between layers. (With the loads beside their use a
// workgroup took 22 us for 16 rows, one load latency per stage.) The waves
// start a layer at different stages: rows of W are 1 KB apart, so in one
// column of it every wave would ask the same few L2 channels.
struct Stage {
  f4 b[8];
};
__device__ __forceinline__ int stage_k(int i, int wave) { return 64 * ((i + wave) & 3); }

// acc[rt][t] += A W^T for the wave's columns c0 + 16 t + l % 16: A the
// workgroup's 16 RT rows in LDS (row stride ld), W [256][K] row-major. A k
// step of 16 is four matrix instructions whose lane groups take k = 4 (l /
// 16) + s, so both operands are read 16 bytes at a time.
template <int K, int Q = 4>
__device__ __forceinline__ void wt_load(Stage& S, const float* __restrict__ W, int k0, int c0, int l) {
  const float* w = W + (c0 + (l & 15)) * K + k0 + 4 * (l >> 4);
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    S.b[q] = ld4(w + 16 * q);
    S.b[4 + q] = ld4(w + 16 * K + 16 * q);
  }
  __builtin_amdgcn_sched_barrier(0);  // the loads are issued here, not where they are used
}
template <int RT, int Q = 4>
__device__ __forceinline__ void wt_mul(f4 acc[RT][2], const Stage& S, const float* act, int ld, int k0, int l) {
  const float* ap = act + (l & 15) * ld + k0 + 4 * (l >> 4);
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    f4 a[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) a[rt] = *reinterpret_cast<const f4*>(ap + 16 * rt * ld + 16 * q);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc[rt][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[rt][s], S.b[4 * t + q][s], acc[rt][t], 0, 0, 0);
  }
}

// acc[rt][t] += A W for the wave's columns c0 + 2 (l % 16) + t: W [256][256]
// row-major, read 8 bytes a lane (16 lanes on 128 consecutive bytes).
__device__ __forceinline__ void w_load(Stage& S, const float* __restrict__ W, int k0, int c0, int l) {
  const float* w = W + (k0 + 4 * (l >> 4)) * kHid + c0 + 2 * (l & 15);
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int s = 0; s < 4; s += 2) {
      const f2 u = ld2(w + (16 * q + s) * kHid), v = ld2(w + (16 * q + s + 1) * kHid);
      S.b[2 * q + s / 2] = f4{u[0], u[1], v[0], v[1]};
    }
  __builtin_amdgcn_sched_barrier(0);
}
template <int RT>
__device__ __forceinline__ void w_mul(f4 acc[RT][2], const Stage& S, const float* act, int k0, int l) {
  const float* ap = act + (l & 15) * kLd + k0 + 4 * (l >> 4);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f4 a[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) a[rt] = *reinterpret_cast<const f4*>(ap + 16 * rt * kLd + 16 * q);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int t = 0; t < 2; ++t)
          acc[rt][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[rt][s], S.b[2 * q + s / 2][2 * (s & 1) + t], acc[rt][t],
                                                            0, 0, 0);
  }
}

template <int RT>
__device__ __forceinline__ void clear(f4 acc[RT][2]) {
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt][0] = acc[rt][1] = f4{0.f, 0.f, 0.f, 0.f};
}

// rows [r0, r0 + R) of src [n][W] into LDS, zero past n
template <int R, int W>
__device__ __forceinline__ void stage_rows(float* dst, int ld, const float* __restrict__ src, long long r0, int n) {
  constexpr int kQ = W / 4;
  for (int i = threadIdx.x; i < R * kQ; i += kThreads) {
    const int row = i / kQ, q = i - row * kQ;
    const f4 v = r0 + row < n ? ld4(src + (r0 + row) * W + 4 * q) : f4{0.f, 0.f, 0.f, 0.f};
    *reinterpret_cast<f4*>(dst + row * ld + 4 * q) = v;
  }
}

// --------------------------------------------------------------- forward ----
// All four layers of R rows in one workgroup: the activations stay in LDS and
// the weights (0.58 MB) come from L2. KEEP stores Z and H of each layer. The
// bound is the CU's own reads of the weights (64 bytes of each of 16 rows an
// instruction) beside the products: 23 us for up to 4096 rows, where four
// launches of a VALU product took 120 us; 84 of 148 TFLOP/s at 121,904 rows
// (45 before).
template <int R, bool KEEP>
__device__ __forceinline__ void layer_out(f4 acc[R / 16][2], float* act, const float bias[2], float* __restrict__ Z,
                                          float* __restrict__ H, long long r0, int n, int c0, int l) {
  constexpr int RT = R / 16;
  __syncthreads();  // every wave has read the tile
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int c = c0 + 16 * t + (l & 15);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = 16 * rt + 4 * (l >> 4) + q;
        const float z = acc[rt][t][q] + bias[t], h = gelu(z);
        act[row * kLd + c] = h;
        if (KEEP && r0 + row < n) {
          Z[(r0 + row) * kHid + c] = z;
          H[(r0 + row) * kHid + c] = h;
        }
      }
  }
  __syncthreads();
  clear<RT>(acc);
}

template <int R, bool KEEP>
__global__ void __launch_bounds__(kThreads) kFewWaves forward_kernel(const float* __restrict__ prm, int n,
                                                                     const float* __restrict__ x,
                                                                     float* __restrict__ y, float* __restrict__ work) {
  constexpr int RT = R / 16;
  __shared__ __align__(16) float act[R * kLd];
  __shared__ __align__(16) float w4[kOut * kHid];
  const long long r0 = (long long)blockIdx.x * R, L = (long long)n * kHid;
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6, c0 = 32 * w;
  const float *W1 = prm + kOffW1, *W2 = prm + kOffW2, *W3 = prm + kOffW3;
  stage_rows<R, kIn>(act, kLdIn, x, r0, n);
  if (threadIdx.x < kOut * kHid / 4) *reinterpret_cast<f4*>(w4 + 4 * threadIdx.x) = ld4(prm + kOffW4 + 4 * threadIdx.x);
  const int c = c0 + (l & 15);
  const float b1[2] = {prm[kOffB1 + c], prm[kOffB1 + c + 16]}, b2[2] = {prm[kOffB2 + c], prm[kOffB2 + c + 16]},
              b3[2] = {prm[kOffB3 + c], prm[kOffB3 + c + 16]};
  const int k0 = stage_k(0, w), k1 = stage_k(1, w), k2 = stage_k(2, w), k3 = stage_k(3, w);
  Stage A, B, C;
  wt_load<kIn, kIn / 16>(A, W1, 0, c0, l);
  wt_load<kHid>(B, W2, k0, c0, l);
  wt_load<kHid>(C, W2, k1, c0, l);
  f4 acc[RT][2];
  clear<RT>(acc);
  __syncthreads();
  wt_mul<RT, kIn / 16>(acc, A, act, kLdIn, 0, l);
  wt_load<kHid>(A, W2, k2, c0, l);
  layer_out<R, KEEP>(acc, act, b1, work, work + L, r0, n, c0, l);
  wt_mul<RT>(acc, B, act, kLd, k0, l);
  wt_load<kHid>(B, W2, k3, c0, l);
  wt_mul<RT>(acc, C, act, kLd, k1, l);
  wt_load<kHid>(C, W3, k0, c0, l);
  wt_mul<RT>(acc, A, act, kLd, k2, l);
  wt_load<kHid>(A, W3, k1, c0, l);
  wt_mul<RT>(acc, B, act, kLd, k3, l);
  wt_load<kHid>(B, W3, k2, c0, l);
  layer_out<R, KEEP>(acc, act, b2, work + 2 * L, work + 3 * L, r0, n, c0, l);
  wt_mul<RT>(acc, C, act, kLd, k0, l);
  wt_load<kHid>(C, W3, k3, c0, l);
  wt_mul<RT>(acc, A, act, kLd, k1, l);
  wt_mul<RT>(acc, B, act, kLd, k2, l);
  wt_mul<RT>(acc, C, act, kLd, k3, l);
  layer_out<R, KEEP>(acc, act, b3, work + 4 * L, work + 5 * L, r0, n, c0, l);
  // the three outputs of a row: kPer lanes, 4 values of H at a time
  constexpr int kPer = kThreads / R;
  const int row = threadIdx.x / kPer, part = threadIdx.x % kPer;
  float s[kOut] = {0.f, 0.f, 0.f};
  for (int k = 4 * part; k < kHid; k += 4 * kPer) {
    const f4 h = *reinterpret_cast<const f4*>(act + row * kLd + k);
#pragma unroll
    for (int o = 0; o < kOut; ++o) {
      const f4 v = *reinterpret_cast<const f4*>(w4 + o * kHid + k);
#pragma unroll
      for (int q = 0; q < 4; ++q) s[o] = fmaf(h[q], v[q], s[o]);
    }
  }
#pragma unroll
  for (int m = kPer / 2; m > 0; m >>= 1)
#pragma unroll
    for (int o = 0; o < kOut; ++o) s[o] += __shfl_xor(s[o], m, kPer);
  if (part == 0 && r0 + row < n) {
#pragma unroll
    for (int o = 0; o < kOut; ++o) y[(r0 + row) * kOut + o] = s[o] + prm[kOffB4 + o];
  }
}

// -------------------------------------------------------------- backward ----
// dZ3 = (dy W4) * gelu'(Z3) into dz3, dZ2 = (dZ3 W3) * gelu'(Z2) into dz2,
// R rows a workgroup.
template <int R>
__global__ void __launch_bounds__(kThreads) kFewWaves backward_rows_kernel(const float* __restrict__ prm, int n,
                                                                 const float* __restrict__ work,
                                                                 const float* __restrict__ dy, float* __restrict__ dz3,
                                                                 float* __restrict__ dz2) {
  constexpr int RT = R / 16;
  __shared__ __align__(16) float act[R * kLd];
  const long long r0 = (long long)blockIdx.x * R, L = (long long)n * kHid;
  const float *Z2 = work + 2 * L, *Z3 = work + 4 * L, *W3 = prm + kOffW3;
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6, c0 = 32 * w;
  const int k0 = stage_k(0, w), k1 = stage_k(1, w), k2 = stage_k(2, w), k3 = stage_k(3, w);
  Stage A, B, C;
  w_load(A, W3, k0, c0, l);
  w_load(B, W3, k1, c0, l);
  {
    const int c = threadIdx.x % kHid;
    const float* W4 = prm + kOffW4;
    const float u[kOut] = {W4[c], W4[kHid + c], W4[2 * kHid + c]};
    for (int row = threadIdx.x / kHid; row < R; row += kThreads / kHid) {
      float d = 0.f;
      if (r0 + row < n) {
        const float* dr = dy + (r0 + row) * kOut;
#pragma unroll
        for (int o = 0; o < kOut; ++o) d = fmaf(dr[o], u[o], d);
        d *= gelu_grad(Z3[(r0 + row) * kHid + c]);
        dz3[(r0 + row) * kHid + c] = d;
      }
      act[row * kLd + c] = d;
    }
  }
  w_load(C, W3, k2, c0, l);
  const int c = c0 + 2 * (l & 15), g = l >> 4;
  f2 z[RT][4];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const long long row = r0 + 16 * rt + 4 * g + q;
      z[rt][q] = row < n ? ld2(Z2 + row * kHid + c) : f2{0.f, 0.f};
    }
  __syncthreads();
  f4 acc[RT][2];
  clear<RT>(acc);
  w_mul<RT>(acc, A, act, k0, l);
  w_load(A, W3, k3, c0, l);
  w_mul<RT>(acc, B, act, k1, l);
  w_mul<RT>(acc, C, act, k2, l);
  w_mul<RT>(acc, A, act, k3, l);
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const long long row = r0 + 16 * rt + 4 * g + q;
      if (row < n)
        st2(dz2 + row * kHid + c,
            f2{acc[rt][0][q] * gelu_grad(z[rt][q][0]), acc[rt][1][q] * gelu_grad(z[rt][q][1])});
    }
}

// The parameter gradients, added into grad, in one launch of three kinds of
// workgroups: 40 us for 4096 rows, where the eight launches of a VALU product
// with three row splits (48 workgroups for 256 CUs) took 940 us. Each splits
// the batch rows, so that the small outputs (147k values) still fill the chip;
// a split adds its sums with one fp32 atomic a value, each of which rounds at
// the size of the whole sum, so there are at most kMaxSplits of them, and
// kMaxAdders of layer 1, whose splits are its tiles.
//   [0, b1)        layer 1: dZ1 = (dZ2 W2) * gelu'(Z1) of 64 rows in LDS,
//                  then dW1 += dZ1^T x and db1
//   [b1, b1 + b23) layers 3 and 2: a 64 x 128 tile of dW += dZ^T H, its rows
//                  split over the splits and again over four wave pairs,
//                  summed in LDS; db from the first column tile's operand
//   the rest       layer 4: dW4 += dy^T H3, db4
// A batch of more than kMaxAdders tiles takes layer 1 in a launch of its own
// after these (b1 = 0): a tile's sums go to memory, over its rows of dZ3, which
// nothing reads any more, and layer1_sum_kernel adds them up in fp64. Adding
// every tile's by atomics, 1905 a value for 121,904 rows, put an error of
// 6.4e-7 into dW1 where dy and x are positive (6e-8 so); the 128 of 8192 rows
// leave 1.7e-7, less than the 2.7e-7 of the VALU product's chain, and the two
// launches more cost 40 us there (78 against 117).
constexpr int kRows1 = 64;
constexpr int kTileR = 64, kTileC = 128;
constexpr int kTiles = (kHid / kTileR) * (kHid / kTileC);  // of one layer's dW
constexpr int kMaxSplits = 16;
constexpr int kMaxAdders = 128;
constexpr int kLayer1 = kHid * kIn + kHid;  // dW1 and db1, neighbours in grad
static_assert(kOffB1 == kOffW1 + kHid * kIn, "dW1 and db1 are neighbours");

// A tile's dW1 and db1: into grad by atomics, or (PART) stored to part.
template <bool PART>
__device__ __forceinline__ void layer1_block(float* lds, int block, const float* __restrict__ prm, int n,
                                             const float* __restrict__ x, const float* __restrict__ Z1,
                                             const float* __restrict__ dz2, float* out) {
  constexpr int RT = kRows1 / 16;
  float* act = lds;
  float* xs = lds + kRows1 * kLd;
  const long long r0 = (long long)block * kRows1;
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6, c0 = 32 * w;
  const float* W2 = prm + kOffW2;
  const int k0 = stage_k(0, w), k1 = stage_k(1, w), k2 = stage_k(2, w), k3 = stage_k(3, w);
  Stage A, B;
  w_load(A, W2, k0, c0, l);
  stage_rows<kRows1, kHid>(act, kLd, dz2, r0, n);
  stage_rows<kRows1, kIn>(xs, kLdIn, x, r0, n);
  w_load(B, W2, k1, c0, l);
  __syncthreads();
  const int j = l & 15, g = l >> 4;
  {
    const int c = c0 + 2 * j;
    f4 acc[RT][2];
    clear<RT>(acc);
    w_mul<RT>(acc, A, act, k0, l);
    w_load(A, W2, k2, c0, l);
    w_mul<RT>(acc, B, act, k1, l);
    w_load(B, W2, k3, c0, l);
    w_mul<RT>(acc, A, act, k2, l);
    w_mul<RT>(acc, B, act, k3, l);
    __syncthreads();  // every wave has read the tile
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = 16 * rt + 4 * g + q;
        f2 d = f2{0.f, 0.f};
        if (r0 + row < n) {
          const f2 z = ld2(Z1 + (r0 + row) * kHid + c);
          d = f2{acc[rt][0][q] * gelu_grad(z[0]), acc[rt][1][q] * gelu_grad(z[1])};
        }
        *reinterpret_cast<f2*>(act + row * kLd + c) = d;
      }
  }
  __syncthreads();
  // dW1 rows [c0, c0 + 32) of this wave: 2 x 3 tiles over the 64 batch rows
  f4 acc[2][3];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) acc[a][b] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < kRows1; k += 4) {
    float av[2], bv[3];
#pragma unroll
    for (int a = 0; a < 2; ++a) av[a] = act[(k + g) * kLd + c0 + 16 * a + j];
#pragma unroll
    for (int b = 0; b < 3; ++b) bv[b] = xs[(k + g) * kLdIn + 16 * b + j];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 3; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[a], bv[b], acc[a][b], 0, 0, 0);
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float* o = out + (c0 + 16 * a + 4 * g + q) * kIn + 16 * b + j;
        if (PART) *o = acc[a][b][q];
        else unsafeAtomicAdd(o, acc[a][b][q]);
      }
  if (threadIdx.x < kHid) {
    float s = 0.f;
    for (int r = 0; r < kRows1; ++r) s += act[r * kLd + threadIdx.x];
    float* o = out + kHid * kIn + threadIdx.x;
    if (PART) *o = s;
    else unsafeAtomicAdd(o, s);
  }
}

__device__ __forceinline__ void dw_tile_block(float* lds, int tile, int k_begin, int k_end, const float* __restrict__ dz,
                                              const float* __restrict__ h, float* dW, float* db) {
  constexpr int kAhead = 4;  // pairs of batch rows loaded ahead of their use
  const int tr0 = (tile / (kHid / kTileC)) * kTileR, tc0 = (tile % (kHid / kTileC)) * kTileC;
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int sub = w & 1, ks = w >> 1;
  const int i = l & 31, half = l >> 5;
  const int span = (k_end - k_begin + 3) / 4;
  const int kb = k_begin + ks * span, ke = min(k_end, kb + span);
  const float* ap = dz + tr0 + 2 * i;
  const float* bp = h + tc0 + 64 * sub + 2 * i;
  f16 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[a][b][q] = 0.f;
  f2 sum = f2{0.f, 0.f};
  f2 av[kAhead], bv[kAhead];
  auto load = [&](int k, f2* a, f2* b) {
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
      const int r = k + 2 * s + half;
      a[s] = b[s] = f2{0.f, 0.f};
      if (r < ke) {
        a[s] = ld2(ap + (long long)r * kHid);
        b[s] = ld2(bp + (long long)r * kHid);
      }
    }
  };
  load(kb, av, bv);
  for (int k = kb; k < ke; k += 2 * kAhead) {
    f2 an[kAhead], bn[kAhead];
    load(k + 2 * kAhead, an, bn);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
      sum += av[s];
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[s][a], bv[s][b], acc[a][b], 0, 0, 0);
    }
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
      av[s] = an[s];
      bv[s] = bn[s];
    }
  }
  // rows tr0 + 2 m + a, columns tc0 + 64 sub + 2 i + b: the four waves of a
  // column half are summed through LDS, one row parity at a time
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    float* mine = lds + w * (32 * 64);
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int m = 8 * (q / 4) + 4 * half + q % 4;
      *reinterpret_cast<f2*>(mine + m * 64 + 2 * i) = f2{acc[a][0][q], acc[a][1][q]};
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 32 * kTileC; e += kThreads) {
      const int m = e / kTileC, c = e % kTileC;
      const float* p = lds + (c / 64) * (32 * 64) + m * 64 + c % 64;
      const float v = (p[0] + p[2 * 32 * 64]) + (p[4 * 32 * 64] + p[6 * 32 * 64]);
      unsafeAtomicAdd(dW + (tr0 + 2 * m + a) * kHid + tc0 + c, v);
    }
    __syncthreads();
  }
  if (tc0 == 0) {
    if (sub == 0) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const float s = sum[b] + __shfl_xor(sum[b], 32, 64);
        if (half == 0) lds[ks * kTileR + 2 * i + b] = s;
      }
    }
    __syncthreads();
    if (threadIdx.x < kTileR) {
      const float* p = lds + threadIdx.x;
      unsafeAtomicAdd(db + tr0 + threadIdx.x, (p[0] + p[kTileR]) + (p[2 * kTileR] + p[3 * kTileR]));
    }
  }
}

__device__ __forceinline__ void layer4_block(float* lds, int k_begin, int k_end, const float* __restrict__ dy,
                                             const float* __restrict__ H3, float* grad) {
  // fp32 sums of kFold rows, those in fp64: one chain of a split's rows lost
  // more the larger the batch
  constexpr int kFold = 32, kParts = kThreads / kHid;
  const int c = threadIdx.x % kHid, part = threadIdx.x / kHid;
  double sd[kOut] = {0.0, 0.0, 0.0}, bd[kOut] = {0.0, 0.0, 0.0};
  for (int r0 = k_begin + part; r0 < k_end; r0 += kFold * kParts) {
    float s[kOut] = {0.f, 0.f, 0.f}, b[kOut] = {0.f, 0.f, 0.f};
    const int r1 = min(k_end, r0 + kFold * kParts);
#pragma unroll 4
    for (int r = r0; r < r1; r += kParts) {
      const float hv = H3[(long long)r * kHid + c];
#pragma unroll
      for (int o = 0; o < kOut; ++o) {
        const float d = dy[(long long)r * kOut + o];
        s[o] = fmaf(d, hv, s[o]);
        b[o] += d;
      }
    }
#pragma unroll
    for (int o = 0; o < kOut; ++o) {
      sd[o] += s[o];
      bd[o] += b[o];
    }
  }
  double* sums = reinterpret_cast<double*>(lds);
  if (part == 1) {
#pragma unroll
    for (int o = 0; o < kOut; ++o) sums[o * kHid + c] = sd[o];
    if (c == 0) {
#pragma unroll
      for (int o = 0; o < kOut; ++o) sums[kOut * kHid + o] = bd[o];
    }
  }
  __syncthreads();
  if (part == 0) {
#pragma unroll
    for (int o = 0; o < kOut; ++o) unsafeAtomicAdd(grad + kOffW4 + o * kHid + c, float(sd[o] + sums[o * kHid + c]));
    if (c == 0) {
#pragma unroll
      for (int o = 0; o < kOut; ++o) unsafeAtomicAdd(grad + kOffB4 + o, float(bd[o] + sums[kOut * kHid + o]));
    }
  }
}

__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) gradients_kernel(const float* __restrict__ prm, int n,
                                                             const float* __restrict__ x,
                                                             const float* __restrict__ work,
                                                             const float* __restrict__ dy,
                                                             const float* __restrict__ dz3,
                                                             const float* __restrict__ dz2, float* grad, int b1,
                                                             int b23, int chunk) {
  __shared__ __align__(16) float lds[kRows1 * (kLd + kLdIn)];
  static_assert(kRows1 * (kLd + kLdIn) >= 8 * 32 * 64, "the tiles' sums fit");
  const long long L = (long long)n * kHid;
  int blk = blockIdx.x;
  if (blk < b1) {
    layer1_block<false>(lds, blk, prm, n, x, work, dz2, grad + kOffW1);
    return;
  }
  blk -= b1;
  if (blk < b23) {
    // a split's tiles are neighbours, so that they share its rows in L2
    const int split = blk / (2 * kTiles), tile = blk % (2 * kTiles);
    const int k0 = split * chunk, k1 = min(n, k0 + chunk);
    if (tile < kTiles) dw_tile_block(lds, tile, k0, k1, dz3, work + 3 * L, grad + kOffW3, grad + kOffB3);
    else dw_tile_block(lds, tile - kTiles, k0, k1, dz2, work + L, grad + kOffW2, grad + kOffB2);
    return;
  }
  blk -= b23;
  layer4_block(lds, blk * chunk, min(n, (blk + 1) * chunk), dy, work + 5 * L, grad);
}

// Layer 1 of a large batch: the sums of the first `parts` tiles over their
// rows of `part` (dZ3's memory), a last tile of too few rows for that by
// atomics.
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) layer1_kernel(
    const float* __restrict__ prm, int n, const float* __restrict__ x, const float* __restrict__ work,
    const float* __restrict__ dz2, float* part, int parts, float* grad) {
  __shared__ __align__(16) float lds[kRows1 * (kLd + kLdIn)];
  const int blk = blockIdx.x;
  if (blk < parts) layer1_block<true>(lds, blk, prm, n, x, work, dz2, part + (long long)blk * kRows1 * kHid);
  else layer1_block<false>(lds, blk, prm, n, x, work, dz2, grad + kOffW1);
}

// grad += the tiles' sums: a lane a value, the tiles split over gridDim.y.
__global__ void __launch_bounds__(256) layer1_sum_kernel(const float* __restrict__ part, int parts, float* grad) {
  const int v = blockIdx.x * 256 + threadIdx.x;
  const int chunk = (parts + gridDim.y - 1) / gridDim.y;
  const int p0 = blockIdx.y * chunk, p1 = min(parts, p0 + chunk);
  if (p0 >= p1) return;
  double s = 0.0;
#pragma unroll 8
  for (int p = p0; p < p1; ++p) s += part[(long long)p * kRows1 * kHid + v];
  unsafeAtomicAdd(grad + kOffW1 + v, float(s));
}
static_assert(kLayer1 % 256 == 0, "whole workgroups of values");

// Weighted mean squared error over [n][3]: loss += sum w_i |y_i - t_i|^2 / W,
// dy = 2 w_i (y_i - t_i) / W with W = sum of weights (passed in).
__global__ void __launch_bounds__(256) mse_kernel(int n, const float* __restrict__ y, const float* __restrict__ t,
                                                  const float* __restrict__ w, float inv_wsum, float* __restrict__ dy,
                                                  double* loss) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  double l = 0.0;
  if (i < n) {
    float wi = w ? w[i] : 1.0f;
    for (int k = 0; k < kOut; ++k) {
      float d = y[3 * i + k] - t[3 * i + k];
      l += double(wi) * d * d;
      if (dy) dy[3 * i + k] = 2.0f * wi * d * inv_wsum;
    }
  }
  for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off, 64);
  __shared__ double part[4];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = l;
  __syncthreads();
  if (threadIdx.x == 0 && loss) {
    double s = part[0] + part[1] + part[2] + part[3];
    unsafeAtomicAdd(loss, s * double(inv_wsum));
  }
}

// Adam (Kingma & Ba 2015) with bias correction, step t >= 1.
__global__ void __launch_bounds__(256) adam_kernel(long long n, float* __restrict__ p, const float* __restrict__ g,
                                                   float* __restrict__ m, float* __restrict__ v, float lr, float b1,
                                                   float b2, float eps, float c1, float c2) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float gi = g[i];
  float mi = b1 * m[i] + (1.0f - b1) * gi;
  float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

__global__ void __launch_bounds__(256) zero_f32_kernel(long long n, float* p) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

// --------------------------------------------------------------- launchers ----
static inline unsigned gblocks(long long n, int bs) { return unsigned((n + bs - 1) / bs); }

// 32 rows a workgroup halve the reads of the weights; below 256 of those
// workgroups half of the chip would stand idle, and 16 rows are the better
// split.
constexpr int kWideRows = 32 * 256;

hipError_t mlp_forward(const float* prm, int n, const float* x, float* y, float* work, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const dim3 block(kThreads);
  if (n >= kWideRows) {
    if (work) hipLaunchKernelGGL((forward_kernel<32, true>), dim3(gblocks(n, 32)), block, 0, s, prm, n, x, y, work);
    else hipLaunchKernelGGL((forward_kernel<32, false>), dim3(gblocks(n, 32)), block, 0, s, prm, n, x, y, work);
  } else {
    if (work) hipLaunchKernelGGL((forward_kernel<16, true>), dim3(gblocks(n, 16)), block, 0, s, prm, n, x, y, work);
    else hipLaunchKernelGGL((forward_kernel<16, false>), dim3(gblocks(n, 16)), block, 0, s, prm, n, x, y, work);
  }
  return hipGetLastError();
}

hipError_t mlp_backward(const float* prm, int n, const float* x, const float* work, const float* dy, float* grad,
                        float* tmp, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const long long L = (long long)n * kHid;
  float *dz3 = tmp, *dz2 = tmp + L;
  if (n >= kWideRows)
    hipLaunchKernelGGL(backward_rows_kernel<32>, dim3(gblocks(n, 32)), dim3(kThreads), 0, s, prm, n, work, dy, dz3,
                       dz2);
  else
    hipLaunchKernelGGL(backward_rows_kernel<16>, dim3(gblocks(n, 16)), dim3(kThreads), 0, s, prm, n, work, dy, dz3,
                       dz2);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  int splits = gblocks(n, 256);
  if (splits > kMaxSplits) splits = kMaxSplits;
  const int chunk = gblocks(n, splits);
  splits = gblocks(n, chunk);
  const int tiles1 = gblocks(n, kRows1), b1 = tiles1 <= kMaxAdders ? tiles1 : 0, b23 = 2 * kTiles * splits;
  hipLaunchKernelGGL(gradients_kernel, dim3(b1 + b23 + splits), dim3(kThreads), 0, s, prm, n, x, work, dy, dz3, dz2,
                     grad, b1, b23, chunk);
  if (b1 == 0) {
    // the last tile's rows hold its sums if there are enough of them
    const int last = n - (tiles1 - 1) * kRows1;
    const int parts = last * kHid >= kLayer1 ? tiles1 : tiles1 - 1;
    hipLaunchKernelGGL(layer1_kernel, dim3(tiles1), dim3(kThreads), 0, s, prm, n, x, work, dz2, dz3, parts, grad);
    const int sums = gblocks(parts, 128);
    hipLaunchKernelGGL(layer1_sum_kernel, dim3(kLayer1 / 256, sums < kMaxSplits ? sums : kMaxSplits), dim3(256), 0, s,
                       dz3, parts, grad);
  }
  return hipGetLastError();
}

hipError_t mlp_mse(const float* y, const float* t, const float* w, int n, float wsum, float* dy, double* loss,
                   hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(mse_kernel, dim3(gblocks(n, 256)), dim3(256), 0, s, n, y, t, w, 1.0f / wsum, dy, loss);
  return hipGetLastError();
}

hipError_t mlp_adam(float* p, const float* g, float* m, float* v, long long n, float lr, float b1, float b2, float eps,
                    int step, hipStream_t s) {
  float c1 = 1.0f - powf(b1, float(step)), c2 = 1.0f - powf(b2, float(step));
  hipLaunchKernelGGL(adam_kernel, dim3(gblocks(n, 256)), dim3(256), 0, s, n, p, g, m, v, lr, b1, b2, eps, c1, c2);
  return hipGetLastError();
}

hipError_t zero_f32(float* p, long long n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(zero_f32_kernel, dim3(gblocks(n, 256)), dim3(256), 0, s, n, p);
  return hipGetLastError();
}

}  // namespace ipcd

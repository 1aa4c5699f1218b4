// HIP kernels of the learned subgrid-stress (SGS) closure for gfx950: the
// box filter of a DNS velocity field with its subgrid stress, the velocity
// gradient and its invariants on an LES grid, the closure network (a 3x3x3
// convolution of the invariant field and an MLP that gives the coefficients
// of a tensor basis), its training (FP32 forward, backward, Adam) and its
// inference in FP32 and on the bf16 matrix cores.
//
// The reference (a DNS code) has no LES closure; these kernels serve the LES
// that runs the same pseudo-spectral step on a coarse grid with the
// predicted stress added to the physical-space products.
//
// Fields are physical [c][y][z][x] (P = n^3 points per component, as the
// step's ux array); symmetric tensors are 6 components (11, 12, 13, 22, 23,
// 33).  Network (parameter vector theta, FP32, in this order):
//   W0[16][135] b0[16]   conv 3x3x3 over the 5 invariant fields, tanh; the
//                        input index k = ch * 27 + ((dy+1) * 3 + dz+1) * 3 + dx+1
//   W1[64][21]  b1[64]   input [lambda(5), h0(16)], tanh
//   W2[64][64]  b2[64]   tanh
//   W3[64][64]  b3[64]   tanh
//   W4[4][64]   b4[4]    basis coefficients g; tau = sum_n g_n T_n
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "fft_line.hpp"
#include "psdns_internal.h"
#include "sgs_internal.h"

namespace psdns {
namespace sgs {

__constant__ float kCw[6] = {1.f, 2.f, 2.f, 1.f, 2.f, 1.f};

// offsets of the parameter blocks in theta
constexpr int oW0 = 0, ob0 = oW0 + kConv * kIn0, oW1 = ob0 + kConv, ob1 = oW1 + kHid * kIn1, oW2 = ob1 + kHid,
              ob2 = oW2 + kHid * kHid, oW3 = ob2 + kHid, ob3 = oW3 + kHid * kHid, oW4 = ob3 + kHid,
              ob4 = oW4 + kBasis * kHid;
static_assert(ob4 + kBasis == kParams, "parameter layout");

__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

// ---------------------------------------------------------------------------
// Box filter: coarse point (y, z, x) = fine point (r y, r z, r x); separable
// (r + 1)-tap top-hat [1/2, 1, .., 1, 1/2] / r per direction (periodic).
// ubar_i and tau_ij = filter(u_i u_j) - ubar_i ubar_j (deviatoric) summed in
// FP64.  A work-group takes one coarse row (y, z): its threads lie along x, TX
// of them per fine row and 256 / TX fine rows at a time, so the (r + 1)^2 fine
// rows are read in whole lines, a thread's two half cells as vectors and the
// right end tap from the neighbour's line.  A fine row is read by up to four
// coarse rows, which are close in time on one XCD (xcd_block): from memory
// about once.  512^3 FP32 to 64^3: 1650 us with a thread per coarse point and
// strided taps, 394 us this way (1.6 GB read, 4.1 TB/s).  A row's loads are kept
// ahead of its sums, which the compiler does by itself in FP32 but not in FP64
// from r = 8 on: 512^3 FP64 to 32^3 2.49 ms with strided taps, 3.95 ms with the
// loads among the sums, 0.86 ms (3.2 GB, 3.8 TB/s); 1024^3 FP64 to 32^3 18.7,
// 30.1 and 5.5 ms; 256^3 FP64 to 32^3 268, 168 and 95 us.  r = 2 takes its right
// half and end tap as one vector: 256^3 to 128^3 FP32 118 -> 93 us (114 with
// strided taps).
// ---------------------------------------------------------------------------
template <typename R, int H>
struct Half {  // H consecutive values
  static constexpr int V = H >= 16 / (int)sizeof(R) ? 16 / (int)sizeof(R) : H;  // per load
  R v[H];
  __device__ __forceinline__ void load(const R* p) {
    typedef R vec __attribute__((ext_vector_type(V)));
#pragma unroll
    for (int i = 0; i < H / V; i++) {
      if constexpr (V == 1) {
        v[i] = p[i];
      } else {
        const vec q = *reinterpret_cast<const vec*>(p + V * i);
#pragma unroll
        for (int j = 0; j < V; j++) v[V * i + j] = q[j];
      }
    }
  }
};

template <typename R, int r>
__global__ void __launch_bounds__(256)
    k_box_filter(const R* __restrict__ u, int n, R* __restrict__ ubar, float* __restrict__ tau, int nc) {
  __shared__ double red[9][256];
  const size_t P = (size_t)nc * nc * nc, N3 = (size_t)n * n * n;
  const double inv = 1.0 / r;
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  const int cy = blk / nc, cz = blk % nc, m = n - 1;
  const int tx = min(nc, 256), nslot = 256 / tx, slot = threadIdx.x / tx;
  for (int cx = threadIdx.x % tx; cx < nc; cx += tx) {
    double s[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};  // u v w uu uv uw vv vw ww
    const int x0 = (cx * r - r / 2) & m, x1 = cx * r, x2 = (cx * r + r / 2) & m;
    for (int k = slot; k < (r + 1) * (r + 1); k += nslot) {
      const int dy = k / (r + 1), dz = k % (r + 1);
      const double wyz = ((dy == 0 || dy == r) ? 0.5 * inv : inv) * ((dz == 0 || dz == r) ? 0.5 * inv : inv);
      const R* row = u + ((size_t)((cy * r + dy - r / 2) & m) * n + ((cz * r + dz - r / 2) & m)) * n;
      Half<R, r / 2> lo[3], hi[3];
      R end[3];
#pragma unroll
      for (int v = 0; v < 3; v++) {
        lo[v].load(row + v * N3 + x0);
        if constexpr (r == 2) {
          Half<R, 2> p;  // x2 is x1 + 1
          p.load(row + v * N3 + x1);
          hi[v].v[0] = p.v[0];
          end[v] = p.v[1];
        } else {
          hi[v].load(row + v * N3 + x1);
          end[v] = row[v * N3 + x2];
        }
      }
      // the lanes of a wave are r values apart: a line that is not taken whole by
      // loads in a row is gone from the cache before its next one
      if constexpr (sizeof(R) == 8) __builtin_amdgcn_sched_barrier(0);
      double t[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i <= r; i++) {
        const double a = (double)(i < r / 2 ? lo[0].v[i % (r / 2)] : i < r ? hi[0].v[i % (r / 2)] : end[0]);
        const double b = (double)(i < r / 2 ? lo[1].v[i % (r / 2)] : i < r ? hi[1].v[i % (r / 2)] : end[1]);
        const double c = (double)(i < r / 2 ? lo[2].v[i % (r / 2)] : i < r ? hi[2].v[i % (r / 2)] : end[2]);
        const double h = i == 0 || i == r ? 0.5 : 1.0;
        const double ha = h * a, hb = h * b, hc = h * c;
        t[0] += ha;
        t[1] += hb;
        t[2] += hc;
        t[3] = fma(ha, a, t[3]);
        t[4] = fma(ha, b, t[4]);
        t[5] = fma(ha, c, t[5]);
        t[6] = fma(hb, b, t[6]);
        t[7] = fma(hb, c, t[7]);
        t[8] = fma(hc, c, t[8]);
      }
#pragma unroll
      for (int q = 0; q < 9; q++) s[q] = fma(wyz * inv, t[q], s[q]);
    }
    if (nslot > 1) {
#pragma unroll
      for (int q = 0; q < 9; q++) red[q][threadIdx.x] = s[q];
      __syncthreads();
      if (slot == 0)
        for (int i = 1; i < nslot; i++)
#pragma unroll
          for (int q = 0; q < 9; q++) s[q] += red[q][i * tx + cx];
    }
    if (slot == 0) {
      double t[6] = {s[3] - s[0] * s[0], s[4] - s[0] * s[1], s[5] - s[0] * s[2],
                     s[6] - s[1] * s[1], s[7] - s[1] * s[2], s[8] - s[2] * s[2]};
      const double tr = (t[0] + t[3] + t[5]) / 3.0;
      t[0] -= tr;
      t[3] -= tr;
      t[5] -= tr;
      const size_t p = ((size_t)cy * nc + cz) * nc + cx;
#pragma unroll
      for (int v = 0; v < 3; v++) ubar[v * P + p] = (R)s[v];
#pragma unroll
      for (int c = 0; c < 6; c++) tau[c * P + p] = (float)t[c];
    }
  }
}

// ---------------------------------------------------------------------------
// Invariants and tensor basis of A (9 physical fields, A[3 i + j] = du_i/dx_j)
// per point, in FP64: S = sym(A) - tr(A)/3 I, W = skew(A), q = |S|^2 + |W|^2;
// lambda = (tr S^2, tr W^2) / q, (tr S^3, tr W^2 S) / q^1.5, tr W^2 S^2 / q^2;
// T = delta^2 (|S| S, S W - W S, S^2 - tr S^2 / 3 I, W^2 - tr W^2 / 3 I).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void mm3(const double* a, const double* b, double* c) {
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int j = 0; j < 3; j++) c[3 * i + j] = a[3 * i] * b[j] + a[3 * i + 1] * b[3 + j] + a[3 * i + 2] * b[6 + j];
}

template <typename R>
__global__ void __launch_bounds__(256)
    k_invariants(const R* __restrict__ A, size_t P, double delta2, float* __restrict__ lam, float* __restrict__ T) {
  constexpr int si[6] = {0, 0, 0, 1, 1, 2}, sj[6] = {0, 1, 2, 1, 2, 2};
  for (size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x; p < P; p += (size_t)gridDim.x * blockDim.x) {
    double a[9];
#pragma unroll
    for (int e = 0; e < 9; e++) a[e] = (double)A[e * P + p];
    const double tra = (a[0] + a[4] + a[8]) / 3.0;
    double S[9], W[9];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = 0; j < 3; j++) {
        S[3 * i + j] = 0.5 * (a[3 * i + j] + a[3 * j + i]) - (i == j ? tra : 0.0);
        W[3 * i + j] = 0.5 * (a[3 * i + j] - a[3 * j + i]);
      }
    double S2[9], W2[9], S3[9], W2S[9], W2S2[9], SW[9], WS[9];
    mm3(S, S, S2);
    mm3(W, W, W2);
    mm3(S2, S, S3);
    mm3(W2, S, W2S);
    mm3(W2, S2, W2S2);
    mm3(S, W, SW);
    mm3(W, S, WS);
    const double s2 = S2[0] + S2[4] + S2[8], w2 = W2[0] + W2[4] + W2[8];
    const double q = fmax(s2 - w2, kQeps);
    const double q15 = q * sqrt(q);
    lam[0 * P + p] = (float)(s2 / q);
    lam[1 * P + p] = (float)(w2 / q);
    lam[2 * P + p] = (float)((S3[0] + S3[4] + S3[8]) / q15);
    lam[3 * P + p] = (float)((W2S[0] + W2S[4] + W2S[8]) / q15);
    lam[4 * P + p] = (float)((W2S2[0] + W2S2[4] + W2S2[8]) / (q * q));
    const double sm = sqrt(2.0 * s2);
#pragma unroll
    for (int c = 0; c < 6; c++) {
      const int e = 3 * si[c] + sj[c];
      const double d = si[c] == sj[c] ? 1.0 : 0.0;
      T[(0 * 6 + c) * P + p] = (float)(delta2 * sm * S[e]);
      T[(1 * 6 + c) * P + p] = (float)(delta2 * (SW[e] - WS[e]));
      T[(2 * 6 + c) * P + p] = (float)(delta2 * (S2[e] - s2 / 3.0 * d));
      T[(3 * 6 + c) * P + p] = (float)(delta2 * (W2[e] - w2 / 3.0 * d));
    }
  }
}

// ---------------------------------------------------------------------------
// Training (FP32).  A minibatch of B points is drawn from the snapshot store
// by the counter map g = splitmix64(base + b) mod (S P), base =
// splitmix64(seed * 0xD1B54A32D192ED03 + step).  k_train takes tiles of 64
// points through the whole network and back in one work-group: the gather,
// the layers, the loss, the gradients of the pre-activations and the weight
// gradients, which stay in the registers of its four waves over its tiles
// (tile t to work-group t mod gridDim) and leave as one row of partial sums;
// k_train_fold adds the rows in row order in FP64 and applies Adam.  No
// atomics and a grid that depends on B only: a step gives the same bits
// every time.
//
// The layers run on v_mfma_f32_16x16x4_f32 (FP32 operands, products and sums),
// transposed (Y^T = W X^T) with a wave's 16 points as the columns.  Lane l
// (r or c = l % 16, g = l / 16) supplies A[r][k] and B[k][c] for one k per
// instruction and receives D[4 g + jj][c].  With the K order k = 16 ob + 4 g +
// jj for step (ob, jj) the accumulators of a layer are the next layer's
// operand B, forward and (with W^T as operand A) backward, so activations and
// gradients stay in registers; the weights are read from LDS.  A weight
// gradient is dZ X^T over the tile's 64 points: dZ and X pass through LDS as
// [feature][point] rows, wave w forms the row block o = 16 w .. of it.
// What bounds it: the chain of a tile (gather, about 560 matrix instructions
// of 32 cycles, 52 tanhf, five exchanges through LDS) with one wave per SIMD:
// 45 us at B = 16384 (a tile per CU), 28 us at B = 1000 (52 and 35 with the
// weights copied to LDS by loops of a load and its store); its arithmetic (6
// x 12164 flops per point) would take 8 us on the matrix cores.
// 20 steps of B = 16384 took 37.4 ms as a gather, five layer kernels, four
// backward ones, five weight-gradient kernels with their folds and Adam (one
// thread per output: 286 us for a 64 x 64 weight gradient); 1.04 ms this way.
// ---------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTS = 64;        // points per tile
constexpr int kLd = kTS + 4;   // row stride of the [feature][point] and 64-wide weight rows
constexpr int kW0ld = kIn0 + 2;  // W0 rows, zero at k = 135 (K runs in fours)

__global__ void __launch_bounds__(256)
    k_train(const float* __restrict__ lam_s, const float* __restrict__ T_s, const float* __restrict__ tau_s, int n,
            int nsnap, uint64_t base, int B, float inv, const float* __restrict__ theta, float* __restrict__ part,
            double* __restrict__ lpart) {
  __shared__ float W0s[kConv * kW0ld], W1s[kHid * kIn1], W4s[kBasis * kLd];
  __shared__ __attribute__((aligned(16))) float W2s[kHid * kLd], W3s[kHid * kLd];
  __shared__ float b0s[kConv], b1s[kHid], b2s[kHid], b3s[kHid], b4s[kBasis];
  __shared__ __attribute__((aligned(16))) float X0s[144 * kLd];  // conv inputs, rows 135.. zero
  __shared__ __attribute__((aligned(16))) float Ps[kHid * kLd], Qs[kHid * kLd];
  __shared__ float Ts[24 * kTS], taus[6 * kTS];
  __shared__ double red[4];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
  {
    // all loads first: a loop of a load and its store waits for each
    f32x4 w2[4], w3[4];
    float w0[9], w1[6];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      w2[i] = *(const f32x4*)(theta + oW2 + 4 * (tid + 256 * i));
      w3[i] = *(const f32x4*)(theta + oW3 + 4 * (tid + 256 * i));
    }
#pragma unroll
    for (int i = 0; i < 9; i++) w0[i] = theta[oW0 + min(tid + 256 * i, kConv * kIn0 - 1)];
#pragma unroll
    for (int i = 0; i < 6; i++) w1[i] = theta[oW1 + min(tid + 256 * i, kHid * kIn1 - 1)];
    const float w4 = theta[oW4 + tid];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int e = 4 * (tid + 256 * i), o = e / kHid * kLd + e % kHid;
      *(f32x4*)(W2s + o) = w2[i];
      *(f32x4*)(W3s + o) = w3[i];
    }
#pragma unroll
    for (int i = 0; i < 9; i++) {
      const int e = tid + 256 * i;
      if (e < kConv * kIn0) W0s[e / kIn0 * kW0ld + e % kIn0] = w0[i];
    }
#pragma unroll
    for (int i = 0; i < 6; i++)
      if (tid + 256 * i < kHid * kIn1) W1s[tid + 256 * i] = w1[i];
    W4s[tid / kHid * kLd + tid % kHid] = w4;
    if (tid < 2 * kConv) W0s[tid / 2 * kW0ld + kIn0 + tid % 2] = 0.f;
  }
  if (tid < kHid) {
    b1s[tid] = theta[ob1 + tid];
    b2s[tid] = theta[ob2 + tid];
    b3s[tid] = theta[ob3 + tid];
  }
  if (tid < kConv) b0s[tid] = theta[ob0 + tid];
  if (tid < kBasis) b4s[tid] = theta[ob4 + tid];
  for (int i = tid; i < (144 - kIn0) * kLd; i += 256) X0s[kIn0 * kLd + i] = 0.f;

  auto mm = [](float a, float b, f32x4 d) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, d, 0, 0, 0); };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 gW0[3] = {zero, zero, zero}, gW1[2] = {zero, zero}, gW2[4] = {zero, zero, zero, zero},
        gW3[4] = {zero, zero, zero, zero}, gW4 = zero;
  float gb0 = 0.f, gb1 = 0.f, gb2 = 0.f, gb3 = 0.f, gb4 = 0.f;
  double lsum = 0.0;
  const size_t P = (size_t)n * n * n;
  const int m = n - 1, col = 16 * w + c;
  // rows 16 ob + 4 g + jj of a layer's D to an LDS array
  auto put = [&](float* S, const f32x4* d, int nob) {
#pragma unroll
    for (int o = 0; o < 4; o++)
      if (o < nob)
#pragma unroll
        for (int jj = 0; jj < 4; jj++) S[(16 * o + 4 * g + jj) * kLd + col] = d[o][jj];
  };
  // acc += the 16 x 16 block (rows of dz, rows of x) of dZ X^T over 64 points
  auto wgrad = [&](f32x4& acc, const float* dz, const float* x) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const f32x4 a = *(const f32x4*)(dz + c * kLd + 16 * q + 4 * g), b = *(const f32x4*)(x + c * kLd + 16 * q + 4 * g);
#pragma unroll
      for (int jj = 0; jj < 4; jj++) acc = mm(a[jj], b[jj], acc);
    }
  };
  // row sums (this lane's share) of a 16-row block
  auto bgrad = [&](float& acc, const float* dz) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const f32x4 a = *(const f32x4*)(dz + c * kLd + 16 * q + 4 * g);
      acc += (a[0] + a[1]) + (a[2] + a[3]);
    }
  };
  // dense 64 -> 64: rows of W (or, TR, of W^T) against the registers x
  auto dense = [&](const float* W, const f32x4* x, f32x4 d, int ob, bool tr) {
#pragma unroll
    for (int o = 0; o < 4; o++) {
      f32x4 a;
      if (tr) {
#pragma unroll
        for (int jj = 0; jj < 4; jj++) a[jj] = W[(16 * o + 4 * g + jj) * kLd + 16 * ob + c];
      } else {
        a = *(const f32x4*)(W + (16 * ob + c) * kLd + 16 * o + 4 * g);
      }
#pragma unroll
      for (int jj = 0; jj < 4; jj++) d = mm(a[jj], x[o][jj], d);
    }
    return d;
  };

  const int ntiles = (B + kTS - 1) / kTS;
  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    // gather: point lane of the tile; wave w takes every fourth row of three
    // x neighbours, basis entry and stress component (points past B repeat the
    // batch's last one with a zero gradient, so that no value meets the sums
    // that the batch does not have: not a point that was not drawn, and not a
    // zero input to an infinite weight)
    {
      const int b = min(t * kTS + lane, B - 1);
      const uint64_t gidx = splitmix64(base + (uint64_t)b) % ((uint64_t)nsnap * P);
      const size_t s = gidx / P, p = gidx % P;
      const int y = (int)(p / ((size_t)n * n)), z = (int)((p / n) & m), x = (int)(p & m);
      const float* lam = lam_s + s * kLam * P;
      float v[12][3], tv[6], uv[2];
#pragma unroll
      for (int i = 0; i < 12; i++) {
        const int row = min(w + 4 * i, kLam * 9 - 1);  // ch, dy, dz
        const float* src = lam + (row / 9) * P +
                           (((size_t)((y + (row / 3) % 3 - 1) & m) * n + ((z + row % 3 - 1) & m)) * n);
        v[i][0] = src[(x - 1) & m];
        v[i][1] = src[x];
        v[i][2] = src[(x + 1) & m];
      }
#pragma unroll
      for (int i = 0; i < 6; i++) tv[i] = T_s[(s * 24 + w + 4 * i) * P + p];
#pragma unroll
      for (int i = 0; i < 2; i++) uv[i] = tau_s[(s * 6 + min(w + 4 * i, 5)) * P + p];
#pragma unroll
      for (int i = 0; i < 12; i++)
        if (w + 4 * i < kLam * 9)
#pragma unroll
          for (int d = 0; d < 3; d++) X0s[(3 * (w + 4 * i) + d) * kLd + lane] = v[i][d];
#pragma unroll
      for (int i = 0; i < 6; i++) Ts[(w + 4 * i) * kTS + lane] = tv[i];
#pragma unroll
      for (int i = 0; i < 2; i++)
        if (w + 4 * i < 6) taus[(w + 4 * i) * kTS + lane] = uv[i];
    }
    __syncthreads();
    // forward
    f32x4 h0, h1[4], h2[4], h3[4];
#pragma unroll
    for (int jj = 0; jj < 4; jj++) h0[jj] = b0s[4 * g + jj];
#pragma unroll
    for (int k = 0; k < 136; k += 4) h0 = mm(W0s[c * kW0ld + k + g], X0s[(k + g) * kLd + col], h0);
#pragma unroll
    for (int jj = 0; jj < 4; jj++) h0[jj] = tanhf(h0[jj]);
    const float l0 = X0s[(27 * g + 13) * kLd + col], l1 = g == 0 ? X0s[(27 * 4 + 13) * kLd + col] : 0.f;
#pragma unroll
    for (int ob = 0; ob < 4; ob++) {
      const float* wr = W1s + (16 * ob + c) * kIn1;
      f32x4 d;
#pragma unroll
      for (int jj = 0; jj < 4; jj++) d[jj] = b1s[16 * ob + 4 * g + jj];
      d = mm(wr[g], l0, d);
      d = mm(g == 0 ? wr[4] : 0.f, l1, d);  // an empty slot is zero in both operands
#pragma unroll
      for (int jj = 0; jj < 4; jj++) d = mm(wr[kLam + 4 * g + jj], h0[jj], d);
#pragma unroll
      for (int jj = 0; jj < 4; jj++) h1[ob][jj] = tanhf(d[jj]);
    }
#pragma unroll
    for (int ob = 0; ob < 4; ob++) {
      f32x4 d;
#pragma unroll
      for (int jj = 0; jj < 4; jj++) d[jj] = b2s[16 * ob + 4 * g + jj];
      d = dense(W2s, h1, d, ob, false);
#pragma unroll
      for (int jj = 0; jj < 4; jj++) h2[ob][jj] = tanhf(d[jj]);
    }
#pragma unroll
    for (int ob = 0; ob < 4; ob++) {
      f32x4 d;
#pragma unroll
      for (int jj = 0; jj < 4; jj++) d[jj] = b3s[16 * ob + 4 * g + jj];
      d = dense(W3s, h2, d, ob, false);
#pragma unroll
      for (int jj = 0; jj < 4; jj++) h3[ob][jj] = tanhf(d[jj]);
    }
    // output layer: rows 0..3 (lanes 0..15) are the coefficients of point col
    f32x4 gc;
#pragma unroll
    for (int jj = 0; jj < 4; jj++) gc[jj] = b4s[jj];
#pragma unroll
    for (int o = 0; o < 4; o++)
#pragma unroll
      for (int jj = 0; jj < 4; jj++)
        gc = mm(W4s[(c & 3) * kLd + 16 * o + 4 * g + jj], h3[o][jj], gc);
    // loss terms: e = sum_n g_n T_n - tau; dG_n = 2 inv sum_c cw_c e_c T_n,c
    double l = 0.0;
    if (g == 0) {
      const bool live = t * kTS + col < B;
      float dg[kBasis] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < 6; q++) {
        float e = -taus[q * kTS + col];
#pragma unroll
        for (int k = 0; k < kBasis; k++) e = fmaf(gc[k], Ts[(k * 6 + q) * kTS + col], e);
        l += (double)kCw[q] * (double)e * (double)e;
#pragma unroll
        for (int k = 0; k < kBasis; k++) dg[k] = fmaf(kCw[q] * e, Ts[(k * 6 + q) * kTS + col], dg[k]);
      }
      if (!live) l = 0.0;
#pragma unroll
      for (int k = 0; k < kBasis; k++) Ps[k * kLd + col] = live ? 2.f * inv * dg[k] : 0.f;
    }
    for (int off = 8; off > 0; off >>= 1) l += __shfl_xor(l, off);
    lsum += l;
    put(Qs, h3, 4);
    __syncthreads();
    // W4 (rows 4 .. 15 of the block are not used) and dZ3 = W4^T dG (1 - h3^2)
    wgrad(gW4, Ps, Qs + 16 * w * kLd);
    bgrad(gb4, Ps);
    f32x4 d3[4], d2[4], d1[4], d0;
    const float dgk = Ps[g * kLd + col];
#pragma unroll
    for (int ob = 0; ob < 4; ob++) {
      d3[ob] = mm(W4s[g * kLd + 16 * ob + c], dgk, zero);
#pragma unroll
      for (int jj = 0; jj < 4; jj++) d3[ob][jj] *= 1.f - h3[ob][jj] * h3[ob][jj];
    }
    __syncthreads();
    put(Ps, d3, 4);
    put(Qs, h2, 4);
    __syncthreads();
#pragma unroll
    for (int ib = 0; ib < 4; ib++) wgrad(gW3[ib], Ps + 16 * w * kLd, Qs + 16 * ib * kLd);
    bgrad(gb3, Ps + 16 * w * kLd);
#pragma unroll
    for (int ob = 0; ob < 4; ob++) {
      d2[ob] = dense(W3s, d3, zero, ob, true);
#pragma unroll
      for (int jj = 0; jj < 4; jj++) d2[ob][jj] *= 1.f - h2[ob][jj] * h2[ob][jj];
    }
    __syncthreads();
    put(Ps, d2, 4);
    put(Qs, h1, 4);
    __syncthreads();
#pragma unroll
    for (int ib = 0; ib < 4; ib++) wgrad(gW2[ib], Ps + 16 * w * kLd, Qs + 16 * ib * kLd);
    bgrad(gb2, Ps + 16 * w * kLd);
#pragma unroll
    for (int ob = 0; ob < 4; ob++) {
      d1[ob] = dense(W2s, d2, zero, ob, true);
#pragma unroll
      for (int jj = 0; jj < 4; jj++) d1[ob][jj] *= 1.f - h1[ob][jj] * h1[ob][jj];
    }
    __syncthreads();
    put(Ps, d1, 4);
    // the first layer's inputs [lambda, h0] (rows 21 .. 31 are not used)
#pragma unroll
    for (int jj = 0; jj < 4; jj++) Qs[(kLam + 4 * g + jj) * kLd + col] = h0[jj];
    Qs[g * kLd + col] = l0;
    if (g == 0) Qs[4 * kLd + col] = l1;
    __syncthreads();
#pragma unroll
    for (int ib = 0; ib < 2; ib++) wgrad(gW1[ib], Ps + 16 * w * kLd, Qs + 16 * ib * kLd);
    bgrad(gb1, Ps + 16 * w * kLd);
    // dZ0 = (W1^T dZ1)(h0 inputs) (1 - h0^2)
    d0 = zero;
#pragma unroll
    for (int o = 0; o < 4; o++)
#pragma unroll
      for (int jj = 0; jj < 4; jj++)
        d0 = mm(W1s[(16 * o + 4 * g + jj) * kIn1 + kLam + c], d1[o][jj], d0);
#pragma unroll
    for (int jj = 0; jj < 4; jj++) d0[jj] *= 1.f - h0[jj] * h0[jj];
    __syncthreads();
    put(Ps, &d0, 1);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 3; i++)
      if (i < 2 || w == 0) wgrad(gW0[i], Ps, X0s + 16 * (w + 4 * i) * kLd);
    bgrad(gb0, Ps);
    __syncthreads();  // X0s, Ts and taus are refilled by the next tile
  }
  // the partial sums in the layout of theta: D rows o, column i
  float* row = part + (size_t)blockIdx.x * kParams;
#pragma unroll
  for (int jj = 0; jj < 4; jj++) {
    const int o = 16 * w + 4 * g + jj;
#pragma unroll
    for (int ib = 0; ib < 4; ib++) {
      row[oW2 + o * kHid + 16 * ib + c] = gW2[ib][jj];
      row[oW3 + o * kHid + 16 * ib + c] = gW3[ib][jj];
    }
#pragma unroll
    for (int ib = 0; ib < 2; ib++)
      if (16 * ib + c < kIn1) row[oW1 + o * kIn1 + 16 * ib + c] = gW1[ib][jj];
    if (g == 0) row[oW4 + jj * kHid + 16 * w + c] = gW4[jj];
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int k = 16 * (w + 4 * i) + c;
      if ((i < 2 || w == 0) && k < kIn0) row[oW0 + (4 * g + jj) * kIn0 + k] = gW0[i][jj];
    }
  }
  auto rows = [](float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
  };
  const float s0 = rows(gb0), s1 = rows(gb1), s2 = rows(gb2), s3 = rows(gb3), s4 = rows(gb4);
  if (g == 0) {
    row[ob1 + 16 * w + c] = s1;
    row[ob2 + 16 * w + c] = s2;
    row[ob3 + 16 * w + c] = s3;
    if (w == 0) row[ob0 + c] = s0;
    if (w == 0 && c < kBasis) row[ob4 + c] = s4;
  }
  if (lane == 0) red[w] = lsum;
  __syncthreads();
  if (tid == 0) lpart[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// grad = the sum of the nrow partial rows (FP64, in a fixed order: four
// interleaved sums per parameter, then those four), and with an Adam state the
// update of theta (Kingma & Ba, Algorithm 1, the bias corrections c1 = 1/(1 -
// b1^t) and c2 = 1/(1 - b2^t) from the host).  The last work-group folds the
// loss: loss[0] = scale sum lpart.
struct Adam {
  float *th, *m, *v;
  float lr, b1, b2, eps, c1, c2;
};
__global__ void __launch_bounds__(256)
    k_train_fold(const float* __restrict__ part, int nrow, const double* __restrict__ lpart, double scale,
                 float* __restrict__ grad, double* __restrict__ loss, Adam ad) {
  __shared__ double red[256];
  const int tid = threadIdx.x;
  if (blockIdx.x == gridDim.x - 1) {
    double l = 0.0;
    for (int i = tid; i < nrow; i += 256) l += lpart[i];
    red[tid] = l;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
      if (tid < h) red[tid] += red[tid + h];
      __syncthreads();
    }
    if (tid == 0) loss[0] = red[0] * scale;
    return;
  }
  const int p = blockIdx.x * 64 + (tid & 63), q = tid >> 6;
  double s = 0.0;
  if (p < kParams) {
#pragma unroll 8
    for (int r = q; r < nrow; r += 4) s += (double)part[(size_t)r * kParams + p];
  }
  red[tid] = s;
  __syncthreads();
  if (q != 0 || p >= kParams) return;
  const float gi = (float)((red[tid] + red[tid + 64]) + (red[tid + 128] + red[tid + 192]));
  grad[p] = gi;
  if (ad.th) {
    const float mi = ad.b1 * ad.m[p] + (1.f - ad.b1) * gi;
    const float vi = ad.b2 * ad.v[p] + (1.f - ad.b2) * gi * gi;
    ad.m[p] = mi;
    ad.v[p] = vi;
    ad.th[p] -= ad.lr * (mi * ad.c1) / (sqrtf(vi * ad.c2) + ad.eps);
  }
}

// ---------------------------------------------------------------------------
// Inference in one kernel, k_closure<BF16>: the 3x3x3 convolution of the
// invariant field and the dense layers on the matrix cores, and the stress
// tau = sum_n g_n T_n; only lambda and T are read and tau written.
//
// A work-group (8 waves) takes blocks of 32 x 4 x 4 points: the block's
// lambda with a halo of one goes to LDS (5 channels of 6 x 6 rows of 34, row
// stride 36), a wave takes its 16 consecutive points along x per tile.  All layers
// are computed transposed, Y^T[O][16 points] = W X^T: lane l (r or c = l % 16,
// g = l / 16) supplies A = W and B = X for its K slots and receives D[4 g +
// jj][c], the outputs o = 16 ob + 4 g + jj of its own point c.
//
// The convolution runs on v_mfma_f32_16x16x4_f32 (FP32 operands and sums), K =
// 135 in 34 steps: steps 0 .. 26 are the taps of channels 0 .. 3 (slot g =
// channel g, so a tap's LDS reads differ by a lane constant and hit all 64
// banks once), steps 27 .. 33 four taps each of channel 4.  The slot past its
// last tap is zero in both operands, as are the empty slots of layer 1: zero
// times an infinite value would be a NaN that the point does not have.  On the
// VALU, a point per thread with its 135 neighbours from the cache, the
// convolution took 178 us at 128^3 (116 us at the full FP32 rate; packed FP32 is
// off), and an earlier matrix form with gathered global reads and a fourth of
// its slots empty 207.
//
// The dense layers, BF16: v_mfma_f32_16x16x32_bf16 (bf16 operands, FP32
// accumulation), eight K slots (g, j) per lane and step; else
// v_mfma_f32_16x16x4_f32.  The K order inside a product is free as long as A
// and B use the same one: with k = 16 (2 s + j / 4) + 4 g + j % 4 (BF16) or k =
// 16 ob + 4 g + jj (FP32) the accumulators of a layer are the next layer's
// operand B, so the activations stay in the lane's registers from layer to
// layer (no LDS tile, no cross-lane exchange).  The weights are in LDS, for
// BF16 as operand-A blocks in that order; the biases are the accumulators'
// initial values.  The sums and biases are FP32; the activations are tanhf, but
// for those of the dense layers with BF16 (tanh_fast).
//
// What bounds it, BF16 at 128^3: issue. Per 16 points 1,440 cycles of matrix
// instructions and about 3,000 of VALU (52 tanh per lane, 48 of them two
// quarter-rate instructions each), 236 us on end where nothing overlaps; 258 us
// per call (240 with the fast form for the convolution's four tanh too, which is
// not exact enough there), against 178 us for the convolution with its 16
// channels stored and 189 us for the dense layers that read them back.  64^3: 39
// us (75), with FP32 layers 87 us (179).  Before the weights were loaded with all
// loads in flight and their LDS addresses formed once per tile: 270 us (209
// without the tanh, 218 without the convolution's products) and 46 us; two tiles
// per wave, sharing each weight read, came to 262-360 us for 2 to 4 waves per SIMD.
// ---------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kCWaves = 8;                          // waves per work-group
constexpr int kBx = 32, kBy = 4, kBz = 4;           // points of a block
constexpr int kHs = kBx + 4;                        // halo row stride
constexpr int kHrows = (kBy + 2) * (kBz + 2);       // halo rows of a channel
constexpr int kHch = kHrows * kHs;                  // channel stride (16 banks apart)
static_assert(kHch % 64 == 16, "the four channels of a step on different banks");
// offset of tap (dy, dz, dx) = (tap / 9, tap / 3 % 3, tap % 3) - 1 from that of tap 0
__device__ __forceinline__ constexpr int tap_off(int tap) {
  return (tap / 9 * (kBz + 2) + tap / 3 % 3) * kHs + tap % 3;
}

// an opaque copy of the lane index: addresses formed from it are recomputed
// where they are used
__device__ __forceinline__ int opaque_lane(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// input k of K step s and slot (g, j) of a layer fed by a 64-wide layer
__device__ __forceinline__ constexpr int slot_k(int s, int g, int j) { return 16 * (2 * s + j / 4) + 4 * g + j % 4; }

// layer 1's input of K slot (g, j): the lane's own h0 channels, lambda_g, and
// lambda_4 in the lane group that reads it for the convolution (-1: none)
__device__ __forceinline__ constexpr int in_k(int g, int j) {
  return j < 4 ? kLam + 4 * g + j : (j == 4 ? g : (j == 5 && g == 1 ? 4 : -1));
}

// operand-A blocks in LDS, 64 lanes x 16 bytes each: W1 ob 0..3, W2 (s, ob)
// 4..11, W3 (s, ob) 12..19, W4 s 20..21 (rows 0..3 of 16)
constexpr int kOpBlocks = 22;
// (no branch, so that the loads of several blocks can be in flight)
__device__ __forceinline__ bf16x8 a_block(const float* __restrict__ theta, int blk, int lane) {
  const int r = lane & 15, g = lane >> 4;
  const bool first = blk < 4, out = blk >= 20;
  const int s = out ? blk - 20 : ((blk - 4) % 8) / 4;
  const int o = first ? 16 * blk + r : (out ? min(r, kBasis - 1) : 16 * ((blk - 4) % 4) + r);
  const int row = first ? oW1 + o * kIn1 : (out ? oW4 : blk < 12 ? oW2 : oW3) + o * kHid;
  float w[8];
#pragma unroll
  for (int j = 0; j < 8; j++) w[j] = theta[row + (first ? max(in_k(g, j), 0) : slot_k(s, g, j))];
  bf16x8 v;
#pragma unroll
  for (int j = 0; j < 8; j++) v[j] = (__bf16)((first && in_k(g, j) < 0) || (out && r >= kBasis) ? 0.f : w[j]);
  return v;
}
// accumulator initial values: bias of outputs 16 ob + 4 g + jj (layer 0..2
// the hidden layers, ob < 4; layer 3 the output, only g = 0 valid)
__device__ __forceinline__ f32x4 bias_block(const float* __restrict__ theta, int layer, int ob, int g) {
  f32x4 b;
#pragma unroll
  for (int jj = 0; jj < 4; jj++) {
    const int o = 16 * ob + 4 * g + jj;
    b[jj] = layer == 0 ? theta[ob1 + o] : layer == 1 ? theta[ob2 + o] : layer == 2 ? theta[ob3 + o]
                                                                              : (o < kBasis ? theta[ob4 + o] : 0.f);
  }
  return b;
}

// tanh(x) = 1 - 2 / (exp(2 x) + 1) with the hardware exponential and
// reciprocal, v_exp_f32 and v_rcp_f32; saturates to +-1 for large |x|.  Its error
// is absolute, about 1e-7 whatever the size of the result: next to the 4e-3
// relative rounding of the bf16 operands of which a dense layer sums 64, of
// order one, but not for the activations of the convolution, which may be small
// throughout.  A division here (even __fdividef) compiles to the full IEEE
// sequence, several times the cost of the rest of the activation.
__device__ __forceinline__ float tanh_fast(float x) {
  // exp(2 x) as v_exp_f32 (2^v) of 2 x log2(e)
  return fmaf(-2.f, __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(2.8853900817779268f * x) + 1.f), 1.f);
}
// operand B of K step s of the next layer: tanh of accumulator blocks 2 s
// and 2 s + 1 of this lane
__device__ __forceinline__ bf16x8 act_operand(f32x4 d0, f32x4 d1) {
  bf16x8 r;
#pragma unroll
  for (int jj = 0; jj < 4; jj++) {
    r[jj] = (__bf16)tanh_fast(d0[jj]);
    r[4 + jj] = (__bf16)tanh_fast(d1[jj]);
  }
  return r;
}

// the dense layers' weights in LDS
template <bool BF16>
struct DenseWeights;
template <>
struct DenseWeights<true> {
  bf16x8 op[kOpBlocks][64];
  template <int NT>
  __device__ __forceinline__ void fill(const float* __restrict__ theta, int tid) {
    constexpr int n = (kOpBlocks * 64 + NT - 1) / NT;
    bf16x8 v[n];
#pragma unroll
    for (int i = 0; i < n; i++) v[i] = a_block(theta, min((tid + NT * i) / 64, kOpBlocks - 1), tid % 64);
#pragma unroll
    for (int i = 0; i < n; i++)
      if (tid + NT * i < kOpBlocks * 64) op[(tid + NT * i) / 64][tid % 64] = v[i];
  }
};
template <>
struct DenseWeights<false> {
  __attribute__((aligned(16))) float W2[kHid * kLd], W3[kHid * kLd], W4[kBasis * kLd];
  float W1[kHid * kIn1];
  template <int NT>
  __device__ __forceinline__ void fill(const float* __restrict__ theta, int tid) {
    constexpr int n1 = (kHid * kIn1 + NT - 1) / NT, n2 = kHid * kHid / 4 / NT;
    static_assert(kHid * kHid % (4 * NT) == 0 && kBasis * kHid <= NT, "whole rounds");
    f32x4 w2[n2], w3[n2];
    float w1[n1];
#pragma unroll
    for (int i = 0; i < n2; i++) {
      w2[i] = *(const f32x4*)(theta + oW2 + 4 * (tid + NT * i));
      w3[i] = *(const f32x4*)(theta + oW3 + 4 * (tid + NT * i));
    }
#pragma unroll
    for (int i = 0; i < n1; i++) w1[i] = theta[oW1 + min(tid + NT * i, kHid * kIn1 - 1)];
    if (tid < kBasis * kHid) W4[tid / kHid * kLd + tid % kHid] = theta[oW4 + tid];
#pragma unroll
    for (int i = 0; i < n2; i++) {
      const int e = 4 * (tid + NT * i), o = e / kHid * kLd + e % kHid;
      *(f32x4*)(W2 + o) = w2[i];
      *(f32x4*)(W3 + o) = w3[i];
    }
#pragma unroll
    for (int i = 0; i < n1; i++)
      if (tid + NT * i < kHid * kIn1) W1[tid + NT * i] = w1[i];
  }
};

template <bool BF16>
__global__ void __launch_bounds__(64 * kCWaves) __attribute__((amdgpu_waves_per_eu(4, 4)))
    k_closure(const float* __restrict__ lam, const float* __restrict__ T, int n, const float* __restrict__ theta,
              float* __restrict__ tau) {
  __shared__ __attribute__((aligned(16))) DenseWeights<BF16> wt;
  __shared__ f32x4 bias[13][4];  // [3 layers x 4 ob + the output layer][g]
  __shared__ float halo[kLam * kHch];
  constexpr int NT = 64 * kCWaves;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
  // this lane's convolution weights (row c) and bias (rows 4 g + jj)
  constexpr int kSteps = 34;
  float wc[kSteps];
#pragma unroll
  for (int s = 0; s < kSteps; s++) {
    const int k = s < kTaps ? g * kTaps + s : 4 * (s - kTaps) + g;
    wc[s] = s < kTaps ? theta[oW0 + c * kIn0 + k] : (k < kTaps ? theta[oW0 + c * kIn0 + 4 * kTaps + k] : 0.f);
  }
  f32x4 b0;
#pragma unroll
  for (int jj = 0; jj < 4; jj++) b0[jj] = theta[ob0 + 4 * g + jj];
  // channel 4's tap offsets of this lane group (the slot past the last tap has
  // weight zero and reads the last tap)
  int off4[kSteps - kTaps];
#pragma unroll
  for (int q = 0; q < kSteps - kTaps; q++) off4[q] = 4 * kHch + tap_off(min(4 * q + g, kTaps - 1));

  const size_t P = (size_t)n * n * n;
  const int m = n - 1, nbx = n / kBx, nbz = n / kBz, nblk = nbx * nbz * (n / kBy);
  // The next block's halo is on its way into registers while this one's points
  // run through the layers (indices formed per block, not held across it).
  constexpr int W = kBx + 2, kTot = kLam * kHrows * W, kPer = (kTot + NT - 1) / NT;
  float hv[kPer];
  auto load_halo = [&](int blk) {
    const int x0 = blk % nbx * kBx, z0 = blk / nbx % nbz * kBz, y0 = blk / (nbx * nbz) * kBy, t0 = opaque_lane(tid);
#pragma unroll
    for (int i0 = 0; i0 < kPer; i0++) {
      const int i = min(t0 + i0 * NT, kTot - 1), row = i / W, xx = i % W, ch = row / kHrows, rr = row % kHrows;
      const int y = (y0 + rr / (kBz + 2) - 1) & m, z = (z0 + rr % (kBz + 2) - 1) & m;
      hv[i0] = lam[ch * P + ((size_t)y * n + z) * n + ((x0 + xx - 1) & m)];
    }
  };
  auto store_halo = [&]() {
    const int t0 = opaque_lane(tid);
#pragma unroll
    for (int i0 = 0; i0 < kPer; i0++) {
      const int i = t0 + i0 * NT, row = i / W, ch = row / kHrows, rr = row % kHrows;
      if (i < kTot) halo[ch * kHch + rr * kHs + i % W] = hv[i0];
    }
  };
  // blocks of an XCD are one contiguous range (their halos share an L2)
  const int x8 = blockIdx.x % 8, per = gridDim.x / 8, q8 = nblk / 8, end = (x8 + 1) * q8;
  int blk = x8 * q8 + blockIdx.x / 8;
  if (blk < end) load_halo(blk);
  wt.template fill<NT>(theta, tid);
  if (tid < 13 * 4) {
    const int b = tid / 4;
    bias[b][tid % 4] = b < 12 ? bias_block(theta, b / 4, b % 4, tid % 4) : bias_block(theta, 3, 0, tid % 4);
  }
  for (; blk < end; blk += per) {
    const int x0 = blk % nbx * kBx, z0 = blk / nbx % nbz * kBz, y0 = blk / (nbx * nbz) * kBy;
    __syncthreads();  // the last block's halo is read
    store_halo();
    __syncthreads();  // (and the weights are there)
    if (blk + per < end) load_halo(blk + per);
#pragma unroll 1
    for (int ty = 0; ty < kBy; ty++) {
      const int tz = wave >> 1, tx = 16 * (wave & 1);
      const size_t p = ((size_t)(y0 + ty) * n + z0 + tz) * n + x0 + tx + c;
      // the basis of the stress lanes (lane < 48: point c, components 2 g + cc),
      // in flight during the layers (from one address per tile: eight of them
      // held across the loop would spill)
      const size_t gp = (size_t)(2 * opaque_lane(g)) * P + p;
      float tb[8];
      if (lane < 48) {
        const float* tp = T + gp;
#pragma unroll
        for (int cc = 0; cc < 2; cc++)
#pragma unroll
          for (int k = 0; k < kBasis; k++) tb[4 * cc + k] = tp[(k * 6 + cc) * P];
      }
      // convolution
      const float* hp = halo + (ty * (kBz + 2) + tz) * kHs + tx + c;
      f32x4 ca = b0, cb = {0.f, 0.f, 0.f, 0.f};
      float lg = 0.f, l4 = 0.f;  // lambda_g, and lambda_4 in group 1
      static_for<kSteps>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        float v;
        if constexpr (s < kTaps) v = hp[g * kHch + tap_off(s)];
        else v = hp[off4[s - kTaps]];
        if constexpr (s == kSteps - 1) v = g == 3 ? 0.f : v;  // past the last tap
        if constexpr (s == 13) lg = v;
        if constexpr (s == kTaps + 3) l4 = g == 1 ? v : 0.f;
        f32x4& acc = s % 2 ? cb : ca;
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[s], v, acc, 0, 0, 0);
        // (the layers' weights not ahead of the convolution: registers)
        if constexpr (s == kSteps - 1) __builtin_amdgcn_sched_barrier(0);
      });
      f32x4 h0;
      f32x4 gc;  // rows 0..3 (lanes 0..15): the basis coefficients of point c
      // weights and biases are read per tile, through a lane index the compiler
      // cannot hoist their reads with
      const int ln = opaque_lane(lane), lg4 = ln >> 4;
      auto bc = [&](int b) { return bias[b][lg4]; };
      if constexpr (BF16) {
#pragma unroll
        for (int jj = 0; jj < 4; jj++) h0[jj] = tanhf(ca[jj] + cb[jj]);
        auto wa = [&](int b) { return wt.op[b][ln]; };
        const bf16x8 x = {(__bf16)h0[0], (__bf16)h0[1], (__bf16)h0[2], (__bf16)h0[3],
                          (__bf16)lg,    (__bf16)l4,    (__bf16)0.f,   (__bf16)0.f};
        f32x4 d[4];
#pragma unroll
        for (int ob = 0; ob < 4; ob++) d[ob] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa(ob), x, bc(ob), 0, 0, 0);
#pragma unroll
        for (int layer = 1; layer < 3; layer++) {
          const bf16x8 v0 = act_operand(d[0], d[1]), v1 = act_operand(d[2], d[3]);
#pragma unroll
          for (int ob = 0; ob < 4; ob++) {
            const int b = 4 + 8 * (layer - 1) + ob;
            const f32x4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa(b), v0, bc(4 * layer + ob), 0, 0, 0);
            d[ob] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa(b + 4), v1, acc, 0, 0, 0);
          }
        }
        const bf16x8 v0 = act_operand(d[0], d[1]), v1 = act_operand(d[2], d[3]);
        gc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa(20), v0, bc(12), 0, 0, 0);
        gc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa(21), v1, gc, 0, 0, 0);
      } else {
        auto mm = [](float a, float b, f32x4 d) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, d, 0, 0, 0); };
#pragma unroll
        for (int jj = 0; jj < 4; jj++) h0[jj] = tanhf(ca[jj] + cb[jj]);
        f32x4 h[4], d[4];
#pragma unroll
        for (int ob = 0; ob < 4; ob++) {
          const float* wr = wt.W1 + (16 * ob + c) * kIn1;
          d[ob] = mm(wr[g], lg, bc(ob));
          d[ob] = mm(g == 1 ? wr[4] : 0.f, l4, d[ob]);
#pragma unroll
          for (int jj = 0; jj < 4; jj++) d[ob] = mm(wr[kLam + 4 * g + jj], h0[jj], d[ob]);
        }
#pragma unroll
        for (int layer = 1; layer < 3; layer++) {
          const float* W = layer == 1 ? wt.W2 : wt.W3;
#pragma unroll
          for (int ob = 0; ob < 4; ob++) {
#pragma unroll
            for (int jj = 0; jj < 4; jj++) h[ob][jj] = tanhf(d[ob][jj]);
          }
#pragma unroll
          for (int ob = 0; ob < 4; ob++) {
            d[ob] = bc(4 * layer + ob);
#pragma unroll
            for (int o = 0; o < 4; o++) {
              const f32x4 a = *(const f32x4*)(W + (16 * ob + c) * kLd + 16 * o + 4 * g);
#pragma unroll
              for (int jj = 0; jj < 4; jj++) d[ob] = mm(a[jj], h[o][jj], d[ob]);
            }
          }
        }
        gc = bc(12);
#pragma unroll
        for (int o = 0; o < 4; o++) {
          const f32x4 a = *(const f32x4*)(wt.W4 + (c & 3) * kLd + 16 * o + 4 * g);
#pragma unroll
          for (int jj = 0; jj < 4; jj++) gc = mm(a[jj], tanhf(d[o][jj]), gc);
        }
      }
      // the stress: lanes < 48 take the coefficients of their point from lane c
      float gk[kBasis];
#pragma unroll
      for (int k = 0; k < kBasis; k++) gk[k] = __shfl(gc[k], c);
      if (lane < 48) {
#pragma unroll
        for (int cc = 0; cc < 2; cc++) {
          float sacc = 0.f;
#pragma unroll
          for (int k = 0; k < kBasis; k++) sacc = fmaf(gk[k], tb[4 * cc + k], sacc);
          tau[gp + cc * P] = sacc;
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// LES: the predicted stress added to the realspace_vel products (ux slots
// 0..4: u^2 - v^2, uv, w^2 - v^2, vw, uw), i.e. u_i u_j -> u_i u_j + tau_ij
// in the flux whose divergence transform() and wavespace_vel() form.
// ---------------------------------------------------------------------------
template <typename R>
__global__ void __launch_bounds__(256) k_add_stress(R* __restrict__ ux, const float* __restrict__ tau, size_t P) {
  for (size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x; p < P; p += (size_t)gridDim.x * blockDim.x) {
    const float t11 = tau[p], t12 = tau[P + p], t13 = tau[2 * P + p], t22 = tau[3 * P + p], t23 = tau[4 * P + p],
                t33 = tau[5 * P + p];
    ux[p] += (R)(t11 - t22);
    ux[P + p] += (R)t12;
    ux[2 * P + p] += (R)(t33 - t22);
    ux[3 * P + p] += (R)t23;
    ux[4 * P + p] += (R)t13;
  }
}

// squared-error sum of predicted vs target stress (loss numerator over all
// points) in fixed-order partial sums
__global__ void __launch_bounds__(256)
    k_field_err(const float* __restrict__ tp, const float* __restrict__ tt, size_t P, double* __restrict__ part) {
  __shared__ double red[256];
  double l = 0.0;
  for (size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x; p < P; p += (size_t)gridDim.x * blockDim.x) {
#pragma unroll
    for (int c = 0; c < 6; c++) {
      const double e = (double)tp[c * P + p] - (double)tt[c * P + p];
      l += (double)kCw[c] * e * e;
    }
  }
  red[threadIdx.x] = l;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// Frobenius norm^2 of stored targets in fixed-order partial sums
__global__ void __launch_bounds__(256) k_target_norm(const float* __restrict__ tau_s, size_t P, int nsnap,
                                                     double* __restrict__ part) {
  __shared__ double red[256];
  double l = 0.0;
  const size_t tot = (size_t)nsnap * P;
  for (size_t g = blockIdx.x * (size_t)blockDim.x + threadIdx.x; g < tot; g += (size_t)gridDim.x * blockDim.x) {
    const size_t s = g / P, p = g % P;
#pragma unroll
    for (int c = 0; c < 6; c++) {
      const double v = (double)tau_s[(s * 6 + c) * P + p];
      l += (double)kCw[c] * v * v;
    }
  }
  red[threadIdx.x] = l;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static unsigned blocks(size_t work, size_t per = 256, size_t cap = 65536) {
  size_t b = (work + per - 1) / per;
  if (b > cap) b = cap;
  return (unsigned)(b ? b : 1);
}

template <typename R>
static int box_filter_r(hipStream_t st, const R* u, int n, int r, R* ubar, float* tau) {
  const int nc = n / r;
  const dim3 grid(nc * nc), block(256);
  switch (r) {
    case 2: hipLaunchKernelGGL((k_box_filter<R, 2>), grid, block, 0, st, u, n, ubar, tau, nc); return 0;
    case 4: hipLaunchKernelGGL((k_box_filter<R, 4>), grid, block, 0, st, u, n, ubar, tau, nc); return 0;
    case 8: hipLaunchKernelGGL((k_box_filter<R, 8>), grid, block, 0, st, u, n, ubar, tau, nc); return 0;
    case 16: hipLaunchKernelGGL((k_box_filter<R, 16>), grid, block, 0, st, u, n, ubar, tau, nc); return 0;
    case 32: hipLaunchKernelGGL((k_box_filter<R, 32>), grid, block, 0, st, u, n, ubar, tau, nc); return 0;
  }
  return -1;
}
int launch_box_filter(hipStream_t st, int prec, const void* u, int n, int r, void* ubar, float* tau) {
  return prec == 8 ? box_filter_r(st, (const double*)u, n, r, (double*)ubar, tau)
                   : box_filter_r(st, (const float*)u, n, r, (float*)ubar, tau);
}

void launch_invariants(hipStream_t st, int prec, const void* A, size_t P, double delta2, float* lam, float* T) {
  if (prec == 8)
    hipLaunchKernelGGL(k_invariants<double>, dim3(blocks(P)), dim3(256), 0, st, (const double*)A, P, delta2, lam, T);
  else
    hipLaunchKernelGGL(k_invariants<float>, dim3(blocks(P)), dim3(256), 0, st, (const float*)A, P, delta2, lam, T);
}

template <bool BF16>
static void closure(hipStream_t st, const float* lam, const float* T, int n, const float* theta, float* tau) {
  // as many work-groups as are resident (each fills the weights once and walks
  // its blocks), at most one per block; n >= 32, so both are multiples of 8
  static const unsigned resident = [] {
    int dev = 0, cus = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void*)k_closure<BF16>, 64 * kCWaves, 0) !=
            hipSuccess ||
        per < 1)
      per = 1;
    return (unsigned)((cus > 8 ? cus : 256) * per) / 8 * 8;
  }();
  const unsigned want = (unsigned)((size_t)n * n * n / (kBx * kBy * kBz));
  hipLaunchKernelGGL(k_closure<BF16>, dim3(want < resident ? want : resident), dim3(64 * kCWaves), 0, st, lam, T, n,
                     theta, tau);
}
void launch_predict(hipStream_t st, bool bf16, const float* lam, const float* T, int n, const float* theta,
                    float* tau) {
  if (bf16) closure<true>(st, lam, T, n, theta, tau);
  else closure<false>(st, lam, T, n, theta, tau);
}

void launch_add_stress(hipStream_t st, int prec, void* ux, const float* tau, size_t P) {
  if (prec == 8)
    hipLaunchKernelGGL(k_add_stress<double>, dim3(blocks(P)), dim3(256), 0, st, (double*)ux, tau, P);
  else
    hipLaunchKernelGGL(k_add_stress<float>, dim3(blocks(P)), dim3(256), 0, st, (float*)ux, tau, P);
}

int field_err_blocks() { return 1024; }
void launch_field_err(hipStream_t st, const float* tp, const float* tt, size_t P, double* part) {
  hipLaunchKernelGGL(k_field_err, dim3(1024), dim3(256), 0, st, tp, tt, P, part);
}
void launch_target_norm(hipStream_t st, const float* tau_s, size_t P, int nsnap, double* part) {
  hipLaunchKernelGGL(k_target_norm, dim3(1024), dim3(256), 0, st, tau_s, P, nsnap, part);
}

// One minibatch: the partial rows (train_rows(B) of kParams floats) into part
// and the loss partial sums into lpart, then their fold into grad and loss
// (scale: of the loss), and with t > 0 Adam step t of learning rate lr on
// theta and its moments.
void launch_train_batch(hipStream_t st, float* theta, const float* lam_s, const float* T_s, const float* tau_s, int n,
                        int nsnap, uint64_t base, int B, float inv, float* part, double* lpart, double scale,
                        float* grad, double* loss, float* m, float* v, float lr, long long t) {
  const int rows = train_rows(B);
  hipLaunchKernelGGL(k_train, dim3(rows), dim3(256), 0, st, lam_s, T_s, tau_s, n, nsnap, base, B, inv, theta, part,
                     lpart);
  Adam ad = {nullptr, nullptr, nullptr, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (t > 0)
    ad = {theta, m, v, lr, 0.9f, 0.999f, 1e-8f, (float)(1.0 / (1.0 - std::pow(0.9, (double)t))),
          (float)(1.0 / (1.0 - std::pow(0.999, (double)t)))};
  hipLaunchKernelGGL(k_train_fold, dim3((kParams + 63) / 64 + 1), dim3(256), 0, st, part, rows, lpart, scale, grad,
                     loss, ad);
}

}  // namespace sgs
}  // namespace psdns

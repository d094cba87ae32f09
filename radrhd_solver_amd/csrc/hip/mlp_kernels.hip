// Training and evaluation kernels of the c2p surrogate MLP (see mlp.h).
//
// Training step (captured several to a hipGraph and replayed):
//   k_mlp_grad   one workgroup per 64 samples: forward (BF16 MFMA with K = 32,
//                FP32 accumulate),
//                backward, gradient partials written to global memory;
//   k_mlp_adam   fixed-order sum of the partials (deterministic), Adam on the
//                FP32 master weights, BF16 copies of W2 and W2^T, the step's
//                loss and the device step counter; and on the CUs that the sum
//                leaves idle the next step's samples: seeded primitives -> FP64
//                p2c -> FP64 c2p (reference start) -> normalised features and
//                targets (failed states are masked).
// k_mlp_gen makes the samples of the normalisation and of the first step.
#include <hip/hip_runtime.h>

#include "mlp.h"
#include "mlp_internal.h"
#include "rhllc_physics.h"

namespace rhllc_mlp {

using rhllc_dev::Ieee;
using rhllc_dev::State;

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__device__ __forceinline__ double u01(uint64_t r) { return (double)(r >> 11) * (1.0 / 9007199254740992.0); }

// Primitive sample k of the training distribution (log-uniform rho in
// [1e-4, 1e2], p/rho in [1e-6, 1e2], Lorentz factor in [1, 50], isotropic v).
__device__ void sample_state(uint64_t seed, uint64_t k, State<double> &W) {
  const uint64_t b = mix64(seed) ^ (k * 0x9E3779B97F4A7C15ull);
  const double rho = exp(2.302585092994046 * (-4.0 + 6.0 * u01(mix64(b + 1))));
  const double pr = exp(2.302585092994046 * (-6.0 + 8.0 * u01(mix64(b + 2))));
  const double lor = exp(3.912023005428146 * u01(mix64(b + 3)));  // ln 50
  const double v = sqrt(1.0 - 1.0 / (lor * lor));
  const double z = 2.0 * u01(mix64(b + 4)) - 1.0;
  const double ph = 6.283185307179586 * u01(mix64(b + 5));
  const double s = sqrt(fmax(0.0, 1.0 - z * z));
  W.d = rho;
  W.v[0] = v * s * cos(ph), W.v[1] = v * s * sin(ph), W.v[2] = v * z;
  W.p = rho * pr;
}

// Raw (un-normalised) features and target of sample k; ok = 0 when c2p fails.
__device__ void make_sample(double gamma, uint64_t seed, uint64_t k, float x[3], float &y, int &ok) {
  State<double> W, U, Wc;
  sample_state(seed, k, W);
  const double Gg = gamma / (gamma - 1.0);
  rhllc_dev::p2c<double, Ieee>(Gg, W, U);
  int it = 0;
  // The states of the box are ordinary unless gamma is extreme; the same bits
  // either way (k_mlp_adam, which waits for these, 12.0 -> 11.8 us).
  const int code = rhllc_dev::ordinary(U) ? rhllc_dev::c2p<rhllc_dev::IeeeOrd>(Gg, U, Wc, -1.0, it)
                                          : rhllc_dev::c2p<Ieee>(Gg, U, Wc, -1.0, it);
  const double m = sqrt(rhllc_dev::dot3(U.v, U.v));
  double p0;
  raw_features(Gg, U.d, m, U.p, x, p0);
  ok = code == 0 && Wc.p > 0.0 && p0 > 0.0 && isfinite(x[0] + x[1] + x[2]);
  y = ok ? (float)log(Wc.p / p0) : 0.0f;
  if (!ok) x[0] = x[1] = x[2] = 0.0f;
}

// Entry i of a batch: sample k of the stream, normalised unless norm is null.
__device__ void put_sample(double gamma, uint64_t seed, uint64_t k, int i, const float *norm, float *X, float *Y,
                           float *OK) {
  float x[3], y;
  int ok;
  make_sample(gamma, seed, k, x, y, ok);
  if (norm) {
    for (int f = 0; f < 3; ++f) x[f] = (x[f] - norm[f]) / norm[3 + f];
    y = (y - norm[6]) / norm[7];
  }
  X[3 * i] = x[0], X[3 * i + 1] = x[1], X[3 * i + 2] = x[2];
  Y[i] = ok ? y : 0.0f;
  OK[i] = ok ? 1.0f : 0.0f;
}

__global__ void k_mlp_gen(double gamma, uint64_t seed, int n, const float *norm, float *X, float *Y, float *OK) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) put_sample(gamma, seed, (uint64_t)i, i, norm, X, Y, OK);
}

// v plus v of the lane across bit 0, 1, 2 or 3 of the lane number, the sum of
// 16 lanes in the order of a butterfly of lane exchanges: each level adds two
// values that all lanes of their halves hold alike, so a mirrored lane serves
// as well as the exchanged one.  One VALU instruction a level (DPP); the
// exchange through LDS that __shfl_xor makes costs a round trip each.
template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float sum16(float v) {
  v = dpp_add<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  v = dpp_add<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  v = dpp_add<0x141>(v);  // row_half_mirror
  return dpp_add<0x140>(v);  // row_mirror
}

// The operand of a product that contracts over the samples, from the block of
// 16 samples x 16 units that f holds as the lanes made it (lane (g, c): units
// 4 g + e of sample c): lane (g, c) gets unit c of the samples 4 g + e.  The
// transposing read hands lane i of each 16 the element i % 4 of the lanes
// i / 4, i / 4 + 4, .. of the 16, so lane (g, c) names the entry (c % 4, 4 g + c / 4);
// the 64 lanes read all 512 bytes once.
__device__ __forceinline__ bf16x4 read_transposed(bf16x4 *f, int g, int c) {
  typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_bf16x4 *)(f + 16 * (c & 3) + 4 * g + (c >> 2)));
}

// One workgroup = 64 consecutive samples ("wave" of the partials: a single wave
// once took them).  grad[wave][kGradStride] receives their gradient of
// sum_s ok_s (out_s - y_s)^2 * inv_n; loss[wave] the sum of squared errors.
//
// The four waves share the hidden units: wave w has the units of block w
// (16 w .. 16 w + 15) of both layers, and lane (g, c) of it the units
// 16 w + 4 g + e of the samples 16 t + c.  The operands of the products that
// contract over all units go through LDS as they are, and dW2's, which
// contracts over the samples, are read from there transposed; the output's
// sum over the units is taken in unit order from the waves' terms, so every
// value is rounded as one wave taking all the units would.  A batch of 65,536
// is then four waves a SIMD where it was one, waiting for its own chain; each
// activation's derivative is formed with it from one sigmoid, the sums over 16
// lanes use DPP and the vectors come in 16-byte loads.  Values used late are
// loaded late, which leaves registers for four workgroups a CU: all 1,024 of
// such a batch run at once.  dW2's partials, 16.8 MB of it, are stored past L2:
// the sum reads them on other XCDs, and the kernel's end would wait for them to
// be written back.  Measured at 65,536 samples: 38.2 us as one wave with spilled
// registers, 25.2 as one wave without, 18.4 as four waves with three workgroups
// a CU and operands transposed by 2-byte LDS writes, 17.6 without those, 14.0
// with the streaming stores (11.4 with no stores of dW2 at all).
//
// PACKED: W2 and its transpose come as the BF16 copies that training keeps,
// else they are rounded here from P (a call of its own would first need a
// launch that makes the copies: 3.3 us and a gap).
template <bool PACKED>
__global__ __launch_bounds__(256, 4) void k_mlp_grad(const float *__restrict__ P, const short *__restrict__ W2b,
                                                     const short *__restrict__ W2Tb, const float *__restrict__ X,
                                                     const float *__restrict__ Y, const float *__restrict__ OK,
                                                     float inv_n, float *__restrict__ grad, float *__restrict__ loss,
                                                     uint32_t *step) {
  if (step && blockIdx.x == 0 && threadIdx.x == 0) step[1] = step[0];
  __shared__ bf16x4 h1s[4][4][64], dzs[4][4][64];  // [block][t][lane]: H1 and dZ2
  __shared__ f32x4 part0[64], term[3][4][64];  // block 0's sum and the others' terms [r][lane] of the 4 samples
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = l >> 4, c = l & 15;
  const int base = blockIdx.x * 64;
  const int h0 = 16 * w + 4 * g;  // this lane's units of both layers
  // the 4 samples s_t = 16 t + c this lane works on
  float x[4][3];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int f = 0; f < 3; ++f) x[t][f] = X[3 * (base + 16 * t + c) + f];
  float w1[12];
#pragma unroll
  for (int k = 0; k < 3; ++k) *reinterpret_cast<f32x4u *>(w1 + 4 * k) = ld4(P + kOffW1 + 3 * h0 + 4 * k);
  const f32x4u b1 = ld4(P + kOffB1 + h0), b2 = ld4(P + kOffB2 + h0), w3 = ld4(P + kOffW3 + h0);
  bf16x4 a2w[4];  // rows of W2
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if constexpr (PACKED) {
      a2w[q] = *reinterpret_cast<const bf16x4 *>(W2b + (16 * w + c) * kH + 16 * q + 4 * g);
    } else {
      const f32x4u row = ld4(P + kOffW2 + (16 * w + c) * kH + 16 * q + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) a2w[q][e] = f2bf(row[e]);
    }
  }
  // ---- layer 1
  float d1[4][4];  // [t][e] dsilu
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f32x4 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float z = ((w1[3 * e] * x[t][0] + w1[3 * e + 1] * x[t][1]) + w1[3 * e + 2] * x[t][2]) + b1[e];
      const float s = sigmoid(z);
      d1[t][e] = s * (1.0f + z * (1.0f - s));
      h[e] = z * s;
    }
    h1s[w][t][l] = f2bf4(h);
  }
  __syncthreads();
  // The sample, its target and W2^T's rows are loaded (again) where they are
  // used: through pointers the compiler cannot tell to be the ones above, else
  // it would hold the values in registers.
  asm volatile("" : "+s"(X), "+s"(Y), "+s"(OK), "+s"(W2Tb));
  // ---- layer 2
  float a2[4][4], d2[4][4];  // [t][r] silu and dsilu
  f32x4 tr[4];               // [r] the terms of the 4 samples' outputs
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 4; q += 2) acc = mfma32(a2w[q], a2w[q + 1], h1s[q][t][l], h1s[q + 1][t][l], acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float z = acc[r] + b2[r];
      const float s = sigmoid(z);
      a2[t][r] = z * s;
      d2[t][r] = s * (1.0f + z * (1.0f - s));
      tr[r][t] = w3[r] * a2[t][r];
    }
  }
  if (w == 0) {
    f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) p += tr[r];
    part0[l] = p;
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) term[w - 1][r][l] = tr[r];
  }
  __syncthreads();
  // ---- output, the same in all four waves
  f32x4 out = part0[l];
#pragma unroll
  for (int u = 0; u < 3; ++u)
#pragma unroll
    for (int r = 0; r < 4; ++r) out += term[u][r][l];
  float dout[4];
  float sq = 0.f;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    float v = out[t];
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    const float d = (v + P[kOffB3] - Y[base + 16 * t + c]) * OK[base + 16 * t + c];
    dout[t] = 2.0f * d * inv_n;
    sq += d * d;
  }
  float *G = grad + (size_t)blockIdx.x * kGradStride;
  // ---- dZ2; b2 and W3 gradients, summed over the 16 sample lanes
  float aw[4] = {}, ab[4] = {};
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f32x4 dzv;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      aw[r] += dout[t] * a2[t][r];
      const float dz = dout[t] * w3[r] * d2[t][r];
      ab[r] += dz;
      dzv[r] = dz;
    }
    dzs[w][t][l] = f2bf4(dzv);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float sw = sum16(aw[r]), sb = sum16(ab[r]);
    if (c == 0) G[kOffW3 + h0 + r] = sw, G[kOffB2 + h0 + r] = sb;
  }
  __syncthreads();
  // ---- dH1^T = W2^T dZ2^T, dZ1; W1 and b1 gradients
  bf16x4 a1w[4];  // rows of W2^T
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if constexpr (PACKED) {
      a1w[q] = *reinterpret_cast<const bf16x4 *>(W2Tb + (16 * w + c) * kH + 16 * q + 4 * g);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) a1w[q][e] = f2bf(P[kOffW2 + (16 * q + 4 * g + e) * kH + 16 * w + c]);
    }
  }
  float gW1[4][3] = {}, gB1[4] = {};
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 4; u += 2) acc = mfma32(a1w[u], a1w[u + 1], dzs[u][t][l], dzs[u + 1][t][l], acc);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float dz = acc[e] * d1[t][e];
      const float *xs = X + 3 * (base + 16 * t + c);
      gB1[e] += dz;
      gW1[e][0] += dz * xs[0];
      gW1[e][1] += dz * xs[1];
      gW1[e][2] += dz * xs[2];
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float v0 = sum16(gW1[e][0]), v1 = sum16(gW1[e][1]), v2 = sum16(gW1[e][2]), vb = sum16(gB1[e]);
    const int h = h0 + e;
    if (c == 0) G[kOffW1 + 3 * h] = v0, G[kOffW1 + 3 * h + 1] = v1, G[kOffW1 + 3 * h + 2] = v2, G[kOffB1 + h] = vb;
  }
  // ---- dW2^T = H1^T dZ2: a lane's 4 values are 4 of a row of dW2
  bf16x4 dzt[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) dzt[t] = read_transposed(dzs[w][t], g, c);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; t += 2)
      acc = mfma32(read_transposed(h1s[q][t], g, c), read_transposed(h1s[q][t + 1], g, c), dzt[t], dzt[t + 1], acc);
    __builtin_nontemporal_store((f32x4u)acc,
                                reinterpret_cast<f32x4u *>(G + kOffW2 + (16 * w + c) * kH + 16 * q + 4 * g));
  }
  // b3: sum of dout over the samples (group g = 0 holds each sample once)
  if (w == 0) {
    float db = (g == 0) ? (dout[0] + dout[1] + dout[2] + dout[3]) : 0.f;
    float ls = (g == 0) ? sq : 0.f;
    db = sum16(db), ls = sum16(ls);
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) db += __shfl_xor(db, o, 64), ls += __shfl_xor(ls, o, 64);
    if (l == 0) G[kOffB3] = db, loss[blockIdx.x] = ls;
  }
}

// Fixed-order column sums of the wave partials: column p of the nw x kGradStride
// array, added in row (wave) order in FP32, whatever the grid.  One thread per
// column walking the rows waits for memory once per few rows (289 us for the
// 1,024 rows of a 65,536-sample batch).  Here a workgroup of 1,024 threads owns
// kSumCols columns: all of it loads kSumRows rows into LDS and one thread per
// column adds them in order, four rows a read and the next reads in flight,
// while the next chunk is on its way into the other buffer.  32 columns are one
// 128-byte line of a row and make 141 workgroups of the 4,481 columns; the
// training step gives the CUs they leave the next step's samples.  What bounds
// it is the chain of adds and, before it, the first chunk's arrival: a call for
// 65,536 gradients takes 24.0 us with 512 rows and each read waited for, 22.6
// with the next reads in flight, 21.4 so with 256 rows, 21.3 with 128 (22.4 with
// the loads of four chunks in flight).
constexpr int kSumCols = 32;
constexpr int kSumRows = 128;
constexpr int kSumThreads = 1024;
constexpr int kSumPer = kSumRows * kSumCols / kSumThreads;          // rows a thread loads of a chunk
constexpr int kSumBlocks = (kParams + kSumCols - 1) / kSumCols;     // workgroups of the columns
constexpr int kSumLd = kSumRows + 4;  // rows of a column in LDS, padded: 16-byte reads of 16 columns meet all banks
static_assert(kGradStride == kSumBlocks * kSumCols, "a partial's row is the workgroups' columns");
static_assert(kSumThreads % kSumCols == 0 && kSumPer * (kSumThreads / kSumCols) == kSumRows, "chunk split");
struct SumLds {
  float v[2][kSumCols][kSumLd];
};

// s plus v[0..m) in order.  The barriers keep the reads where they are, half a
// turn before their adds.
__device__ __forceinline__ float add_in_order(float s, const float *v, int m) {
  int r = 0;
  const auto load = [&](f32x4(&t)[4], int at) {
#pragma unroll
    for (int k = 0; k < 4; ++k) t[k] = *reinterpret_cast<const f32x4 *>(v + at + 4 * k);
  };
  const auto add = [&](const f32x4(&t)[4]) {
#pragma unroll
    for (int k = 0; k < 16; ++k) s += t[k / 4][k % 4];
  };
  if (m >= 32) {
    f32x4 a[4], b[4];
    load(a, 0);
    for (; r + 64 <= m; r += 32) {
      load(b, r + 16);
      __builtin_amdgcn_sched_barrier(0);
      add(a);
      load(a, r + 32);
      __builtin_amdgcn_sched_barrier(0);
      add(b);
    }
    load(b, r + 16);
    add(a);
    add(b);
    r += 32;
  }
  for (; r < m; ++r) s += v[r];
  return s;
}

// The sum of column col0 + threadIdx.x in the threads below kSumCols (0 for
// columns past the last; other threads: unspecified).  Called by the whole block.
__device__ __forceinline__ float ordered_column_sum(const float *__restrict__ part, int nw, int col0, SumLds &lds) {
  const int c = threadIdx.x % kSumCols, r0 = threadIdx.x / kSumCols;
  constexpr int kStep = kSumThreads / kSumCols;
  const bool in = col0 + c < kParams;
  float v[kSumPer], s = 0.f;
  auto load = [&](int base) {
#pragma unroll
    for (int k = 0; k < kSumPer; ++k) {
      const int r = base + r0 + k * kStep;
      v[k] = in && r < nw ? part[(size_t)r * kGradStride + col0 + c] : 0.f;
    }
  };
  load(0);
  for (int base = 0, b = 0; base < nw; base += kSumRows, b ^= 1) {
    // The buffer was last read two chunks ago, before the last barrier.
#pragma unroll
    for (int k = 0; k < kSumPer; ++k) lds.v[b][c][r0 + k * kStep] = v[k];
    if (base + kSumRows < nw) load(base + kSumRows);
    __syncthreads();
    if (threadIdx.x < kSumCols) s = add_in_order(s, lds.v[b][c], nw - base < kSumRows ? nw - base : kSumRows);
  }
  return s;
}

// The sum of the nw wave losses in wave order, in thread 0 of the block.
__device__ __forceinline__ float ordered_loss_sum(const float *__restrict__ loss, int nw, SumLds &lds) {
  constexpr int kChunk = kSumCols * kSumLd;
  float *v = &lds.v[0][0][0];
  float s = 0.f;
  for (int base = 0; base < nw; base += kChunk) {
    const int m = nw - base < kChunk ? nw - base : kChunk;
    __syncthreads();
    for (int k = threadIdx.x; k < m; k += kSumThreads) v[k] = loss[base + k];
    __syncthreads();
    if (threadIdx.x == 0) s = add_in_order(s, v, m);
  }
  return s;
}

// Sum of the wave partials in wave order, then Adam (bias-corrected) with a
// cosine learning-rate schedule.  The next workgroup sums the losses instead
// and advances the step: step[1] is this step's number, which k_mlp_grad copied
// from step[0]; only this workgroup writes step[0], which nobody reads here.
// The workgroups after it write the next step's samples over this step's, which
// k_mlp_grad has finished reading, spread over the CUs that the sum leaves (114
// of 256; a workgroup's 16 waves fill its CU): the fewer waves a SIMD has, the
// sooner its samples are done.  With one step a graph, which adds about 5 us to each, a
// training step takes 18.5 us at 1,024 samples (24.8 with
// 640 samples a workgroup at every size), 19.9 at 16,384 (26.5), 28 at 49,152
// (31), 34 at 65,536 (34; with a launch of its own for the samples 7 more), 41 at
// 98,304 (51).  A batch that does not fit the idle CUs at once takes 640 each:
// 55 us at 131,072, 60 with all 1,024 threads.  (So does any batch where the sum
// takes every CU, as on a partitioned GPU.)
int gen_per(int n, int cus) {
  const int idle = cus - (kSumBlocks + 1);
  if (idle < 1 || (n + idle - 1) / idle > kSumThreads) return 640;
  return ((n + idle - 1) / idle + 63) / 64 * 64;
}
__global__ __launch_bounds__(kSumThreads) void k_mlp_adam(float *P, float *Mo, float *Vo, short *W2b, short *W2Tb,
                                                          const float *grad, int nwaves, uint32_t *step,
                                                          int total_steps, float lr0, const float *loss,
                                                          float *loss_hist, Batch next, int per) {
  __shared__ __align__(16) SumLds lds;
  const uint32_t s = step[1];
  if (blockIdx.x > kSumBlocks) {
    const int i = (blockIdx.x - kSumBlocks - 1) * per + threadIdx.x;
    if ((int)threadIdx.x < per && i < next.n)
      put_sample(next.gamma, next.seed, (uint64_t)(s + 1u) * (uint64_t)next.n + (uint64_t)i, i, next.norm, next.X,
                 next.Y, next.OK);
    return;
  }
  if (blockIdx.x == kSumBlocks) {
    const float t = ordered_loss_sum(loss, nwaves, lds);
    if (threadIdx.x == 0) {
      loss_hist[s] = t;
      step[0] = s + 1u;
    }
    return;
  }
  const int col0 = blockIdx.x * kSumCols;
  const float gsum = ordered_column_sum(grad, nwaves, col0, lds);
  const int p = col0 + threadIdx.x;
  if (threadIdx.x < kSumCols && p < kParams) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float m = b1 * Mo[p] + (1.f - b1) * gsum;
    const float v = b2 * Vo[p] + (1.f - b2) * gsum * gsum;
    Mo[p] = m, Vo[p] = v;
    const float tt = (float)(s + 1);
    const float mh = m / (1.f - powf(b1, tt)), vh = v / (1.f - powf(b2, tt));
    const float frac = (float)s / (float)(total_steps > 1 ? total_steps - 1 : 1);
    const float lr = lr0 * (0.02f + 0.98f * 0.5f * (1.f + cosf(3.14159265f * frac)));
    const float np = P[p] - lr * mh / (sqrtf(vh) + eps);
    P[p] = np;
    if (p >= kOffW2 && p < kOffB2) {
      const int i = (p - kOffW2) / kH, j = (p - kOffW2) % kH;
      W2b[i * kH + j] = f2bf(np);
      W2Tb[j * kH + i] = f2bf(np);
    }
  }
}

// The gradient and the loss of one batch from the wave partials, each added in
// wave order in FP32.
__global__ __launch_bounds__(kSumThreads) void k_mlp_sum(const float *part, const float *lpart, int nw, float *grad,
                                                         float *loss) {
  __shared__ __align__(16) SumLds lds;
  if (blockIdx.x == kSumBlocks) {
    const float t = ordered_loss_sum(lpart, nw, lds);
    if (threadIdx.x == 0) *loss = t;
    return;
  }
  const int col0 = blockIdx.x * kSumCols;
  const float g = ordered_column_sum(part, nw, col0, lds);
  if (threadIdx.x < kSumCols && col0 + (int)threadIdx.x < kParams) grad[col0 + threadIdx.x] = g;
}

__global__ void k_mlp_pack(const float *P, short *W2b, short *W2Tb) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= kH * kH) return;
  const int i = k / kH, j = k % kH;
  const short b = f2bf(P[kOffW2 + k]);
  W2b[i * kH + j] = b;
  W2Tb[j * kH + i] = b;
}

// Inference: p = p0 exp(out * sd_y + mu_y) for n conserved states (U: n x 5).
__global__ __launch_bounds__(256) void k_mlp_eval(const float *__restrict__ P, const short *__restrict__ W2b, int64_t n,
                                                  const double *__restrict__ U, double *__restrict__ p_out) {
  const int l = threadIdx.x & 63;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  float xl[3] = {0.f, 0.f, 0.f};
  const float *norm = P + kOffNorm;
  const double gamma = norm[8];
  double p0 = 0.0;
  if (i < n) {
    const double *u = U + 5 * i;
    const double m = sqrt((u[1] * u[1] + u[2] * u[2]) + u[3] * u[3]);
    features(norm, gamma / (gamma - 1.0), u[0], m, u[4], xl, p0);
  }
  float x[4][3];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int f = 0; f < 3; ++f) x[t][f] = __shfl(xl[f], 16 * t + (l & 15), 64);
  float out[4];
  forward_wave(P, W2b, x, out);
  const float o = out[l >> 4];  // this lane's own sample 16 (l/16) + l%16 = l
  if (i < n) p_out[i] = predicted_pressure(norm, o, p0);
}

// MFMA lane-layout self test of mfma32 as the kernels use it: units k of two
// 16-unit blocks, lane group g holding k = 4 g + e (lo) and 16 + 4 g + e (hi).
// A[i][3] = i + 1 and A[i][23] = 0.5, B[3][j] = 16 (j + 1) and B[23][j] = 2, all
// other entries 0, so C[i][j] = 16 (i + 1)(j + 1) + 1 exactly; out[64*4] = C
// per lane (C[i][j] expected in lane j + 16 (i/4), element i%4).
__global__ void k_mlp_selftest(float *out) {
  const int l = threadIdx.x & 63;
  const int g = l >> 4, c = l & 15;
  bf16x4 a[2], b[2];
  for (int h = 0; h < 2; ++h)
    for (int e = 0; e < 4; ++e) {
      const int k = 16 * h + 4 * g + e;
      a[h][e] = f2bf((k == 3 ? (float)(c + 1) : 0.0f) + (k == 23 ? 0.5f : 0.0f));
      b[h][e] = f2bf((k == 3 ? 16.0f * (float)(c + 1) : 0.0f) + (k == 23 ? 2.0f : 0.0f));
    }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = mfma32(a[0], a[1], b[0], b[1], acc);
  for (int r = 0; r < 4; ++r) out[4 * l + r] = acc[r];
}

hipError_t launch_gen(double gamma, uint64_t seed, int n, const float *norm, float *X, float *Y, float *OK,
                      hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_gen, dim3((n + 255) / 256), dim3(256), 0, s, gamma, seed, n, norm, X, Y, OK);
  return hipGetLastError();
}
hipError_t launch_grad(const float *P, const short *W2b, const short *W2Tb, const float *X, const float *Y,
                       const float *OK, float inv_n, int n, float *grad, float *loss, uint32_t *step, hipStream_t s) {
  // n is a multiple of 256, so of the 64 samples of a workgroup
  if (W2b)
    hipLaunchKernelGGL(k_mlp_grad<true>, dim3(n / 64), dim3(256), 0, s, P, W2b, W2Tb, X, Y, OK, inv_n, grad, loss,
                       step);
  else
    hipLaunchKernelGGL(k_mlp_grad<false>, dim3(n / 64), dim3(256), 0, s, P, W2b, W2Tb, X, Y, OK, inv_n, grad, loss,
                       step);
  return hipGetLastError();
}
hipError_t launch_adam(float *P, float *M, float *V, short *W2b, short *W2Tb, const float *grad, int nwaves,
                       uint32_t *step, int total_steps, float lr0, const float *loss, float *loss_hist,
                       const Batch &next, int cus, hipStream_t s) {
  const int per = gen_per(next.n, cus);
  const unsigned int blocks = kSumBlocks + 1 + (next.n + per - 1) / per;
  hipLaunchKernelGGL(k_mlp_adam, dim3(blocks), dim3(kSumThreads), 0, s, P, M, V, W2b, W2Tb, grad, nwaves, step,
                     total_steps, lr0, loss, loss_hist, next, per);
  return hipGetLastError();
}
hipError_t launch_sum(const float *part, const float *lpart, int nw, float *grad, float *loss, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_sum, dim3(kSumBlocks + 1), dim3(kSumThreads), 0, s, part, lpart, nw, grad, loss);
  return hipGetLastError();
}
hipError_t launch_pack(const float *P, short *W2b, short *W2Tb, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_pack, dim3(kH * kH / 256), dim3(256), 0, s, P, W2b, W2Tb);
  return hipGetLastError();
}
hipError_t launch_eval(const float *P, const short *W2b, int64_t n, const double *U, double *p_out, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_mlp_eval, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, P, W2b, n, U, p_out);
  return hipGetLastError();
}
hipError_t launch_selftest(float *out, hipStream_t s) {
  hipLaunchKernelGGL(k_mlp_selftest, dim3(1), dim3(64), 0, s, out);
  return hipGetLastError();
}

}  // namespace rhllc_mlp

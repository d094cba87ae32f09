// Launchers of the surrogate-MLP kernels (mlp_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rhllc_mlp {

// Floats between the gradient partials of two waves: the parameters in whole
// 128-byte lines, so a workgroup of the sums reads whole lines of its own.
constexpr int kGradStride = 4512;

// Samples 0..n-1 of a seed's stream (norm null: not normalised).
hipError_t launch_gen(double gamma, uint64_t seed, int n, const float *norm, float *X, float *Y, float *OK,
                      hipStream_t s);
// The batch of a training run that k_mlp_adam makes for the next step.
struct Batch {
  double gamma;
  uint64_t seed;
  int n;
  const float *norm;
  float *X, *Y, *OK;
};
// nw = n / 64 partials of kGradStride floats in grad and one loss each.  W2b,
// W2Tb: launch_pack's copies, or null (formed from P by every workgroup).  step
// (null outside training): {the next step's number, this step's}, step[1] =
// step[0] here.
hipError_t launch_grad(const float *P, const short *W2b, const short *W2Tb, const float *X, const float *Y,
                       const float *OK, float inv_n, int n, float *grad, float *loss, uint32_t *step, hipStream_t s);
hipError_t launch_adam(float *P, float *M, float *V, short *W2b, short *W2Tb, const float *grad, int nwaves,
                       uint32_t *step, int total_steps, float lr0, const float *loss, float *loss_hist,
                       const Batch &next, int cus, hipStream_t s);
// Samples of the next step that a workgroup of that launch makes, on a device of `cus` CUs.
int gen_per(int n, int cus);
// grad[p] = sum_w part[w * kGradStride + p] and *loss = sum_w lpart[w], in w order (FP32).
hipError_t launch_sum(const float *part, const float *lpart, int nw, float *grad, float *loss, hipStream_t s);
hipError_t launch_pack(const float *P, short *W2b, short *W2Tb, hipStream_t s);
hipError_t launch_eval(const float *P, const short *W2b, int64_t n, const double *U, double *p_out, hipStream_t s);
hipError_t launch_selftest(float *out, hipStream_t s);

}  // namespace rhllc_mlp

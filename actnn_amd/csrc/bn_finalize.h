// The fold of batch norm's partial sums into per-channel statistics, by a wave per channel: a launch of its own
// (batch_norm.hip), or some blocks of the launch that sums up the ranges of the compressed input (calc_precision_dev.hip).
#pragma once
#include "device_utils.h"

namespace actnn {

// what the fold reads and writes
struct BnFinalize {
  const float* part;
  const float* weight;
  const float* bias;
  float* running_mean;
  float* running_var;
  float* save_mean;
  float* save_invstd;
  float* coef;
  int64_t N, C, HW, L;
  int nsplit, slots;
  double momentum, eps;
};

// Folds the table of partial sums of channel c in double precision: the wave's lanes take the
// (span, batch split) entries of the channel in a fixed assignment and are combined by a butterfly,
// so every lane ends with the same totals and the order of the additions is fixed.
// (channels-last tables, slots == 0, hold nsplit consecutive values per channel and sum.)
ACTNN_DEV void channel_totals(const float* __restrict__ part, int64_t c, int64_t HW, int64_t L,
                              int nsplit, int slots, double& s0, double& s1) {
  const int lane = threadIdx.x & 63;
  s0 = 0.0;
  s1 = 0.0;
  if (slots == 0) {
    const float* q0 = part + (c * 2) * (int64_t)nsplit;
    const float* q1 = q0 + nsplit;
#pragma unroll 8
    for (int i = lane; i < nsplit; i += 64) {
      s0 += (double)q0[i];
      s1 += (double)q1[i];
    }
  } else {
    const int64_t j0 = (c * HW) / L, j1 = ((c + 1) * HW - 1) / L;
    const int64_t count = (j1 - j0 + 1) * nsplit;
    for (int64_t i = lane; i < count; i += 64) {
      const int64_t j = j0 + i / nsplit, y = i % nsplit;
      const int64_t slot = c - (j * L) / HW;
      const float* q = part + ((j * nsplit + y) * slots + slot) * 2;
      s0 += (double)q[0];
      s1 += (double)q[1];
    }
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    s0 += __shfl_xor(s0, d);
    s1 += __shfl_xor(s1, d);
  }
}

// mean / inverse standard deviation of the batch, the running estimates (unbiased variance, as
// torch's batch norm keeps them) and the per-channel coefficients of y = a*x + b.
ACTNN_DEV void bn_finalize_channel(const BnFinalize& f, int64_t c) {
  double S, Q;
  channel_totals(f.part, c, f.HW, f.L, f.nsplit, f.slots, S, Q);
  if ((threadIdx.x & 63) != 0) return;
  const double M = (double)f.N * (double)f.HW;
  const double mean = S / M;
  double var = Q / M - mean * mean;
  if (!(var > 0.0)) var = 0.0;
  const double invstd = 1.0 / sqrt(var + f.eps);
  f.save_mean[c] = (float)mean;
  f.save_invstd[c] = (float)invstd;
  if (f.running_mean) f.running_mean[c] = (float)((1.0 - f.momentum) * f.running_mean[c] + f.momentum * mean);
  if (f.running_var) {
    const double unbiased = M > 1.0 ? var * (M / (M - 1.0)) : var;
    f.running_var[c] = (float)((1.0 - f.momentum) * f.running_var[c] + f.momentum * unbiased);
  }
  const double a = (f.weight ? (double)f.weight[c] : 1.0) * invstd;
  f.coef[2 * c] = (float)a;
  f.coef[2 * c + 1] = (float)((f.bias ? (double)f.bias[c] : 0.0) - mean * a);
}

}  // namespace actnn

// Internal interface of the FP32 network kernels (kernels_mlp.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace cghip {

constexpr int kMlpMaxWidth = 256;  // every layer width <= one block of threads

struct MlpDims {
  int in, h1, h2, out;
};

struct AdamStep {
  float lr, beta1, beta2, eps;
  float corr1, corr2;  // 1 / (1 - beta1^t), 1 / (1 - beta2^t)
  int apply;           // 0: only fold the gradient
};

int mlp_param_count(const MlpDims &d);

// Blocks (and loss shares) of mlp_backprop for `rows` samples.
int mlp_tiles(int rows);

// Of every layer k what mlp_backprop leaves for mlp_gradient, one row per
// sample: its inputs followed by a 1 (in[k], widths in + 1, h1 + 1, h2 + 1)
// and its deltas (delta[k], widths h1, h2, out).
struct MlpTables {
  float *in[3], *delta[3];
};

// Slices of the samples whose gradient sums are formed apart (slice g:
// samples g, g + G, ...; G = min(rows, kMlpSlices)), and the table rows of
// one lane in the gradient kernel: a block keeps kMlpSlices * kMlpGradRows *
// 64 slice sums, 64 KB, in LDS.
constexpr int kMlpSlices = 128;
constexpr int kMlpGradRows = 2;

// Once per device before mlp_backprop.
hipError_t mlp_prepare();

hipError_t mlp_forward(const MlpDims &d, const float *P, const float *X, int rows, float *Y,
                       hipStream_t s);
// Forward and backward of the MSE loss: the tables and the loss shares
// Lp[mlp_tiles(rows)].
hipError_t mlp_backprop(const MlpDims &d, const float *P, const float *X, const float *T, int rows,
                        const MlpTables &tab, double *Lp, hipStream_t s);
// The gradient (copied to `grad` when non-null), when a.apply one Adam step
// on P with moments M, V, and the loss.
hipError_t mlp_gradient(const MlpDims &d, int rows, const MlpTables &tab, float *grad, float *P,
                        float *M, float *V, const AdamStep &a, const double *Lp, double *loss,
                        hipStream_t s);

}  // namespace cghip

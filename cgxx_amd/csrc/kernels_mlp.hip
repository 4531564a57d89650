// Small fully connected network in FP32 for gfx950: in -> h1 -> h2 -> out,
// ReLU after the two hidden layers, mean-squared-error loss, full-batch
// gradients and Adam (Kingma & Ba, "Adam: A Method for Stochastic
// Optimization", ICLR 2015, Algorithm 1).
//
// The network is tiny (a few ten thousand parameters) and the batches are a
// few thousand rows: a training step is bound by latency, so it is two
// launches, each with every compute unit busy and no step's intermediate
// slices in memory:
//   k_mlp_backprop   4 or 8 samples per block, forward and backward to the
//                    layers' deltas with the samples and the weights in LDS;
//   k_mlp_gradient   up to 128 parameters per block, the sum over the samples and
//                    the Adam update of those parameters.
// No matrix cores: the products are 40..128 wide, and each output keeps its
// own ascending FP32 sum.
//
// Determinism: every sum has a fixed order.  A forward dot adds inputs in
// ascending index order; a parameter's gradient is the sum over G slices in
// ascending order, slice g being samples g, g + G, ... in ascending order
// (no atomics).
//
// Parameter layout (one contiguous float array):
//   W1[in][h1] b1[h1] W2[h1][h2] b2[h2] W3[h2][out] b3[out]
// (W[i][j] = weight from input i to output j, row-major).

#include "mlp.h"

#include <hip/hip_runtime.h>

#pragma clang fp contract(off)

namespace cghip {
namespace {

constexpr int kThreads = 256;

struct Offsets {
  int w1, b1, w2, b2, w3, b3, total;
};

__host__ __device__ inline Offsets offsets(const MlpDims &d) {
  Offsets o;
  o.w1 = 0;
  o.b1 = o.w1 + d.in * d.h1;
  o.w2 = o.b1 + d.h1;
  o.b2 = o.w2 + d.h1 * d.h2;
  o.w3 = o.b2 + d.h2;
  o.b3 = o.w3 + d.h2 * d.out;
  o.total = o.b3 + d.out;
  return o;
}

// Samples in LDS: one row per sample, rows padded to kPad units (16-byte
// reads of four units, in bounds in the last chunk too).
constexpr int kPad = 8;
__host__ __device__ inline int padded(int width) { return (width + kPad - 1) / kPad * kPad; }

// acc[q] + x_q[0] w[0] + x_q[1] w[1] + ..., added left to right for SP
// samples; x_q at x + q * ldx (ldx a multiple of kPad), weight i at w[i *
// ldw].  32 weights are loaded ahead of their products: one load per product
// waited for every load (a layer of 128 inputs: 128 cache round trips).
template <int SP>
__device__ inline void dot_ascending(const float *__restrict__ w, int ldw, const float *x, int ldx,
                                     int n, float (&acc)[SP]) {
  constexpr int U = 32;
  int i = 0;
  for (; i + U <= n; i += U) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; u++) v[u] = w[(i + u) * ldw];
#pragma unroll
    for (int u = 0; u < U; u += 4)
#pragma unroll
      for (int q = 0; q < SP; q++) {
        const float4 xv = *reinterpret_cast<const float4 *>(x + q * ldx + i + u);
        acc[q] = acc[q] + xv.x * v[u];
        acc[q] = acc[q] + xv.y * v[u + 1];
        acc[q] = acc[q] + xv.z * v[u + 2];
        acc[q] = acc[q] + xv.w * v[u + 3];
      }
  }
  for (; i < n; i += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) v[u] = w[min(i + u, n - 1) * ldw];
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (i + u < n) {
#pragma unroll
        for (int q = 0; q < SP; q++) acc[q] = acc[q] + x[q * ldx + i + u] * v[u];
      }
  }
}

// y[j] = b[j] + sum_i x[i] W[i][j] for j < nout (thread j), optional ReLU.
__device__ inline void dense_layer(const float *__restrict__ W, const float *__restrict__ b,
                                   const float *x, int nin, int nout, bool relu, float *y) {
  const int j = threadIdx.x;
  if (j < nout) {
    float acc[1] = {b[j]};
    dot_ascending<1>(W + j, nout, x, 0, nin, acc);
    y[j] = relu ? fmaxf(acc[0], 0.0f) : acc[0];
  }
}

// One block per sample: the output y.
__global__ __launch_bounds__(kThreads) void k_mlp_forward(MlpDims d, const float *__restrict__ P,
                                                          const float *__restrict__ X, int rows,
                                                          float *__restrict__ Y) {
  __shared__ __attribute__((aligned(16))) float x[kMlpMaxWidth], a1[kMlpMaxWidth], a2[kMlpMaxWidth], y[kMlpMaxWidth];
  const int s = blockIdx.x;
  if (s >= rows) return;
  const Offsets o = offsets(d);
  const int t = threadIdx.x;
  if (t < d.in) x[t] = X[(size_t)s * d.in + t];
  __syncthreads();
  dense_layer(P + o.w1, P + o.b1, x, d.in, d.h1, true, a1);
  __syncthreads();
  dense_layer(P + o.w2, P + o.b2, a1, d.h1, d.h2, true, a2);
  __syncthreads();
  dense_layer(P + o.w3, P + o.b3, a2, d.h2, d.out, false, y);
  if (t < d.out) Y[(size_t)s * d.out + t] = y[t];
}

constexpr int kBackThreads = 512;

// The thread's place in a layer of `nout` outputs for a tile of TILE
// samples: output j, samples q0 .. q0 + SP - 1 of the tile with SP = per (1,
// 2 or 4; 0: none).  Whole waves of a block share a group of samples; a
// weight is read once for the group.
template <int TILE>
struct LayerPlace {
  int j, q0, per;
  __device__ explicit LayerPlace(int nout) {
    const int w = (nout + 63) & ~63;
    const int room = w <= 64 ? 8 : w <= 128 ? 4 : 2;  // groups that fit
    const int groups = min(room, TILE);
    const int g = (int)threadIdx.x / w;
    j = (int)threadIdx.x - g * w;
    q0 = g * (TILE / groups);
    per = g < groups && j < nout ? TILE / groups : 0;
  }
};
static_assert(kBackThreads == 512 && kMlpMaxWidth == 256, "groups of LayerPlace");

// out[q * ldo + j] = f(acc, q) for the place's samples.
template <int SP, typename L, typename F>
__device__ inline void layer_sp(const L &l, float init, const float *w, int ldw, const float *x,
                                int ldx, int nin, float *out, int ldo, F f) {
  float acc[SP];
#pragma unroll
  for (int q = 0; q < SP; q++) acc[q] = init;
  dot_ascending<SP>(w, ldw, x + l.q0 * ldx, ldx, nin, acc);
#pragma unroll
  for (int q = 0; q < SP; q++) out[(l.q0 + q) * ldo + l.j] = f(acc[q], l.q0 + q);
}
template <typename L, typename F>
__device__ inline void layer(const L &l, float init, const float *w, int ldw, const float *x,
                             int ldx, int nin, float *out, int ldo, F f) {
  if (l.per == 1) layer_sp<1>(l, init, w, ldw, x, ldx, nin, out, ldo, f);
  if (l.per == 2) layer_sp<2>(l, init, w, ldw, x, ldx, nin, out, ldo, f);
  if (l.per == 4) layer_sp<4>(l, init, w, ldw, x, ldx, nin, out, ldo, f);
}

// Loss L = sum_{s,o} (Y - T)^2 / (rows * out).  Block b takes samples b *
// TILE .. b * TILE + TILE - 1 (fewer in the last block) forward and back: the
// inputs of every layer with a 1 after them (the bias's input) in IN, the
// deltas in D, the block's loss share in Lp[b].  STAGE: the weights are
// copied to LDS first, every load in flight at once, so that no layer waits
// for memory; W2 with rows of h2 + 1 floats (the odd stride spreads a column
// over the banks): the forward layer reads its columns, the backward one its
// rows, which in memory lie h2 floats apart between lanes.  Bound by the
// chain of five layers in one block; 1200 samples, 37-128-128-13: 21 us
// (227 us with one sample at a time and the weights read through the caches).
template <bool STAGE, int TILE>
__global__ __launch_bounds__(kBackThreads) void k_mlp_backprop(
    MlpDims d, const float *__restrict__ P, const float *__restrict__ X,
    const float *__restrict__ T, int rows, MlpTables tab, double *__restrict__ Lp) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ double lsum[kBackThreads / 64];
  const int li = padded(d.in + 1), l1 = padded(d.h1 + 1), l2 = padded(d.h2 + 1), lo = padded(d.out);
  float *x = lds, *a1 = x + li * TILE, *a2 = a1 + l1 * TILE, *dy = a2 + l2 * TILE,
        *d2 = dy + lo * TILE, *d1 = d2 + l2 * TILE, *s1 = d1 + l1 * TILE, *s3 = s1 + d.in * d.h1,
        *s2 = s3 + d.h2 * d.out;
  const Offsets o = offsets(d);
  const int t = threadIdx.x;
  const int s0 = blockIdx.x * TILE, ns = min(TILE, rows - s0);
  const float scale = 2.0f / ((float)rows * (float)d.out);
  const LayerPlace<TILE> p1(d.h1), p2(d.h2), p3(d.out);
  const float bias1 = p1.per ? P[o.b1 + p1.j] : 0.0f, bias2 = p2.per ? P[o.b2 + p2.j] : 0.0f,
              bias3 = p3.per ? P[o.b3 + p3.j] : 0.0f;
  // samples past the last row are zeros (every width < kBackThreads)
  auto load = [&](const float *g, int width, float *l, int ld) {
    if (t < width) {
#pragma unroll
      for (int q = 0; q < TILE; q++)
        l[q * ld + t] = q < ns ? g[(size_t)(s0 + q) * width + t] : 0.0f;
    }
  };
  auto store = [&](float *g, int width, const float *l, int ld) {
    if (t < width)
      for (int q = 0; q < ns; q++) g[(size_t)(s0 + q) * width + t] = l[q * ld + t];
  };
  const float *w1 = P + o.w1, *w2 = P + o.w2, *w3 = P + o.w3;
  int ld2 = d.h2;
  if (STAGE) {
    // W2: kBackThreads / h2 rows a pass, thread (row0, c) of each
    constexpr int U1 = 12, U2 = 32, U3 = 6;
    const int n1 = d.in * d.h1, n3 = d.h2 * d.out;
    const int R = kBackThreads / d.h2, row0 = t / d.h2, c = t - row0 * d.h2;
    float v1[U1], v2[U2], v3[U3];
#pragma unroll
    for (int u = 0; u < U2; u++) v2[u] = w2[min(row0 + u * R, d.h1 - 1) * d.h2 + c];
#pragma unroll
    for (int u = 0; u < U1; u++) v1[u] = w1[min(t + u * kBackThreads, n1 - 1)];
#pragma unroll
    for (int u = 0; u < U3; u++) v3[u] = w3[min(t + u * kBackThreads, n3 - 1)];
    load(X, d.in, x, li);
    load(T, d.out, dy, lo);
    if (t < TILE) x[t * li + d.in] = a1[t * l1 + d.h1] = a2[t * l2 + d.h2] = 1.0f;
#pragma unroll
    for (int u = 0; u < U2; u++)
      if (row0 < R && row0 + u * R < d.h1) s2[(row0 + u * R) * (d.h2 + 1) + c] = v2[u];
    for (int i = row0 + U2 * R; row0 < R && i < d.h1; i += R)
      s2[i * (d.h2 + 1) + c] = w2[i * d.h2 + c];
#pragma unroll
    for (int u = 0; u < U1; u++)
      if (t + u * kBackThreads < n1) s1[t + u * kBackThreads] = v1[u];
    for (int k = t + U1 * kBackThreads; k < n1; k += kBackThreads) s1[k] = w1[k];
#pragma unroll
    for (int u = 0; u < U3; u++)
      if (t + u * kBackThreads < n3) s3[t + u * kBackThreads] = v3[u];
    for (int k = t + U3 * kBackThreads; k < n3; k += kBackThreads) s3[k] = w3[k];
    ld2 = d.h2 + 1;
  } else {
    load(X, d.in, x, li);
    load(T, d.out, dy, lo);
    if (t < TILE) x[t * li + d.in] = a1[t * l1 + d.h1] = a2[t * l2 + d.h2] = 1.0f;
  }
  __syncthreads();
  const auto relu = [](float v, int) { return fmaxf(v, 0.0f); };
  layer(p1, bias1, (STAGE ? s1 : w1) + p1.j, d.h1, x, li, d.in, a1, l1, relu);
  __syncthreads();
  layer(p2, bias2, (STAGE ? s2 : w2) + p2.j, ld2, a1, l1, d.h1, a2, l2, relu);
  __syncthreads();
  // dy = scale (y - t), over the targets in dy
  double loss = 0.0;
  layer(p3, bias3, (STAGE ? s3 : w3) + p3.j, d.out, a2, l2, d.h2, dy, lo, [&](float y, int q) {
    const float e = q < ns ? y - dy[q * lo + p3.j] : 0.0f;
    loss += (double)e * (double)e;
    return scale * e;
  });
  __syncthreads();
  // d2[j] = (sum_o W3[j][o] dy[o]) * [a2[j] > 0]
  layer(p2, 0.0f, (STAGE ? s3 : w3) + p2.j * d.out, 1, dy, lo, d.out, d2, l2,
        [&](float v, int q) { return a2[q * l2 + p2.j] > 0.0f ? v : 0.0f; });
  __syncthreads();
  // d1[i] = (sum_j W2[i][j] d2[j]) * [a1[i] > 0]
  layer(p1, 0.0f, (STAGE ? s2 : w2) + p1.j * ld2, 1, d2, l2, d.h2, d1, l1,
        [&](float v, int q) { return a1[q * l1 + p1.j] > 0.0f ? v : 0.0f; });
  __syncthreads();
  store(tab.in[0], d.in + 1, x, li);
  store(tab.in[1], d.h1 + 1, a1, l1);
  store(tab.in[2], d.h2 + 1, a2, l2);
  store(tab.delta[0], d.h1, d1, l1);
  store(tab.delta[1], d.h2, d2, l2);
  store(tab.delta[2], d.out, dy, lo);
  for (int off = 32; off >= 1; off >>= 1) loss += __shfl_down(loss, off, 64);
  if ((t & 63) == 0) lsum[t >> 6] = loss;
  __syncthreads();
  if (t == 0) {
    double s = 0.0;
    for (int k = 0; k < kBackThreads / 64; k++) s += lsum[k];
    Lp[blockIdx.x] = s;
  }
}

// Gradient and Adam update of 64 x kGradRows parameters.  A layer's weights
// with its biases below them are one row-major table of nin + 1 rows and nout
// columns, contiguous in the parameters, and parameter (i, j) sums
// in[s][i] delta[s][j] over the samples (in[s][nin] = 1, the bias).  A block
// takes 64 entries of one factor, one per lane, and kGradRows of the other,
// the same for the whole block and staged in LDS.  What bounds it is the
// issue of loads and addresses, not the few MB of the tables: a sample costs
// one coalesced load at an address that is fixed within a round, one LDS
// broadcast and the products.  1200 samples of 37-128-128-13: 12 us;
// 24 us with the second factor in scalar loads (their addresses share one
// scalar unit per compute unit), 32 us with it in vector loads.  The lanes
// lie along the factor that leaves fewer of them empty (mlp_gradient).  The G
// slices (slice g: samples g, g + G, ... in ascending order) are dealt to
// the block's 16 waves in contiguous runs, their sums meet in LDS, and one
// thread per parameter adds them in ascending order.  The last block folds
// the loss.
constexpr int kGradThreads = 1024;
constexpr int kGradRows = kMlpGradRows;
constexpr int kGradMaxSlices = kMlpSlices;
constexpr int kWaves = kGradThreads / 64;
constexpr int kSlices = kGradMaxSlices / kWaves;  // of one wave
constexpr int kRounds = 16;  // staged at once
constexpr int kAhead = 3;    // in flight
struct GradLayer {
  const float *lane, *wave;  // the factors: rows of nl and nw floats
  int nl, nw, groups;        // groups of 64 lanes
  int offset, sl, sw;        // parameter (l, w) is offset + l sl + w sw
  int blocks;
};

__global__ __launch_bounds__(kGradThreads) void k_mlp_gradient(
    GradLayer la, GradLayer lb, GradLayer lc, int rows, int G, float *__restrict__ grad,
    float *__restrict__ P, float *__restrict__ M, float *__restrict__ V, AdamStep a,
    const double *__restrict__ Lp, int tiles, double denom, double *__restrict__ loss) {
  __shared__ float part[kGradMaxSlices * kGradRows * 64];
  __shared__ float w[kRounds * kGradMaxSlices][kGradRows];
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int b = blockIdx.x;
  if (b == la.blocks + lb.blocks + lc.blocks) {
    double s = 0.0;
    for (int k = t; k < tiles; k += kGradThreads) s += Lp[k];
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_down(s, off, 64);
    double *ws = reinterpret_cast<double *>(part);
    if (lane == 0) ws[wave] = s;
    __syncthreads();
    if (t == 0) {
      s = 0.0;
      for (int k = 0; k < kGradThreads / 64; k++) s += ws[k];
      *loss = s / denom;
    }
    return;
  }
  GradLayer l = la;
  if (b >= la.blocks) {
    b -= la.blocks;
    l = lb;
    if (b >= lb.blocks) {
      b -= lb.blocks;
      l = lc;
    }
  }
  // lanes and rows past the table repeat its last ones and store nothing
  const int l0 = b % l.groups * 64 + lane, w0 = b / l.groups * kGradRows;
  const int lo = min(l0, l.nl - 1);
  // slices g0 .. g0 + cnt - 1 of this wave; round m is sample m G + g of each
  const int per = (G + kWaves - 1) / kWaves;
  const int g0 = wave * per, cnt = min(per, G - g0);
  const int rounds = (rows + G - 1) / G;
  float acc[kSlices][kGradRows];
#pragma unroll
  for (int k = 0; k < kSlices; k++)
#pragma unroll
    for (int u = 0; u < kGradRows; u++) acc[k][u] = -0.0f;  // -0 + v is v, for v = -0 too
  int at[kSlices];  // of the slices in a round, from the round's sample g0
#pragma unroll
  for (int k = 0; k < kSlices; k++) at[k] = k * l.nl + lo;
  for (int mc = 0; mc < rounds; mc += kRounds) {
    const int me = min(mc + kRounds, rounds);
    const int64_t s0 = (int64_t)mc * G;
    const int ns = (int)min((int64_t)(me - mc) * G, rows - s0);
    if (mc > 0) __syncthreads();
    for (int i = t; i < ns; i += kGradThreads) {
      const float *r = l.wave + (s0 + i) * l.nw;
#pragma unroll
      for (int u = 0; u < kGradRows; u++) w[i][u] = r[min(w0 + u, l.nw - 1)];
    }
    __syncthreads();
    int m = mc;
    if (cnt == kSlices) {  // whole rounds, kAhead of them in flight
      for (; m + kAhead <= me && (int64_t)(m + kAhead) * G <= rows; m += kAhead) {
        float lv[kAhead][kSlices];
#pragma unroll
        for (int q = 0; q < kAhead; q++) {
          const float *r = l.lane + ((int64_t)(m + q) * G + g0) * l.nl;
#pragma unroll
          for (int k = 0; k < kSlices; k++) lv[q][k] = r[at[k]];
        }
#pragma unroll
        for (int q = 0; q < kAhead; q++)
#pragma unroll
          for (int k = 0; k < kSlices; k++)
#pragma unroll
            for (int u = 0; u < kGradRows; u++)
              acc[k][u] = acc[k][u] + w[(m + q - mc) * G + g0 + k][u] * lv[q][k];
      }
    }
    for (; m < me && cnt > 0; m++) {
      // the slices of the round that have a sample (the same in all lanes)
      const int64_t s = (int64_t)m * G + g0;
      const int live = (int)min((int64_t)cnt, rows - s);
      if (live <= 0) break;
      const float *r = l.lane + s * l.nl;
      float lv[kSlices];
#pragma unroll
      for (int k = 0; k < kSlices; k++) lv[k] = r[k < live ? at[k] : lo];
#pragma unroll
      for (int k = 0; k < kSlices; k++)
        if (k < live) {
#pragma unroll
          for (int u = 0; u < kGradRows; u++)
            acc[k][u] = acc[k][u] + w[(m - mc) * G + g0 + k][u] * lv[k];
        }
    }
  }
#pragma unroll
  for (int k = 0; k < kSlices; k++)
    if (k < cnt) {
#pragma unroll
      for (int u = 0; u < kGradRows; u++)
        part[((g0 + k) * kGradRows + u) * 64 + lane] = acc[k][u];
    }
  __syncthreads();
  if (wave >= kGradRows) return;
  float gsum = 0.0f;  // parameter (l0, w0 + wave)
  for (int g = 0; g < G; g += 16) {
    float v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) v[u] = part[(min(g + u, G - 1) * kGradRows + wave) * 64 + lane];
#pragma unroll
    for (int u = 0; u < 16; u++)
      if (g + u < G) gsum = gsum + v[u];
  }
  if (l0 >= l.nl || w0 + wave >= l.nw) return;
  const int e = l.offset + l0 * l.sl + (w0 + wave) * l.sw;
  if (grad) grad[e] = gsum;
  if (!a.apply) return;
  const float m = a.beta1 * M[e] + (1.0f - a.beta1) * gsum;
  const float v = a.beta2 * V[e] + (1.0f - a.beta2) * (gsum * gsum);
  M[e] = m;
  V[e] = v;
  const float mhat = m * a.corr1;  // corr1 = 1 / (1 - beta1^t)
  const float vhat = v * a.corr2;  // corr2 = 1 / (1 - beta2^t)
  P[e] = P[e] - a.lr * mhat / (sqrtf(vhat) + a.eps);
}

}  // namespace

int mlp_param_count(const MlpDims &d) { return offsets(d).total; }

// Samples per block of k_mlp_backprop: 8 once tiles of 4 would be more than
// one block per compute unit (256), which then run in two rounds.
static int tile_of(int rows) { return rows > 4 * 256 ? 8 : 4; }

int mlp_tiles(int rows) { return (rows + tile_of(rows) - 1) / tile_of(rows); }

hipError_t mlp_forward(const MlpDims &d, const float *P, const float *X, int rows, float *Y,
                       hipStream_t s) {
  if (rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_mlp_forward, dim3(rows), dim3(kThreads), 0, s, d, P, X, rows, Y);
  return hipGetLastError();
}

// The weights go through LDS while they and 8 samples fit a block's share of
// it (up to about 128 x 128 hidden units); wider networks read them from the
// caches.
constexpr size_t kStagedLds = 144 * 1024;

hipError_t mlp_prepare() {
  const void *const staged[2] = {reinterpret_cast<const void *>(&k_mlp_backprop<true, 4>),
                                 reinterpret_cast<const void *>(&k_mlp_backprop<true, 8>)};
  for (const void *k : staged) {
    const hipError_t e =
        hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kStagedLds);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

template <int TILE>
static void backprop(const MlpDims &d, const float *P, const float *X, const float *T, int rows,
                     const MlpTables &tab, double *Lp, hipStream_t s) {
  const dim3 grid(mlp_tiles(rows)), block(kBackThreads);
  const size_t samples = sizeof(float) * TILE *
                         (size_t)(padded(d.in + 1) + 2 * padded(d.h1 + 1) + 2 * padded(d.h2 + 1) +
                                  padded(d.out));
  const size_t weights =
      sizeof(float) * ((size_t)d.in * d.h1 + (size_t)d.h1 * (d.h2 + 1) + (size_t)d.h2 * d.out);
  if (samples + weights <= kStagedLds)
    hipLaunchKernelGGL((k_mlp_backprop<true, TILE>), grid, block, samples + weights, s, d, P, X, T,
                       rows, tab, Lp);
  else
    hipLaunchKernelGGL((k_mlp_backprop<false, TILE>), grid, block, samples, s, d, P, X, T, rows,
                       tab, Lp);
}

hipError_t mlp_backprop(const MlpDims &d, const float *P, const float *X, const float *T, int rows,
                        const MlpTables &tab, double *Lp, hipStream_t s) {
  if (tile_of(rows) == 8)
    backprop<8>(d, P, X, T, rows, tab, Lp, s);
  else
    backprop<4>(d, P, X, T, rows, tab, Lp, s);
  return hipGetLastError();
}

hipError_t mlp_gradient(const MlpDims &d, int rows, const MlpTables &tab, float *grad, float *P,
                        float *M, float *V, const AdamStep &a, const double *Lp, double *loss,
                        hipStream_t s) {
  const Offsets o = offsets(d);
  auto table = [&](int k, int nin, int nout, int offset) {
    auto groups = [](int n) { return (n + 63) / 64; };
    auto blocks = [&](int nl, int nw) { return groups(nl) * ((nw + kGradRows - 1) / kGradRows); };
    const int nr = nin + 1;
    const int columns = blocks(nout, nr), rowwise = blocks(nr, nout);
    return columns <= rowwise
               ? GradLayer{tab.delta[k], tab.in[k], nout, nr, groups(nout), offset, 1, nout, columns}
               : GradLayer{tab.in[k], tab.delta[k], nr, nout, groups(nr), offset, nout, 1, rowwise};
  };
  const GradLayer la = table(0, d.in, d.h1, o.w1), lb = table(1, d.h1, d.h2, o.w2),
                  lc = table(2, d.h2, d.out, o.w3);
  const int G = rows < kGradMaxSlices ? rows : kGradMaxSlices;
  hipLaunchKernelGGL(k_mlp_gradient, dim3(la.blocks + lb.blocks + lc.blocks + 1),
                     dim3(kGradThreads), 0, s, la, lb, lc, rows, G, grad, P, M, V, a, Lp,
                     mlp_tiles(rows), (double)rows * d.out, loss);
  return hipGetLastError();
}

}  // namespace cghip

// Set-up of the symmetric FP64 diagonals (Sym64) from an uploaded CRS or ELL
// matrix, on the device: the distinct off-diagonal offsets, then the diagonal
// and the upper diagonals, then the check that every entry equals its
// transpose bit for bit.  One pass over the matrix each, one row per thread.

#include "device_common.h"

namespace cghip {

namespace {

using namespace dev;

// Entry j of row i of either format.
struct CrsRow {
  const Crs<double> &A;
  int e0, len;
  __device__ CrsRow(const Crs<double> &m, int i) : A(m), e0(m.ptr[i]), len(m.ptr[i + 1] - m.ptr[i]) {}
  __device__ int col(int j) const { return A.index[e0 + j]; }
  __device__ double value(int j) const { return A.value[e0 + j]; }
};
struct EllRow {
  const Ell<double> &A;
  int i, len;
  __device__ EllRow(const Ell<double> &m, int r) : A(m), i(r), len(m.length[r]) {}
  __device__ int col(int j) const { return A.index[(int64_t)j * A.n + i]; }
  __device__ double value(int j) const { return A.data[(int64_t)j * A.n + i]; }
};

constexpr int kFree = INT32_MIN;  // no offset has this value: |offset| < n

// Adds offset o to a set of kDiaMax slots (kFree: empty); false if it is full.
// A slot is written once, so one that holds an offset is only read: swaps at
// one address run one after the other, over the whole device for the common
// set.
__device__ inline bool add_offset(int *set, int o) {
  for (int k = 0; k < kDiaMax; k++) {
    int was = __hip_atomic_load(set + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (was == kFree) was = atomicCAS(set + k, kFree, o);
    if (was == kFree || was == o) return true;
  }
  return false;
}

// Bits of found[0], and the offsets in found[1 .. kDiaMax] (kFree beforehand).
// A block collects its own set in LDS and adds that to the common one; a
// thread asks the set only for offsets that it has not met.  A thread stops
// at the first row that no diagonal layout can hold, and a block with such a
// row leaves the common set alone: 300,000 rows of scattered columns took
// 924 us when every block put its offsets there by swaps, 22 us now.
template <typename Row, typename M>
__global__ __launch_bounds__(kBlock) void k_offsets(M A, int *__restrict__ found) {
  __shared__ int set[kDiaMax];
  __shared__ int block_flags;
  if (threadIdx.x < kDiaMax) set[threadIdx.x] = kFree;
  if (threadIdx.x == 0) block_flags = 0;
  __syncthreads();
  const int64_t T = (int64_t)gridDim.x * kBlock;
  int flags = 0;
  int seen[kDiaMax];
#pragma unroll
  for (int k = 0; k < kDiaMax; k++) seen[k] = kFree;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
       i < A.n && !(flags & kOffsetsIrregular); i += T) {
    const Row row(A, (int)i);
    if (row.len > kDiaMax + 1) flags |= kOffsetsIrregular;
    int prev = -1;
    for (int j = 0; j < row.len && !(flags & kOffsetsIrregular); j++) {
      const int c = row.col(j), o = c - (int)i;
      if (c <= prev) flags |= kOffsetsIrregular;
      if (__builtin_bit_cast(uint64_t, row.value(j)) == kF64Absent) flags |= kOffsetsMarked;
      prev = c;
      bool known = o == 0;
#pragma unroll
      for (int k = 0; k < kDiaMax; k++) known |= seen[k] == o;
      if (known) continue;
      if (!add_offset(set, o)) flags |= kOffsetsIrregular;
      bool put = false;
#pragma unroll
      for (int k = 0; k < kDiaMax; k++)
        if (seen[k] == kFree && !put) {
          seen[k] = o;
          put = true;
        }
    }
  }
  if (flags) atomicOr(&block_flags, flags);
  __syncthreads();
  if (threadIdx.x == 0 && block_flags) atomicOr(found, block_flags);
  if (block_flags & kOffsetsIrregular) return;
  if (threadIdx.x < kDiaMax && set[threadIdx.x] != kFree && !add_offset(found + 1, set[threadIdx.x]))
    atomicOr(found, kOffsetsIrregular);
}

// Column indices against [0, n), one pass at the rate of a copy.
__global__ __launch_bounds__(kBlock) void k_crs_columns(int n, int64_t nnz,
                                                        const int *__restrict__ index,
                                                        int *__restrict__ bad) {
  const int64_t T = (int64_t)gridDim.x * kBlock;
  bool out = false;
  for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < nnz; e += T)
    out |= (uint32_t)index[e] >= (uint32_t)n;
  if (out) bad[0] = 1;
}

__global__ __launch_bounds__(kBlock) void k_ell_columns(int n, const int *__restrict__ length,
                                                        const int *__restrict__ index,
                                                        int *__restrict__ bad) {
  const int64_t T = (int64_t)gridDim.x * kBlock;
  bool out = false;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += T)
    for (int j = 0; j < length[i]; j++) out |= (uint32_t)index[(int64_t)j * n + i] >= (uint32_t)n;
  if (out) bad[0] = 1;
}

// The row's diagonal and upper entries, absent where it has none.
template <typename Row, typename M>
__global__ __launch_bounds__(kBlock) void k_sym64_build(M A, Sym64 S, double *__restrict__ diag,
                                                        double *__restrict__ up) {
  const int64_t T = (int64_t)gridDim.x * kBlock;
  const int64_t stride = (int64_t)A.n + kSym64Pad;
  const double absent = __builtin_bit_cast(double, kF64Absent);
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < A.n; i += T) {
    const Row row(A, (int)i);
    double d = absent, u[kSym64Pairs];
#pragma unroll
    for (int k = 0; k < kSym64Pairs; k++) u[k] = absent;
    for (int j = 0; j < row.len; j++) {
      const int o = row.col(j) - (int)i;
      if (o < 0) continue;
      const double v = row.value(j);
      if (o == 0) d = v;
#pragma unroll
      for (int k = 0; k < kSym64Pairs; k++)
        if (k < S.pairs && o == S.off[k]) u[k] = v;
    }
    diag[i] = d;
#pragma unroll
    for (int k = 0; k < kSym64Pairs; k++)
      if (k < S.pairs) up[k * stride + i] = u[k];
  }
}

// found[0] = 1 if row i's lower entries are not exactly the upper entries of
// rows i - off[k] that point at i.
template <typename Row, typename M>
__global__ __launch_bounds__(kBlock) void k_sym64_check(M A, Sym64 S, int *__restrict__ found) {
  const int64_t T = (int64_t)gridDim.x * kBlock;
  const int64_t stride = (int64_t)A.n + kSym64Pad;
  bool bad = false;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < A.n; i += T) {
    const Row row(A, (int)i);
    uint64_t low[kSym64Pairs];
#pragma unroll
    for (int k = 0; k < kSym64Pairs; k++) low[k] = kF64Absent;
    for (int j = 0; j < row.len; j++) {
      const int o = (int)i - row.col(j);
      if (o <= 0) break;  // columns ascend
      const uint64_t v = __builtin_bit_cast(uint64_t, row.value(j));
#pragma unroll
      for (int k = 0; k < kSym64Pairs; k++)
        if (k < S.pairs && o == S.off[k]) low[k] = v;
    }
#pragma unroll
    for (int k = 0; k < kSym64Pairs; k++)
      if (k < S.pairs) {
        const uint64_t mirror =
            i >= S.off[k] ? __builtin_bit_cast(uint64_t, S.up[k * stride + i - S.off[k]]) : kF64Absent;
        bad |= low[k] != mirror;
      }
  }
  if (bad) found[0] = 1;
}

int setup_grid(int n) {
  const int64_t g = ((int64_t)n + kBlock - 1) / kBlock;
  return (int)(g < 1 ? 1 : g > 8192 ? 8192 : g);
}

__global__ void k_offsets_reset(int *found) {
  if (threadIdx.x <= kDiaMax) found[threadIdx.x] = threadIdx.x == 0 ? 0 : kFree;
}

template <typename Row, typename M>
hipError_t offsets_t(const M &A, int *found, hipStream_t s) {
  hipLaunchKernelGGL(k_offsets_reset, dim3(1), dim3(64), 0, s, found);
  hipLaunchKernelGGL((k_offsets<Row, M>), dim3(setup_grid(A.n)), dim3(kBlock), 0, s, A, found);
  return hipGetLastError();
}

template <typename Row, typename M>
hipError_t build_t(const M &A, const Sym64 &S, double *diag, double *up, int *found,
                   hipStream_t s) {
  hipLaunchKernelGGL((k_sym64_build<Row, M>), dim3(setup_grid(A.n)), dim3(kBlock), 0, s, A, S, diag,
                     up);
  Sym64 B = S;
  B.diag = diag;
  B.up = up;
  hipLaunchKernelGGL((k_sym64_check<Row, M>), dim3(setup_grid(A.n)), dim3(kBlock), 0, s, A, B, found);
  return hipGetLastError();
}

}  // namespace

hipError_t crs_columns(int n, int nnz, const int *index, int *bad, hipStream_t s) {
  hipLaunchKernelGGL(k_crs_columns, dim3(setup_grid(nnz)), dim3(kBlock), 0, s, n, (int64_t)nnz, index,
                     bad);
  return hipGetLastError();
}
hipError_t ell_columns(int n, const int *length, const int *index, int *bad, hipStream_t s) {
  hipLaunchKernelGGL(k_ell_columns, dim3(setup_grid(n)), dim3(kBlock), 0, s, n, length, index, bad);
  return hipGetLastError();
}
hipError_t matrix_offsets(const Crs<double> &A, int *found, hipStream_t s) {
  return offsets_t<CrsRow>(A, found, s);
}
hipError_t matrix_offsets(const Ell<double> &A, int *found, hipStream_t s) {
  return offsets_t<EllRow>(A, found, s);
}
hipError_t sym64_build(const Crs<double> &A, const Sym64 &S, double *diag, double *up, int *found,
                       hipStream_t s) {
  return build_t<CrsRow>(A, S, diag, up, found, s);
}
hipError_t sym64_build(const Ell<double> &A, const Sym64 &S, double *diag, double *up, int *found,
                       hipStream_t s) {
  return build_t<EllRow>(A, S, diag, up, found, s);
}

}  // namespace cghip

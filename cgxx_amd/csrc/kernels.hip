// HIP kernels of the CG hot path for gfx950 (MI355X).
//
// Every kernel is HBM-bound (SpMV: 2 flop per 12 B in FP64), so the design
// goals are many independent bytes in flight per CU, coalesced streams, no
// re-reads, and no cross-block synchronisation inside a kernel:
//   * CRS SpMV: block-level CSR-stream.  A block of 256 threads owns a row
//     block (<= 256 rows, <= 2048 nonzeros); it issues all index/value loads
//     of the row block at once (8 rounds of 256 coalesced threads), then all
//     x gathers, stages the products in LDS, and every thread adds its row's
//     products left to right -- the per-row order of
//     SerialCG::matvecKernelCRS (serial/SerialCG.cpp:87-95).  Blocks walk
//     row blocks g, g + G, g + 2G, ... (G <= 2048), so the partial sums of a
//     fused dot stay few.
//   * ELL SpMV: one thread per row over column-major slots j*N + i
//     (Matrix.cpp:339-361), 8 slots in flight per thread, 64-bit slot offsets.
//   * Vector kernels: 16-byte loads of element pairs, 4 pairs in flight per
//     thread, grid-stride over pairs.
//   * Reductions: wave64 shift-down fold, four wave sums added in LDS, one
//     partial per block written with a plain store.  The next kernel on the
//     stream folds the partials (every block, same fixed order) before it
//     uses the sum.  A device-scope fence inside the hot kernels would write
//     back and invalidate the XCD's L2 once per block; measured on MI355X it
//     cost ~90 us per 940 MB update pass, so none is used.
//
// Floating-point contraction is off (build flag and pragma): a*x+y is a
// rounded multiply then a rounded add, as in the reference's CPU kernels.

#include "device_common.h"

#include <type_traits>

#pragma clang fp contract(off)

namespace cghip {

namespace {

using namespace dev;

template <typename V, typename X>
__global__ __launch_bounds__(kBlock) void k_matvec_crs(Crs<V> A, const X *__restrict__ x,
                                                       X *__restrict__ y) {
  __shared__ X prod[kNnzCap];
  for (int rb = blockIdx.x; rb < A.nrb; rb += gridDim.x) crs_rowblock<V, X, false>(A, x, y, rb, prod);
}

template <typename V, typename X, bool O32>
__global__ __launch_bounds__(kBlock) void k_matvec_ell(Ell<V> A, const X *__restrict__ x,
                                                       X *__restrict__ y) {
  const int nrb = (A.n + kBlock - 1) / kBlock;
  for (int rb = blockIdx.x; rb < nrb; rb += gridDim.x) ell_rowblock<V, X, false, O32>(A, x, y, rb);
}

// First kernel of an iteration: copies the loop scalars `next` -> `cur`
// (block 0), stops at CG_MAX_ITER (CG.cpp:323), else q = A p with the
// partials of <p,q> (CG.cpp:325-328).  Returns false if the iteration is off.
__device__ inline bool begin_iteration(SolveState *st) {
  const Scalars s = st->next;
  // Also when already done: the later kernels of this iteration read `cur`.
  const bool stop = s.done || s.iteration >= st->max_iter;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    Scalars c = s;
    if (stop) c.done = 1;
    st->cur = c;
  }
  return !stop;
}

// One block per row block (not a persistent grid: the hardware keeps new
// blocks streaming while others finish, 334 against 376 us at 256^3 for the
// CRS kernel), one partial of <p,q> per block; k_fold_groups then folds
// them in groups of 256 before the r update reads them.  Consecutive row
// blocks on consecutive XCDs (the dispatch order) measured faster than
// giving each XCD a contiguous range of row blocks (382 vs 402 us at
// 256^3; ELL 338 vs 359 us).
__global__ __launch_bounds__(kBlock) void k_pcg_matvec_dot_crs(Crs<double> A, const double *__restrict__ p,
                                                               double *__restrict__ q, Partials pq,
                                                               SolveState *st) {
  __shared__ double prod[kNnzCap];
  __shared__ double lds[4];
  if (!begin_iteration(st)) return;
  const double t = crs_rowblock<double, double, true>(A, p, q, blockIdx.x, prod);
  const double bp = block_fold(t, lds);
  if (threadIdx.x == 0) pq.a[blockIdx.x] = bp;
}

template <bool O32>
__global__ __launch_bounds__(kBlock) void k_pcg_matvec_dot_ell(Ell<double> A, const double *__restrict__ p,
                                                               double *__restrict__ q, Partials pq,
                                                               SolveState *st) {
  __shared__ double lds[4];
  if (!begin_iteration(st)) return;
  const double t = ell_rowblock<double, double, true, O32>(A, p, q, blockIdx.x);
  const double bp = block_fold(t, lds);
  if (threadIdx.x == 0) pq.a[blockIdx.x] = bp;
}

// Chunk of kBlock rows that block b of the symmetric kernels takes, or -1.
// Blocks are dispatched to the 8 XCDs round robin; each XCD gets a contiguous
// eighth of the chunks, so that a row's neighbours along the nearer diagonals
// are still in that XCD's L2 (chunks in dispatch order: 256^3 ELL iteration
// 430 against 418 us; in strips of the planes on top: no difference).
__device__ inline int sym64_chunk(int n, int b) {
  const int nrb = ell_chunks(n), x = b & 7, per = (nrb + 7) >> 3;
  const int q = x * per + (b >> 3);
  return q < min(nrb, (x + 1) * per) ? q : -1;
}

// Element i of a vector of at most 2^32 bytes.
__device__ inline double elem(const double *__restrict__ v, int i) {
  return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(v) + (uint32_t)i * 8u);
}

// Row r of the symmetric diagonals: lower entries from the farthest, the
// diagonal, the upper entries, added left to right from 0 -- the order of a
// row with ascending columns.  Every load is issued before any is used: the
// addresses are clamped into the streams, and an entry that is absent or
// would lie outside the matrix is dropped by a select.  NT: the diagonal,
// the only stream read once, is loaded non-temporally (sym64_launch).  Bound
// by memory: 48 bytes a row with three pairs against 100 from the uploaded
// arrays; 256^3 product in the loop 303 -> 186 us (5.1 TB/s of the 950 MB
// that the counters show, 1.2 times the bytes it needs), 128^3 40 -> 17 us.
template <int P>
struct Sym64Loads {
  double d, lo[P], hi[P];
};

template <int P, bool NT = false>
__device__ inline void sym64_load(const Sym64 &A, int r, Sym64Loads<P> &l) {
  l.d = NT ? __builtin_nontemporal_load(A.diag + r) : A.diag[r];
#pragma unroll
  for (int k = 0; k < P; k++) {
    const double *u = A.up + k * ((int64_t)A.n + kSym64Pad);
    l.hi[k] = elem(u, r);
    l.lo[k] = elem(u, max(r - A.off[k], 0));
  }
}

// xl, xh: x at r - off[k] and r + off[k].
template <int P>
__device__ inline double sym64_sum(const Sym64 &A, const Sym64Loads<P> &l, const double *xl,
                                   const double *xh, double xr, int r) {
  auto live = [](double v) { return __builtin_bit_cast(uint64_t, v) != kF64Absent; };
  double s = 0.0;
#pragma unroll
  for (int k = P - 1; k >= 0; k--) {
    const double t = s + l.lo[k] * xl[k];
    s = live(l.lo[k]) && r >= A.off[k] ? t : s;
  }
  {
    const double t = s + l.d * xr;
    s = live(l.d) ? t : s;
  }
#pragma unroll
  for (int k = 0; k < P; k++) {
    const double t = s + l.hi[k] * xh[k];
    s = live(l.hi[k]) ? t : s;
  }
  return s;
}

template <int P, bool NT>
__device__ inline double sym64_row(const Sym64 &A, const double *__restrict__ x, int r, double &xr) {
  Sym64Loads<P> l;
  double xl[P], xh[P];
  sym64_load<P, NT>(A, r, l);
  xr = elem(x, r);
#pragma unroll
  for (int k = 0; k < P; k++) {
    xl[k] = elem(x, max(r - A.off[k], 0));
    xh[k] = elem(x, min(r + A.off[k], A.n - 1));
  }
  return sym64_sum<P>(A, l, xl, xh, xr, r);
}

template <int P, bool NT>
__global__ __launch_bounds__(kBlock) void k_matvec_sym64(Sym64 A, const double *__restrict__ x,
                                                         double *__restrict__ y) {
  const int c = sym64_chunk(A.n, blockIdx.x);
  const int r = c * kBlock + (int)threadIdx.x;
  if (c < 0 || r >= A.n) return;
  double xr;
  y[r] = sym64_row<P, NT>(A, x, r, xr);
}

// One partial of <p,q> per chunk, as from k_pcg_matvec_dot_crs and _ell.
template <int P, bool NT>
__global__ __launch_bounds__(kBlock) void k_pcg_matvec_dot_sym64(Sym64 A, const double *__restrict__ p,
                                                                 double *__restrict__ q, Partials pq,
                                                                 SolveState *st) {
  __shared__ double lds[4];
  if (!begin_iteration(st)) return;
  const int c = sym64_chunk(A.n, blockIdx.x);
  if (c < 0) return;
  const int r = c * kBlock + (int)threadIdx.x;
  double t = 0.0;
  if (r < A.n) {
    double pr;
    const double s = sym64_row<P, NT>(A, p, r, pr);
    q[r] = s;
    t = pr * s;
  }
  const double bp = block_fold(t, lds);
  if (threadIdx.x == 0) pq.a[c] = bp;
}

// Group fold: block g folds partials g*256 .. g*256+255 (zero past G) into
// out[g], so that the next kernel folds ceil(G / 256) values instead of G.
__global__ __launch_bounds__(kBlock) void k_fold_groups(const double *__restrict__ in, int G,
                                                        double *__restrict__ out) {
  __shared__ double lds[4];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  const double s = block_fold(i < G ? in[i] : 0.0, lds);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// ---------------------------------------------------------------------------
// Vector kernels.  Element pairs (2q, 2q+1); thread gid of T = 256*G visits
// pairs gid, gid + T, ... in order, element 2q before 2q+1.  The last pair
// of an odd-length vector holds one element.

struct Pairs2 {
  double2 a, b;
};
struct Pairs3 {
  double2 a, b, c;
};
struct Pairs4 {
  double2 a, b, c, d;
};

__global__ __launch_bounds__(kBlock) void k_axpy(int n, double a, const double *__restrict__ x,
                                                 double *__restrict__ y) {
  const Pairs P(n);
  trips<kUnroll>(P, [=](int64_t j) { return Pairs2{v2(x)[j], v2(y)[j]}; })
      .run([&](int64_t j, Pairs2 &v) {
        v.b.x = v.b.x + a * v.a.x;
        v.b.y = v.b.y + a * v.a.y;
        v2(y)[j] = v.b;
      });
  if (owns_rest(P, P.npair)) y[n - 1] = y[n - 1] + a * x[n - 1];
}

__global__ __launch_bounds__(kBlock) void k_xpay(int n, const double *__restrict__ x, double a,
                                                 double *__restrict__ y) {
  const Pairs P(n);
  trips<kUnroll>(P, [=](int64_t j) { return Pairs2{v2(x)[j], v2(y)[j]}; })
      .run([&](int64_t j, Pairs2 &v) {
        v.b.x = v.a.x + a * v.b.x;
        v.b.y = v.a.y + a * v.b.y;
        v2(y)[j] = v.b;
      });
  if (owns_rest(P, P.npair)) y[n - 1] = x[n - 1] + a * y[n - 1];
}

__global__ __launch_bounds__(kBlock) void k_jacobi(int n, const double *__restrict__ C,
                                                   const double *__restrict__ x, double *__restrict__ y) {
  const Pairs P(n);
  trips<kUnroll>(P, [=](int64_t j) { return Pairs2{v2(C)[j], v2(x)[j]}; })
      .run([&](int64_t j, Pairs2 &v) {
        v2(y)[j] = make_double2(v.a.x * v.b.x, v.a.y * v.b.y);
      });
  if (owns_rest(P, P.npair)) y[n - 1] = C[n - 1] * x[n - 1];
}

__global__ __launch_bounds__(kBlock) void k_fill(int n, double v, double *__restrict__ y) {
  const int64_t T = (int64_t)gridDim.x * kBlock;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += T) y[i] = v;
}

__global__ __launch_bounds__(kBlock) void k_dot_partials(int n, const double *__restrict__ a,
                                                         const double *__restrict__ b, Partials pa) {
  __shared__ double lds[4];
  const Pairs P(n);
  double s = 0.0;
  trips<kUnroll>(P, [=](int64_t j) { return Pairs2{v2(a)[j], v2(b)[j]}; })
      .run([&](int64_t, Pairs2 &v) {
        s += v.a.x * v.b.x;
        s += v.a.y * v.b.y;
      });
  if (owns_rest(P, P.npair)) s += a[n - 1] * b[n - 1];
  const double bp = block_fold(s, lds);
  if (threadIdx.x == 0) pa.a[blockIdx.x] = bp;
}

__global__ __launch_bounds__(kBlock) void k_residual_partials(int n, const double *__restrict__ b,
                                                              const double *__restrict__ q,
                                                              Partials pa) {
  __shared__ double lds[4];
  Pairs P(n);
  double s_rr = 0.0, s_bb = 0.0;
  for (; P.q < P.npair; P.q += P.T) {
    for (int64_t e = 2 * P.q; e < 2 * P.q + 2 && e < n; e++) {
      const double ri = b[e] - q[e];
      s_rr += ri * ri;
      s_bb += b[e] * b[e];
    }
  }
  const double b0 = block_fold(s_rr, lds);
  const double b1 = block_fold(s_bb, lds);
  if (threadIdx.x == 0) {
    pa.a[blockIdx.x] = b0;
    pa.b[blockIdx.x] = b1;
  }
}

// One block: out[0] = fold(pa.a), out[1] = fold(pa.b) (if two_sums).
__global__ __launch_bounds__(kBlock) void k_fold_out(Partials pa, int G, int two_sums, double *out) {
  __shared__ double lds[4];
  const double s0 = fold_partials(pa.a, G, lds);
  const double s1 = two_sums ? fold_partials(pa.b, G, lds) : 0.0;
  if (threadIdx.x == 0) {
    out[0] = s0;
    if (two_sums) out[1] = s1;
  }
}

// k_dot_partials and k_fold_out in one block of 1,024 threads, for vectors of
// 1 element to kDotSmall pairs per thread (its loads are clamped to the last
// element, so an empty vector, whose pointers may be null, takes the two): the loop of hooks waits for every dot,
// and a launch costs more than the rest of it (4,096 elements 13.7 us a call
// against 16.1 with two kernels, 8,192 14.7, 16,384 17.0 against 16.1).  Wave
// sums, partials and their fold are those of the two kernels, one pair per
// thread of theirs.
constexpr int kDotSmall = 4;
__global__ __launch_bounds__(1024) void k_dot_small(int n, const double *__restrict__ a,
                                                    const double *__restrict__ b, int G,
                                                    double *__restrict__ out) {
  __shared__ double sums[4 * kDotSmall][4];
  const int t = threadIdx.x, lane = t & 63;
  double s[kDotSmall];
#pragma unroll
  for (int u = 0; u < kDotSmall; u++) {
    s[u] = 0.0;
    if (4 * u < G) {
      const int e = 2 * (u * 1024 + t), e0 = min(e, n - 1), e1 = min(e + 1, n - 1);
      const double p0 = a[e0] * b[e0], p1 = a[e1] * b[e1];
      s[u] = e < n ? 0.0 + p0 : 0.0;
      s[u] = e + 1 < n ? s[u] + p1 : s[u];
    }
  }
#pragma unroll
  for (int u = 0; u < kDotSmall; u++) {
    if (4 * u < G) {
      const double w = wave_fold(s[u]);
      if (lane == 0) sums[4 * u + (t >> 8)][(t >> 6) & 3] = w;
    }
  }
  __syncthreads();
  if (t >= 64) return;
  const int g = min(lane, G - 1);
  const double p = ((sums[g][0] + sums[g][1]) + sums[g][2]) + sums[g][3];
  const double w = wave_fold(lane < G ? 0.0 + p : 0.0);
  if (lane == 0) *out = ((w + 0.0) + 0.0) + 0.0;
}

// One wave: lanes form 64 products at a time, every lane then adds them in
// index order (the shuffle source is wave-uniform).
__global__ __launch_bounds__(64) void k_dot_serial(int n, const double *__restrict__ a,
                                                   const double *__restrict__ b, double *out) {
  const int lane = threadIdx.x;
  double s = 0.0;
  for (int base = 0; base < n; base += 64) {
    const int i = base + lane;
    const double pr = i < n ? a[i] * b[i] : 0.0;
    const int m = min(64, n - base);
    for (int j = 0; j < m; j++) s += __shfl(pr, j, 64);
  }
  if (lane == 0) *out = s;
}

// r = k + (-1) r (xpay(K, -1, R), CG.cpp:295); p = C o r or p = r
// (CG.cpp:297-303); partials of <r,r> and <p,r> (CG.cpp:305-318).
template <bool JAC>
__global__ __launch_bounds__(kBlock) void k_pcg_init(int n, const double *__restrict__ k,
                                                     double *__restrict__ r, double *__restrict__ p,
                                                     const double *__restrict__ C, Partials pa) {
  __shared__ double lds[4];
  const Pairs P(n);
  double s_rr = 0.0, s_pr = 0.0;
  auto init = [&](double ke, double ce, double &re, double &pe) {
    re = ke + (-1.0) * re;
    pe = JAC ? ce * re : re;
    s_rr += re * re;
    s_pr += pe * re;
  };
  trips<kUnroll>(P, [=](int64_t j) {
    return Pairs3{v2(k)[j], v2(r)[j], JAC ? v2(C)[j] : make_double2(0.0, 0.0)};
  }).run([&](int64_t j, Pairs3 &v) {
    double2 pv;
    init(v.a.x, v.c.x, v.b.x, pv.x);
    init(v.a.y, v.c.y, v.b.y, pv.y);
    v2(r)[j] = v.b;
    v2(p)[j] = pv;
  });
  if (owns_rest(P, P.npair)) init(k[n - 1], JAC ? C[n - 1] : 0.0, r[n - 1], p[n - 1]);
  const double b0 = block_fold(s_rr, lds);
  const double b1 = block_fold(s_pr, lds);
  if (threadIdx.x == 0) {
    pa.a[blockIdx.x] = b0;
    pa.b[blockIdx.x] = b1;
  }
}

// One block: r2, rho and nrm2_0 = sqrt(r2) before the loop (CG.cpp:305-318).
template <bool JAC>
__global__ __launch_bounds__(kBlock) void k_pcg_init_finish(Partials pa, int G, SolveState *st,
                                                            History h) {
  __shared__ double lds[4];
  double r2, pr;
  fold_partials2(pa.a, G, pa.b, G, lds, r2, pr);
  if (threadIdx.x == 0) {
    Scalars s{};
    s.r2 = r2;
    s.rho = JAC ? pr : r2;
    s.residual = 1.0;
    s.iteration = 0;
    s.done = 0;
    st->next = s;
    st->cur = s;
    st->nrm2_0 = sqrt(r2);
    if (h.r2 && h.cap > 0) h.r2[0] = r2;
    if (h.rho && h.cap > 0) h.rho[0] = s.rho;
  }
}

// Fold of G <= kFoldDirect partials as k_fold_groups and then fold_partials
// over its group sums give it (adding 0.0 as they do), every load in flight
// at once and one barrier.
__device__ __forceinline__ double fold_two_levels(const double *__restrict__ partial, int G,
                                         double (*lds)[4]) {
  constexpr int M = kFoldDirect / kBlock;
  const int t = threadIdx.x, lane = t & 63, groups = (G + kBlock - 1) / kBlock;
  double v[M];
#pragma unroll
  for (int g = 0; g < M; g++) v[g] = partial[min(g * kBlock + t, G - 1)];
#pragma unroll
  for (int g = 0; g < M; g++) {
    if (g < groups) {
      const double w = wave_fold(g * kBlock + t < G ? v[g] : 0.0);
      if (lane == 0) lds[g][t >> 6] = w;
    }
  }
  __syncthreads();
  const int g = min(lane, groups - 1);
  const double sum = 0.0 + (((lds[g][0] + lds[g][1]) + lds[g][2]) + lds[g][3]);
  const double w = wave_fold(lane < groups ? sum : 0.0);
  __syncthreads();
  return lane_first(w) + 0.0;
}

template <bool JAC>
__device__ inline void update_elem(double &rv, double qv, double cv, double na, double &s_rr,
                                   double &s_rz) {
  rv = rv + na * qv;
  const double zv = JAC ? cv * rv : rv;
  s_rr += rv * rv;
  s_rz += rv * zv;
}
// a = rho / <p,q> (CG.cpp:334), kept in st->alpha; r += (-a) q (CG.cpp:342;
// the x += a p of CG.cpp:340 is done by the last kernel, which reads p
// anyway); partials of <r,r> and <r,z> with z = C o r (CG.cpp:344, 363-366).
// gpq > 0: <p,q> folds the gpq group sums in ppq.a (k_fold_groups).
// gpq = -G (G <= kFoldDirect, small systems, one launch fewer per iteration):
// the block folds the G SpMV partials themselves, to the same bits.
template <bool JAC, bool NT>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8))) void k_pcg_update(
    int n, int gpq, double *__restrict__ r, const double *__restrict__ q,
    const double *__restrict__ C, Partials ppq, Partials prr, SolveState *st, History h) {
  __shared__ double lds[4];
  __shared__ double lds2[kFoldDirect / kBlock][4];
  const Pairs P(n);
  auto pairs = trips<2>(P, [=](int64_t j) {
    return Pairs3{v2(r)[j], NT ? v2_stream(q, j) : v2(q)[j],
                  !JAC ? make_double2(0.0, 0.0) : NT ? v2_stream(C, j) : v2(C)[j]};
  });
  const Scalars c = st->cur;
  if (c.done) return;
  const double pq =
      gpq > 0 ? fold_partials(ppq.a, gpq, lds) : fold_two_levels(ppq.a, -gpq, lds2);
  const double a = c.rho / pq;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->alpha = a;
    if (h.pq && c.iteration < h.cap) h.pq[c.iteration] = pq;
    if (h.alpha && c.iteration < h.cap) h.alpha[c.iteration] = a;
  }
  const double na = -a;
  double s_rr = 0.0, s_rz = 0.0;
  pairs.run([&](int64_t j, Pairs3 &v) {
    update_elem<JAC>(v.a.x, v.b.x, v.c.x, na, s_rr, s_rz);
    update_elem<JAC>(v.a.y, v.b.y, v.c.y, na, s_rr, s_rz);
    v2(r)[j] = v.a;
  });
  if (owns_rest(P, P.npair)) {
    double re = r[n - 1];
    update_elem<JAC>(re, q[n - 1], JAC ? C[n - 1] : 0.0, na, s_rr, s_rz);
    r[n - 1] = re;
  }
  const double b0 = block_fold(s_rr, lds);
  const double b1 = block_fold(s_rz, lds);
  if (threadIdx.x == 0) {
    prr.a[blockIdx.x] = b0;
    prr.b[blockIdx.x] = b1;
  }
}
// End of iteration c: the stop test (CG.cpp:344-355), true if it converged;
// block 0 writes `next` and the history.
__device__ inline bool end_iteration(SolveState *st, const Scalars &c, double r2, double rho,
                                     double b, const History &h) {
  const double res = sqrt(r2) / st->nrm2_0;
  const bool converged = res <= st->tol;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const int it = c.iteration;
    Scalars s = c;
    s.r2 = r2;
    s.residual = res;
    s.iteration = it + 1;
    if (h.r2 && it + 1 < h.cap) h.r2[it + 1] = r2;
    // The reference computes rho and beta only when the loop goes on
    // (CG.cpp:357-370): after the converging iteration their entries are NaN.
    const double nan = __builtin_nan("");
    if (h.rho && it + 1 < h.cap) h.rho[it + 1] = converged ? nan : rho;
    if (h.beta && it < h.cap) h.beta[it] = converged ? nan : b;
    if (converged) {
      s.done = 1;
    } else {
      s.rho = rho;
      s.beta = b;
    }
    st->next = s;
  }
  return converged;
}

// Last kernel of an iteration: x += a p with the old p (CG.cpp:340); r2 and
// the stop test (CG.cpp:344-355); if not converged rho = <r,z>,
// b = rho / rho_old (CG.cpp:357-370) and p = z + b p with z = C o r
// recomputed (CG.cpp:375-381).  Writes `next`.
template <bool JAC, bool NT>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8))) void k_pcg_xpay(
    int n, double *__restrict__ x, double *__restrict__ p, const double *__restrict__ r,
    const double *__restrict__ C, Partials prr, SolveState *st, History h) {
  __shared__ double lds[4];
  const Pairs P(n);
  auto pairs = trips<2>(P, [=](int64_t j) {
    return Pairs4{NT ? v2_stream(x, j) : v2(x)[j], v2(p)[j], NT ? v2_stream(r, j) : v2(r)[j],
                  !JAC ? make_double2(0.0, 0.0) : NT ? v2_stream(C, j) : v2(C)[j]};
  });
  const Scalars c = st->cur;
  if (c.done) return;
  const int G = gridDim.x;  // the update kernel ran on the same grid
  double r2, rz;
  fold_partials2<4>(prr.a, G, prr.b, G, lds, r2, rz);
  const double rho = JAC ? rz : r2;
  const double b = rho / c.rho;
  const double a = st->alpha;
  const bool converged = end_iteration(st, c, r2, rho, b, h);
  // x += a p always; p = z + b p unless the loop stops here.  Four streams
  // per element: unrolled twice to stay within 64 VGPRs.  NT: x, r and C are
  // streamed non-temporally, so that p stays cached for the next SpMV.
  if (converged) {
    for (int64_t g = P.q; g < P.npair; g += P.T)
      for (int64_t e = 2 * g; e < 2 * g + 2 && e < n; e++) x[e] = x[e] + a * p[e];
    return;
  }
  pairs.run([&](int64_t j, Pairs4 &v) {
    v.a.x = v.a.x + a * v.b.x;
    v.a.y = v.a.y + a * v.b.y;
    const double zx = JAC ? v.d.x * v.c.x : v.c.x;
    const double zy = JAC ? v.d.y * v.c.y : v.c.y;
    v.b.x = zx + b * v.b.x;
    v.b.y = zy + b * v.b.y;
    if (NT)
      v2_store_stream(x, j, v.a);
    else
      v2(x)[j] = v.a;
    v2(p)[j] = v.b;
  });
  if (owns_rest(P, P.npair)) {
    const double pe = p[n - 1];
    x[n - 1] = x[n - 1] + a * pe;
    const double ze = JAC ? C[n - 1] * r[n - 1] : r[n - 1];
    p[n - 1] = ze + b * pe;
  }
}

// ---------------------------------------------------------------------------
// The loop of small systems on the symmetric diagonals: two kernels an
// iteration instead of three.  Each kernel's time is its launch and one chain
// of latencies (state and partials, fold, vectors, fold, store), so every load
// is issued before the first fold, and a kernel of an iteration that is off
// is told apart only where it would store.  Iteration with three kernels and
// with two: 256 x 256 12.5 and 8.0 us (9.9 with the vectors loaded after the
// fold), 61 x 47 x 53 15.6 and 11.8, 64^3 17.2 and 14.1; with more than a
// chunk per block the neighbours' r, C and p cost more than the launch:
// 80^3 26.5 and 27.5, 128^3 56 and 65.

// Sums over the block of two values, as block_fold gives each; one barrier,
// lds used once.
__device__ inline void block_fold2(double &a, double &b, double (*lds)[4]) {
  a = wave_fold(a);
  b = wave_fold(b);
  if ((threadIdx.x & 63) == 0) {
    lds[0][threadIdx.x >> 6] = a;
    lds[1][threadIdx.x >> 6] = b;
  }
  __syncthreads();
  a = ((lds[0][0] + lds[0][1]) + lds[0][2]) + lds[0][3];
  b = ((lds[1][0] + lds[1][1]) + lds[1][2]) + lds[1][3];
}

// k_pcg_update for at most one pair per thread, as the iteration's first
// kernel: copies the loop scalars `next` -> `cur` and stops at CG_MAX_ITER
// (CG.cpp:323).
template <bool JAC>
__global__ __launch_bounds__(kBlock) void k_pcg_update_small(int n, int G, double *__restrict__ r,
                                                             const double *__restrict__ q,
                                                             const double *__restrict__ C,
                                                             const double *__restrict__ ppq,
                                                             Partials prr, SolveState *st, History h) {
  __shared__ double lds[2][4];
  __shared__ double lds2[kFoldDirect / kBlock][4];
  const int e = 2 * (blockIdx.x * kBlock + (int)threadIdx.x);
  const int e0 = min(e, n - 1), e1 = min(e + 1, n - 1);
  double r0 = r[e0], r1 = r[e1];
  const double q0 = q[e0], q1 = q[e1];
  const double c0 = JAC ? C[e0] : 0.0, c1 = JAC ? C[e1] : 0.0;
  // field by field: as a struct it took stack, whose move to LDS reads the
  // dispatch packet in host memory (12 us a kernel instead of 4)
  const double rho = st->next.rho, r2 = st->next.r2, res = st->next.residual, beta = st->next.beta;
  const int it = st->next.iteration;
  const bool off = st->next.done || it >= st->max_iter;
  const double pq = fold_two_levels(ppq, G, lds2);
  const double a = rho / pq;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->cur.rho = rho;
    st->cur.r2 = r2;
    st->cur.residual = res;
    st->cur.beta = beta;
    st->cur.iteration = it;
    st->cur.done = off;
  }
  if (off) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->alpha = a;
    if (h.pq && it < h.cap) h.pq[it] = pq;
    if (h.alpha && it < h.cap) h.alpha[it] = a;
  }
  double s_rr = 0.0, s_rz = 0.0;
  if (e < n) {
    update_elem<JAC>(r0, q0, c0, -a, s_rr, s_rz);
    r[e] = r0;
  }
  if (e + 1 < n) {
    update_elem<JAC>(r1, q1, c1, -a, s_rr, s_rz);
    r[e + 1] = r1;
  }
  block_fold2(s_rr, s_rz, lds);
  if (threadIdx.x == 0) {
    prr.a[blockIdx.x] = s_rr;
    prr.b[blockIdx.x] = s_rz;
  }
}

// k_pcg_xpay and the next iteration's k_pcg_matvec_dot_sym64: the product
// takes p = C r + b p of a row's neighbours from r, C and the old p, the
// values that k_pcg_xpay would store, and the new p goes to a buffer of its
// own (neighbours read the old one).  At max_iter the last iteration's x and
// p are still formed, q is left.  G <= 2 kBlock partials of the update.
template <int P, bool JAC>
__global__ __launch_bounds__(kBlock) void k_pcg_step_sym64(
    Sym64 A, double *__restrict__ x, const double *__restrict__ p, double *__restrict__ pnext,
    double *__restrict__ q, const double *__restrict__ r, const double *__restrict__ C,
    Partials prr, int G, Partials pq, SolveState *st, History h) {
  __shared__ double lds[2][4], lds2[4];
  const int chunk = sym64_chunk(A.n, blockIdx.x);
  if (chunk < 0) return;
  const int t = threadIdx.x, i = chunk * kBlock + t, row = min(i, A.n - 1);
  double ra[2], rb[2];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    ra[u] = prr.a[min(t + u * kBlock, G - 1)];
    rb[u] = prr.b[min(t + u * kBlock, G - 1)];
  }
  const Scalars c = st->cur;
  const double a = st->alpha, xi = x[row];
  Sym64Loads<P> l;
  sym64_load<P>(A, row, l);
  double z[2 * P + 1], po[2 * P + 1];
#pragma unroll
  for (int k = 0; k < 2 * P + 1; k++) {
    const int m = k < P ? max(row - A.off[k], 0) : k < 2 * P ? min(row + A.off[k - P], A.n - 1) : row;
    z[k] = JAC ? elem(C, m) * elem(r, m) : elem(r, m);
    po[k] = elem(p, m);
  }
  double r2 = 0.0, rz = 0.0;
#pragma unroll
  for (int u = 0; u < 2; u++) {
    r2 = t + u * kBlock < G ? r2 + ra[u] : r2;
    rz = t + u * kBlock < G ? rz + rb[u] : rz;
  }
  block_fold2(r2, rz, lds);
  if (c.done) return;
  const double rho = JAC ? rz : r2;
  const double b = rho / c.rho;
  const bool converged = end_iteration(st, c, r2, rho, b, h);
  const bool goes_on = !converged && c.iteration + 1 < st->max_iter;
  if (i < A.n) {
    x[i] = xi + a * po[2 * P];
    if (!converged) pnext[i] = z[2 * P] + b * po[2 * P];
  }
  if (!goes_on) return;
  double pn[2 * P + 1];
#pragma unroll
  for (int k = 0; k < 2 * P + 1; k++) pn[k] = z[k] + b * po[k];
  const double s = sym64_sum<P>(A, l, pn, pn + P, pn[2 * P], row);
  double dot = 0.0;
  if (i < A.n) {
    q[i] = s;
    dot = pn[2 * P] * s;
  }
  const double bp = block_fold(dot, lds2);
  if (t == 0) pq.a[chunk] = bp;
}

}  // namespace

// ---------------------------------------------------------------------------
// Host-side helpers and launches.

int crs_rowblocks(int n, const int *ptr, int *starts) {
  int nb = 0, r = 0;
  while (r < n) {
    const int r0 = r;
    r++;
    while (r < n && r - r0 < kRowsMax && ptr[r + 1] - ptr[r0] <= kNnzCap) r++;
    starts[nb++] = r0;
  }
  starts[nb] = n;
  return nb;
}

static inline dim3 vgrid(int n) { return dim3(vec_grid(n)); }

template <typename V, typename X>
hipError_t matvec_crs_t(const Crs<V> &A, const X *x, X *y, hipStream_t s) {
  if (A.n == 0) return hipSuccess;
  // no reduction: one block per row block (more waves in flight than the
  // persistent grid of the fused kernels)
  hipLaunchKernelGGL((k_matvec_crs<V, X>), dim3(A.nrb > 0 ? A.nrb : 1), dim3(kBlock), 0, s, A, x,
                     y);
  return hipGetLastError();
}

template <typename V, typename X>
hipError_t matvec_ell_t(const Ell<V> &A, const X *x, X *y, hipStream_t s) {
  if (A.n == 0) return hipSuccess;
  const dim3 grid(ell_chunks(A.n) > 0 ? ell_chunks(A.n) : 1);
  if (ell_o32(A))
    hipLaunchKernelGGL((k_matvec_ell<V, X, true>), grid, dim3(kBlock), 0, s, A, x, y);
  else
    hipLaunchKernelGGL((k_matvec_ell<V, X, false>), grid, dim3(kBlock), 0, s, A, x, y);
  return hipGetLastError();
}

hipError_t matvec_crs(const Crs<double> &A, const double *x, double *y, hipStream_t s) {
  return matvec_crs_t<double, double>(A, x, y, s);
}

hipError_t matvec_ell(const Ell<double> &A, const double *x, double *y, hipStream_t s) {
  return matvec_ell_t<double, double>(A, x, y, s);
}

hipError_t axpy(int n, double a, const double *x, double *y, hipStream_t s) {
  hipLaunchKernelGGL(k_axpy, vgrid(n), dim3(kBlock), 0, s, n, a, x, y);
  return hipGetLastError();
}

hipError_t xpay(int n, const double *x, double a, double *y, hipStream_t s) {
  hipLaunchKernelGGL(k_xpay, vgrid(n), dim3(kBlock), 0, s, n, x, a, y);
  return hipGetLastError();
}

hipError_t jacobi(int n, const double *C, const double *x, double *y, hipStream_t s) {
  hipLaunchKernelGGL(k_jacobi, vgrid(n), dim3(kBlock), 0, s, n, C, x, y);
  return hipGetLastError();
}

hipError_t fill(int n, double v, double *y, hipStream_t s) {
  hipLaunchKernelGGL(k_fill, vgrid(n), dim3(kBlock), 0, s, n, v, y);
  return hipGetLastError();
}

hipError_t dot_tree(int n, const double *a, const double *b, Partials pa, double *out,
                    hipStream_t s) {
  const int G = vec_grid(n);
  if (n > 0 && G <= 4 * kDotSmall) {
    hipLaunchKernelGGL(k_dot_small, dim3(1), dim3(1024), 0, s, n, a, b, G, out);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_dot_partials, vgrid(n), dim3(kBlock), 0, s, n, a, b, pa);
  hipLaunchKernelGGL(k_fold_out, dim3(1), dim3(kBlock), 0, s, pa, vec_grid(n), 0, out);
  return hipGetLastError();
}

hipError_t residual_norms(int n, const double *b, const double *q, Partials pa, double *out,
                          hipStream_t s) {
  hipLaunchKernelGGL(k_residual_partials, vgrid(n), dim3(kBlock), 0, s, n, b, q, pa);
  hipLaunchKernelGGL(k_fold_out, dim3(1), dim3(kBlock), 0, s, pa, vec_grid(n), 1, out);
  return hipGetLastError();
}

hipError_t dot_serial(int n, const double *a, const double *b, double *out, hipStream_t s) {
  hipLaunchKernelGGL(k_dot_serial, dim3(1), dim3(64), 0, s, n, a, b, out);
  return hipGetLastError();
}

hipError_t pcg_init(int n, const double *k, double *r, double *p, const double *C, Partials pa,
                    SolveState *st, History h, hipStream_t s) {
  if (C) {
    hipLaunchKernelGGL(k_pcg_init<true>, vgrid(n), dim3(kBlock), 0, s, n, k, r, p, C, pa);
    hipLaunchKernelGGL(k_pcg_init_finish<true>, dim3(1), dim3(kBlock), 0, s, pa, vec_grid(n), st, h);
  } else {
    hipLaunchKernelGGL(k_pcg_init<false>, vgrid(n), dim3(kBlock), 0, s, n, k, r, p, C, pa);
    hipLaunchKernelGGL(k_pcg_init_finish<false>, dim3(1), dim3(kBlock), 0, s, pa, vec_grid(n), st, h);
  }
  return hipGetLastError();
}

// SpMV + <p,q> partials into pq.a (one per row block), then their group
// sums into pq2 (fold_groups(G) entries).
hipError_t pcg_matvec_dot_crs(const Crs<double> &A, const double *p, double *q, Partials pq,
                              double *pq2, SolveState *st, hipStream_t s) {
  const int G = A.nrb > 0 ? A.nrb : 1;
  hipLaunchKernelGGL(k_pcg_matvec_dot_crs, dim3(G), dim3(kBlock), 0, s, A, p, q, pq, st);
  if (pq2)
    hipLaunchKernelGGL(k_fold_groups, dim3(fold_groups(G)), dim3(kBlock), 0, s, pq.a, G, pq2);
  return hipGetLastError();
}

hipError_t pcg_matvec_dot_ell(const Ell<double> &A, const double *p, double *q, Partials pq,
                              double *pq2, SolveState *st, hipStream_t s) {
  const int G = ell_chunks(A.n) > 0 ? ell_chunks(A.n) : 1;
  if (ell_o32(A))
    hipLaunchKernelGGL(k_pcg_matvec_dot_ell<true>, dim3(G), dim3(kBlock), 0, s, A, p, q, pq, st);
  else
    hipLaunchKernelGGL(k_pcg_matvec_dot_ell<false>, dim3(G), dim3(kBlock), 0, s, A, p, q, pq, st);
  if (pq2)
    hipLaunchKernelGGL(k_fold_groups, dim3(fold_groups(G)), dim3(kBlock), 0, s, pq.a, G, pq2);
  return hipGetLastError();
}

// f(grid, pairs, non-temporal diagonal) of the symmetric kernels.  The
// diagonal is streamed past the caches once a product's own bytes, 8 (3 +
// pairs) a row, outgrow the 256 MB last-level cache: FP64 iteration at 160^3
// 102.7 cached against 111.2 us, at 180^3 159 against 152, at 256^3 438
// against 418.
template <typename F>
static hipError_t sym64_launch(const Sym64 &A, F f) {
  if (A.pairs < 1 || A.pairs > kSym64Pairs) return hipErrorInvalidValue;
  const dim3 grid(8 * ((ell_chunks(A.n) + 7) / 8));
  const bool nt = 8 * (3 + (int64_t)A.pairs) * A.n > (int64_t(1) << 28);
  auto pick = [&](auto pairs) {
    nt ? f(grid, pairs, std::true_type()) : f(grid, pairs, std::false_type());
  };
  switch (A.pairs) {
    case 1: pick(std::integral_constant<int, 1>()); break;
    case 2: pick(std::integral_constant<int, 2>()); break;
    default: pick(std::integral_constant<int, 3>()); break;
  }
  return hipGetLastError();
}

hipError_t matvec_sym64(const Sym64 &A, const double *x, double *y, hipStream_t s) {
  return sym64_launch(A, [&](dim3 grid, auto p, auto nt) {
    hipLaunchKernelGGL((k_matvec_sym64<p(), nt()>), grid, dim3(kBlock), 0, s, A, x, y);
  });
}

hipError_t pcg_matvec_dot_sym64(const Sym64 &A, const double *p, double *q, Partials pq,
                                double *pq2, SolveState *st, hipStream_t s) {
  const hipError_t e = sym64_launch(A, [&](dim3 grid, auto pairs, auto nt) {
    hipLaunchKernelGGL((k_pcg_matvec_dot_sym64<pairs(), nt()>), grid, dim3(kBlock), 0, s, A, p, q,
                       pq, st);
  });
  const int G = ell_chunks(A.n);
  if (e == hipSuccess && pq2)
    hipLaunchKernelGGL(k_fold_groups, dim3(fold_groups(G)), dim3(kBlock), 0, s, pq.a, G, pq2);
  return e == hipSuccess ? hipGetLastError() : e;
}

hipError_t pcg_step_sym64(const Sym64 &A, double *x, const double *p, double *pnext, double *q,
                          const double *r, const double *C, Partials pr, Partials pq,
                          SolveState *st, History h, hipStream_t s) {
  if (A.pairs < 1 || A.pairs > kSym64Pairs || ell_chunks(A.n) > kSmallChunks)
    return hipErrorInvalidValue;
  const dim3 grid(8 * ((ell_chunks(A.n) + 7) / 8));
  auto launch = [&](auto k) {
    hipLaunchKernelGGL(k, grid, dim3(kBlock), 0, s, A, x, p, pnext, q, r, C, pr, vec_grid(A.n), pq,
                       st, h);
  };
  switch (A.pairs) {
    case 1: C ? launch(k_pcg_step_sym64<1, true>) : launch(k_pcg_step_sym64<1, false>); break;
    case 2: C ? launch(k_pcg_step_sym64<2, true>) : launch(k_pcg_step_sym64<2, false>); break;
    default: C ? launch(k_pcg_step_sym64<3, true>) : launch(k_pcg_step_sym64<3, false>); break;
  }
  return hipGetLastError();
}

hipError_t pcg_update_small(int n, int G, double *r, const double *q, const double *C, Partials pq,
                            Partials pr, SolveState *st, History h, hipStream_t s) {
  if (ell_chunks(n) > kSmallChunks || G < 1 || G > kFoldDirect) return hipErrorInvalidValue;
  auto launch = [&](auto k) {
    hipLaunchKernelGGL(k, vgrid(n), dim3(kBlock), 0, s, n, G, r, q, C, pq.a, pr, st, h);
  };
  C ? launch(k_pcg_update_small<true>) : launch(k_pcg_update_small<false>);
  return hipGetLastError();
}

hipError_t pcg_update(int n, int gpq, double *r, const double *q, const double *C, Partials pq,
                      Partials pr, SolveState *st, History h, bool nt, hipStream_t s) {
  auto launch = [&](auto k) {
    hipLaunchKernelGGL(k, vgrid(n), dim3(kBlock), 0, s, n, gpq, r, q, C, pq, pr, st, h);
  };
  if (C)
    nt ? launch(k_pcg_update<true, true>) : launch(k_pcg_update<true, false>);
  else
    nt ? launch(k_pcg_update<false, true>) : launch(k_pcg_update<false, false>);
  return hipGetLastError();
}

hipError_t pcg_xpay(int n, double *x, double *p, const double *r, const double *C, Partials pr,
                    SolveState *st, History h, bool nt, hipStream_t s) {
  auto launch = [&](auto k) {
    hipLaunchKernelGGL(k, vgrid(n), dim3(kBlock), 0, s, n, x, p, r, C, pr, st, h);
  };
  if (C)
    nt ? launch(k_pcg_xpay<true, true>) : launch(k_pcg_xpay<true, false>);
  else
    nt ? launch(k_pcg_xpay<false, true>) : launch(k_pcg_xpay<false, false>);
  return hipGetLastError();
}

}  // namespace cghip

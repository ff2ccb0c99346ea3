// sgemv (wgblas src/sgemv/sgemv.mjs:19-254, shaders sgemv_n.wgsl,
// sgemv_t.wgsl, reduce_partials.wgsl) and its native-fp64 form dgemv
// (src/dgemv/dgemv.mjs:23-341), column-major as in BLAS, and further down
// the rank-1 / rank-2 updates sger / dger, ssyr / dsyr, ssyr2 / dsyr2
// (src/{sger,dger,ssyr,dsyr,ssyr2,dsyr2}/*.mjs). gemv:
//   trans = N: y (m) <- alpha A x + beta y, x of length n;
//   trans = T: y (n) <- alpha A^T x + beta y, x of length m.
//
// Both forms read A once and are HBM-bound. A lane's loads are 4 consecutive
// elements (16 bytes in fp32, 32 in fp64).
//   N: a lane owns 4 consecutive rows (one 4-element load per column, kStepN
//      columns per step), and a block walks a long run of columns (few, deep
//      blocks; where those are too few, narrower ones whose waves share the
//      columns); a column whose x entry is zero is
//      skipped, as reference BLAS does for this form (so 0 * Inf or 0 * NaN
//      in that column never reaches y).
//   T: a wave owns 8 columns (4 for short columns) and walks the rows 512
//      at a time (2 x 4 per lane, 4-element loads), keeping each x chunk in
//      registers for all of its columns;
//      the dot products are folded with wave shuffles. No zero skipping: the
//      dot-product form of reference BLAS takes every term.
// When the output alone gives too few blocks to stream HBM, the contraction
// dimension is split: each split writes partial sums, and a fold kernel adds
// the splits in order (deterministic) and applies alpha and beta.
#include "common.h"

#include <hip/hip_runtime.h>

#include "wgblas_hip.h"

namespace {

using wgb::fail;

constexpr int kThreads = 256;
// T form: columns per wave. 8 (x reused from registers for 8 columns);
// columns of at most kShortColsRows rows take 4, which gives twice the
// waves: measured on MI355X at 2048 x 65536, 4.8 -> 6.4 TB/s, while 4 was
// slower at 8192^2 (5.3 -> 4.8) and even at 16384^2 and 32768^2.
constexpr int kColsPerWave = 8;
constexpr int kColsPerWaveShort = 4;
constexpr int64_t kShortColsRows = 4096;
// N form: columns loaded per step, and for blocks of 1024 rows the number
// aimed for and the fewest columns per split. Measured on MI355X over
// 2048 x 65536, 8192^2, 16384^2, 32768^2 and 65536 x 2048 (sweep of 1 or 2
// groups, 256 / 512 / 1024 target blocks, 256 or 512 columns): one group,
// 8 columns per step, about 256 blocks of at least 256 columns each gave
// the best geometric mean, 5.92 TB/s against 5.06 for 4 groups x 4 columns
// with 2048 blocks of 64 columns (16384^2: 6.24 against 5.77 TB/s); fewer
// splits also mean fewer partial sums to write and fold.
constexpr int kStepN = 8;
constexpr int kTargetBlocksN = 256;
constexpr int kMinColsN = 256;
// Beside them, for small matrices and few rows (plan_n): blocks of 256 rows whose
// kColWaves waves share at least kMinColsNarrow
// columns, partial sums added in LDS. 4096^2, fp32: 64 wide blocks 38.2 us, 256
// narrow ones 12.9 (5.2 TB/s; 4 waves 16.4); fp64 70.2 and 27.1. Splits of at
// least 64 / 128 / 256 columns: fp32 512^2 6.9 / 6.6 / 8.6 us, fp64 8.7 / 10.2 /
// 17.7, fp64 2048^2 11.5 / 15.2 / 19.7.
constexpr int kColWaves = 8;
constexpr int kMinColsNarrow = 64;
constexpr int kTargetBlocks = 2048;  // T form: blocks that keep HBM streaming

int64_t imax(int64_t a, int64_t b) { return a > b ? a : b; }
int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

template <typename T>
using vec4 = T __attribute__((ext_vector_type(4)));
// The same four elements at element alignment: multi-dword global accesses
// need dword alignment only, so any lda and base takes vector accesses.
template <typename T>
using vec4u = T __attribute__((ext_vector_type(4), aligned(sizeof(T))));

// A is streamed once: non-temporal 4-element loads keep it from displacing x
// and the partial sums in the caches.
template <typename T>
__device__ __forceinline__ vec4<T> ld_nt(const T *p) {
  return __builtin_nontemporal_load(reinterpret_cast<const vec4u<T> *>(p));
}

// How a kernel accesses A (its VEC parameter): kElems, fewer rows than a
// vector; kVecU, vectors at element alignment; kVecA, vectors at their own
// alignment (lda % 4 == 0 and A aligned to 4 elements), non-temporal. Neighbour
// lanes' unaligned vectors share lines, which a non-temporal access fetches
// again (ger 5001^2, lda 5002, non-temporal / not: fp32 47.7 / 36.7 us, fp64
// 110 / 72; with element accesses 68.5 / 94.7).
constexpr int kElems = 0, kVecU = 1, kVecA = 2;

template <int VEC, typename T>
__device__ __forceinline__ vec4<T> ld(const T *p) {
  if constexpr (VEC == kVecA) return ld_nt(p);
  return *reinterpret_cast<const vec4u<T> *>(p);
}

template <typename T>
int vector_access(const T *A, int64_t lda) {
  return lda % 4 == 0 && (uintptr_t)A % (4 * sizeof(T)) == 0 ? kVecA : kVecU;
}

template <typename T>
int access_of(int64_t rows, const T *A, int64_t lda) {
  return rows < 4 ? kElems : vector_access(A, lda);
}

// Pins a value in its register(s) here: nothing before this point is moved past
// it. held_scalar: a value that is the same in every lane, in scalar registers.
template <typename T>
__device__ __forceinline__ T held(T v) {
  asm volatile("" : "+v"(v));
  return v;
}
template <typename T>
__device__ __forceinline__ T held_scalar(T v) {
  constexpr int W = sizeof(T) / 4;
  int w[W];
  __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
  for (int k = 0; k < W; ++k) {
    w[k] = __builtin_amdgcn_readfirstlane(w[k]);
    asm volatile("" : "+s"(w[k]));
  }
  __builtin_memcpy(&v, w, sizeof(T));
  return v;
}

// gemv T's access (incx == 1). Unaligned columns: element by element below 64 rows
// (a column is then a few lines, most of them shared with its neighbours:
// sgemv 33 x 1000001, lda 37, elements 92 us, vectors 99, non-temporal ones
// 122), else vectors; through the caches where they can hold A or in fp64, whose
// vectors are two lines wide (non-temporal / not: sgemv 2048^2, lda 2049, 9.0 /
// 8.5, 8191^2 49 / 45, 2001 x 60001 74 / 79, 12001^2 97 / 102; dgemv 2048^2 14.0 /
// 10.7, elements 13.1, 4096^2 31 / 28, 8191^2 103 / 101).
constexpr int64_t kCacheBytes = (int64_t)256 << 20;
template <typename T>
int access_t(int64_t m, int64_t n, const T *A, int64_t lda) {
  const int vec = vector_access(A, lda);
  if (vec == kVecA) return kVecA;
  if (m < 64) return kElems;
  return sizeof(T) == 8 || lda * n <= kCacheBytes / (int64_t)sizeof(T) ? kVecU : kVecA;
}

// Writes one output element: alpha * acc + beta * y (beta == 0 never reads y).
template <typename T>
__device__ __forceinline__ void store_y(T *y, int64_t idx, T acc, T alpha, T beta) {
  T v = alpha * acc;
  if (beta != (T)0) v = fma(beta, y[idx], v);
  y[idx] = v;
}

// N form. A block is RW x CW waves: RW of them side by side over the rows
// (256 each, 4 consecutive rows per lane: every load instruction of a wave
// reads 256 elements of one column), CW over the split's columns. Block b,
// split s: rows [256 RW b, +256 RW), columns [s cps, min(n, (s+1) cps)), cps a
// multiple of CW kStepN where CW > 1; the CW partial sums of a row are added through LDS in wave
// order. VEC not kElems (m >= 4): a lane whose rows cross m (or lie past it) reads
// the matrix's last 4 rows instead, in bounds, and stores only its own.
//
// The wide blocks' (CW == 1) whole waves keep every load of a step in flight
// before its arithmetic, in the form that measured best for the type: in fp32
// behind a per-lane branch that every lane of theirs takes, in fp64 by reading
// the x entries and then the columns into registers before the first is used.
// (fp32 20480^2 297 us, with fp64's form 332; fp64 16384^2 336, with fp32's 560.)
// Left to itself the compiler sinks each load of A and x into the branch on its
// column's x entry (fp64 512 x 200000 192 us). The wave that crosses m has its own loop: as
// a per-lane choice between vectors and elements it ran both for each column,
// and the launch waited for it (dgemv 8191^2, lda 8191, 183 us; now 93).
template <typename T, int VEC, int RW, int CW>
__global__ __launch_bounds__(64 * RW *CW) void gemv_n_kernel(int64_t m, int64_t n,
                                                              const T *__restrict__ A, int64_t lda,
                                                              const T *__restrict__ x, int64_t incx,
                                                              int64_t cps, T *__restrict__ part,
                                                              T alpha, T beta,
                                                              T *__restrict__ y, int64_t incy) {
  typedef vec4<T> f4;
  constexpr bool HELD = CW == 1 && sizeof(T) == 8;    // a step's operands held before its arithmetic
  constexpr bool BRANCH = CW == 1 && sizeof(T) == 4;  // whole waves load behind a per-lane branch
  // (uniform: x entries and column origins stay scalar)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rw = wave % RW, cw = wave / RW;
  const int64_t wr = (int64_t)blockIdx.x * (256 * RW) + 256 * rw;  // the wave's rows start here
  const int64_t rb = wr + 4 * lane;
  if (CW == 1 && wr >= m) return;
  const int64_t i0 = VEC ? (rb <= m - 4 ? rb : m - 4) : (rb < m ? rb : 0);
  int64_t j = (int64_t)blockIdx.y * cps;
  int64_t j1 = j + cps < n ? j + cps : n;
  j += cw * (cps / CW);
  if (CW > 1 && j1 > j + cps / CW) j1 = j + cps / CW;
  T acc[4] = {(T)0, (T)0, (T)0, (T)0};
  // kStepN columns per step. LAST: columns past j1 repeat the last one against a
  // zero x entry, which skips them
  auto step = [&](auto last_tag, auto whole_tag) {
    constexpr bool LAST = decltype(last_tag)::value, WHOLE = decltype(whole_tag)::value;
    const int64_t i = WHOLE && HELD ? rb : i0;
    T xv[kStepN];
    f4 av[kStepN];
#pragma unroll
    for (int c = 0; c < kStepN; ++c) {
      const T v = x[(!LAST || j + c < j1 ? j + c : j1 - 1) * incx];
      xv[c] = !LAST || j + c < j1 ? v : (T)0;
    }
#pragma unroll
    for (int c = 0; c < kStepN; ++c) {
      const T *col = A + (!LAST || j + c < j1 ? j + c : j1 - 1) * lda;
      if (WHOLE && BRANCH ? rb + 4 <= m : VEC != kElems) {
        av[c] = ld<VEC>(col + i);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) av[c][q] = col[i + q < m ? i + q : m - 1];
      }
    }
    if constexpr (HELD) {
#pragma unroll
      for (int c = 0; c < kStepN; ++c) xv[c] = held_scalar(xv[c]);
#pragma unroll
      for (int c = 0; c < kStepN; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) av[c][q] = held(av[c][q]);
    }
    // The step's own sums, then one add each: a chain of kStepN products and
    // per / kStepN adds in place of one of per products. Error against 64 bits
    // (sgemv) and a compensated sum (dgemv), without / with: sgemv 8100 x 7900
    // 2.1e-7 / 1.2e-7, dgemv 15000 x 4000 5.4e-16 / 2.7e-16; no time in sgemv,
    // 0.4 % in dgemv (geometric means of 117 timings each).
    T sum[4] = {(T)0, (T)0, (T)0, (T)0};
#pragma unroll
    for (int c = 0; c < kStepN; ++c) {
      if (xv[c] != (T)0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) sum[q] = fma(av[c][q], xv[c], sum[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] += sum[q];
  };
  auto walk = [&](auto whole_tag) {
    for (; j + kStepN <= j1; j += kStepN) step(std::false_type{}, whole_tag);
    if (j < j1) step(std::true_type{}, whole_tag);
  };
  if (CW == 1 && VEC && wr + 256 <= m)  // a wave's choice
    walk(std::true_type{});
  else
    walk(std::false_type{});
  if constexpr (CW > 1) {
    __shared__ T red[CW - 1][RW * 64][4];
    if (cw > 0) {
#pragma unroll
      for (int q = 0; q < 4; ++q) red[cw - 1][64 * rw + lane][q] = acc[q];
    }
    __syncthreads();
    if (cw > 0) return;
#pragma unroll
    for (int c = 0; c < CW - 1; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] += red[c][64 * rw + lane][q];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int64_t i = i0 + q;
    if (i < rb || i >= m) continue;  // another lane's row, or none
    if (part)
      part[(int64_t)blockIdx.y * m + i] = acc[q];
    else
      store_y(y, i * incy, acc[q], alpha, beta);
  }
}

// T form. Wave w (4 per block) owns columns [CPW w, CPW w + CPW) of split s, rows
// [s*rps, min(m, (s+1)*rps)). VEC not kElems: incx == 1, vectors of A and x at any
// alignment (rows past a split's last whole vector one by one); access_t says
// which.
template <typename T, int VEC, int CPW>
__global__ __launch_bounds__(kThreads) void gemv_t_kernel(int64_t m, int64_t n,
                                                          const T *__restrict__ A, int64_t lda,
                                                          const T *__restrict__ x, int64_t incx,
                                                          int64_t rps, T *__restrict__ part,
                                                          T alpha, T beta,
                                                          T *__restrict__ y, int64_t incy) {
  typedef vec4<T> f4;
  const int lane = threadIdx.x & 63;
  const int64_t col0 = ((int64_t)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6)) * CPW;
  if (col0 >= n) return;  // wave-uniform
  const int64_t r0 = (int64_t)blockIdx.y * rps;
  const int64_t r1 = r0 + rps < m ? r0 + rps : m;
  // columns past n repeat column n-1 (in bounds) and are never stored
  const T *col[CPW];
#pragma unroll
  for (int c = 0; c < CPW; ++c) col[c] = A + (col0 + c < n ? col0 + c : n - 1) * lda;
  T acc[CPW];
#pragma unroll
  for (int c = 0; c < CPW; ++c) acc[c] = (T)0;
  int64_t i = r0 + 4 * lane;
  if (VEC) {
    // two 256-row groups per step: 16 loads of A in flight per lane
    for (; i + 256 + 4 <= r1; i += 512) {
      const f4 xv0 = *reinterpret_cast<const vec4u<T> *>(x + i);
      const f4 xv1 = *reinterpret_cast<const vec4u<T> *>(x + i + 256);
      f4 av0[CPW], av1[CPW];
#pragma unroll
      for (int c = 0; c < CPW; ++c) {
        av0[c] = ld<VEC>(col[c] + i);
        av1[c] = ld<VEC>(col[c] + i + 256);
      }
      // fp64: every load of the step is issued before the arithmetic. Left
      // to itself the scheduler placed each 16-byte load just before its
      // FMAs and waited for it (one load in flight: 16384^2 at 3.5 TB/s).
      if constexpr (sizeof(T) == 8) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < CPW; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[c] = fma(av0[c][q], xv0[q], acc[c]);
#pragma unroll
      for (int c = 0; c < CPW; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[c] = fma(av1[c][q], xv1[q], acc[c]);
    }
  }
  for (; i < r1; i += 256) {
    if (VEC && i + 4 <= r1) {
      const f4 xv = *reinterpret_cast<const vec4u<T> *>(x + i);
      f4 av[CPW];
#pragma unroll
      for (int c = 0; c < CPW; ++c) av[c] = ld<VEC>(col[c] + i);
#pragma unroll
      for (int c = 0; c < CPW; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[c] = fma(av[c][q], xv[q], acc[c]);
    } else {
      const int cnt = r1 - i < 4 ? (int)(r1 - i) : 4;
      for (int q = 0; q < cnt; ++q) {
        const T xv = x[(i + q) * incx];
#pragma unroll
        for (int c = 0; c < CPW; ++c) acc[c] = fma(col[c][i + q], xv, acc[c]);
      }
    }
  }
#pragma unroll
  for (int c = 0; c < CPW; ++c) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc[c] += __shfl_xor(acc[c], off, 64);
  }
  if (lane < CPW && col0 + lane < n) {
    T v = acc[0];
#pragma unroll
    for (int c = 1; c < CPW; ++c) v = lane == c ? acc[c] : v;
    if (part)
      part[(int64_t)blockIdx.y * n + col0 + lane] = v;
    else
      store_y(y, (col0 + lane) * incy, v, alpha, beta);
  }
}

// One fold pass over groups of kFold splits: block (b, g) adds splits
// [g*kFold, min(splits, (g+1)*kFold)) of outputs [256 b, 256 b + 256) in
// split order, with all of a group's loads in flight (clamped addresses, so
// none is guarded). The last pass (one group) writes alpha * sum + beta * y;
// earlier ones write the group sums to out[g*len + i] for the next pass.
constexpr int kFold = 32;
template <typename T>
__global__ __launch_bounds__(kThreads) void gemv_fold_kernel(int64_t len, int64_t splits,
                                                             const T *__restrict__ part,
                                                             T *__restrict__ out, T alpha,
                                                             T beta, T *__restrict__ y,
                                                             int64_t incy) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= len) return;
  const int64_t s0 = (int64_t)blockIdx.y * kFold;
  const int64_t last = (s0 + kFold < splits ? s0 + kFold : splits) - 1;
  T v[kFold];
#pragma unroll
  for (int q = 0; q < kFold; ++q) v[q] = part[(s0 + q < last ? s0 + q : last) * len + i];
  T sum = v[0];
#pragma unroll
  for (int q = 1; q < kFold; ++q)
    if (s0 + q <= last) sum += v[q];
  if (gridDim.y == 1 && out == nullptr)
    store_y(y, i * incy, sum, alpha, beta);
  else
    out[(int64_t)blockIdx.y * len + i] = sum;
}

// y <- beta * y over len elements (0 when beta == 0): alpha == 0.
template <typename T>
__global__ __launch_bounds__(kThreads) void scale_y_kernel(int64_t len, T beta, T *y,
                                                           int64_t incy) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i < len) y[i * incy] = beta == (T)0 ? (T)0 : beta * y[i * incy];
}

// Triangles of order n are walked as chunks of 1024 rows (4 consecutive rows
// per lane of a block), each with the columns that its rows meet, kTriStep
// columns at a time. All chunks' columns are laid end to end, each chunk's
// count rounded up to whole steps, and cut into equal runs, one per block: a
// rectangular grid over (chunk, panel) launches the other triangle's blocks
// for nothing and leaves the last round of working ones uneven.
constexpr int64_t kChunkRows = 4 * kThreads;
constexpr int kTriStep = 8;

// First column of chunk r (0 for a lower triangle, its first row for an upper
// one) and the columns laid before and within it.
template <bool LOWER>
__host__ __device__ __forceinline__ int64_t chunk_first(int64_t r) {
  return LOWER ? 0 : r * kChunkRows;
}
template <bool LOWER>
__host__ __device__ __forceinline__ int64_t chunk_offset(int64_t n, int64_t r) {
  const int64_t n8 = (n + kTriStep - 1) / kTriStep * kTriStep;
  return LOWER ? kChunkRows * (r * (r + 1) / 2) : r * n8 - kChunkRows * (r * (r - 1) / 2);
}
template <bool LOWER>
__host__ __device__ __forceinline__ int64_t chunk_columns(int64_t n, int64_t r) {
  const int64_t n8 = (n + kTriStep - 1) / kTriStep * kTriStep;
  return LOWER ? ((r + 1) * kChunkRows < n8 ? (r + 1) * kChunkRows : n8) : n8 - r * kChunkRows;
}
template <bool LOWER>
int64_t triangle_columns(int64_t n) {
  const int64_t last = (n - 1) / kChunkRows;
  return chunk_offset<LOWER>(n, last) + chunk_columns<LOWER>(n, last);
}

// Calls body(r, c0, c1) for each chunk r of which block b's run, [b run,
// (b + 1) run), holds columns [c0, c1).
template <bool LOWER, class Body>
__device__ __forceinline__ void walk_triangle(int64_t n, int64_t run, Body body) {
  const int64_t f = (int64_t)blockIdx.x * run;
  int64_t off = 0;
  for (int64_t r = 0; r * kChunkRows < n && off < f + run; ++r) {
    const int64_t cols = chunk_columns<LOWER>(n, r), first = chunk_first<LOWER>(r);
    const int64_t a = f > off ? f - off : 0, b = f + run - off < cols ? f + run - off : cols;
    if (a < b) body(r, first + a, first + b < n ? first + b : n);
    off += cols;
  }
}

// Rank-1 and rank-2 updates, A m x n column-major:
//   ger  (UPLO 0, !TWO): A += alpha x y^T;
//   syr  (UPLO 1 / 2, !TWO, y = x): the lower (i >= j) / upper (i <= j)
//        triangle of A += alpha x x^T;
//   syr2 (UPLO 1 / 2, TWO): that triangle of A += alpha x y^T + alpha y x^T.
// A block takes 1024 rows (4 consecutive ones per lane, its x (and y) entries
// held in registers) of a run of columns: for ger, block (b, c) rows
// [1024 b, +1024) and columns [c cpb, min(n, (c+1) cpb)); for a triangle, block
// b its run of cpb of the chunks' columns (walk_triangle). Columns go
// kStepG at a time with all of a step's A loads in flight. Column j takes
// t1 = alpha y[j] (and t2 = alpha x[j]) and A(i, j) = fma(x[i], t1, A(i, j))
// (then fma(y[i], t2, .)); a column whose y entry (for syr2: both entries)
// is zero is neither computed nor written, reference BLAS's skip: Infinity or
// NaN in the row vector never meets that zero. A is read and written once:
// HBM-bound, 2 m n elements of traffic (half that for a triangle).
constexpr int kStepG = kTriStep;
template <typename T, int VEC, int UPLO, bool TWO>
__global__ __launch_bounds__(kThreads) void rank_update_kernel(
    int64_t m, int64_t n, T alpha, const T *__restrict__ x, int64_t incx, const T *__restrict__ y,
    int64_t incy, T *__restrict__ A, int64_t lda, int64_t cpb) {
  typedef vec4<T> f4;
  constexpr int kVecCut = 3;
  // columns [j0, j1) of the 1024 rows from r0 on
  auto chunk = [&](const int64_t r0, int64_t j0, int64_t j1) {
  const int64_t ib = r0 + 4 * threadIdx.x;  // the lane's own rows start here
  if (ib >= m) return;
  // VEC not kElems (m >= 4): a lane whose rows cross m takes the matrix's last 4 rows, in
  // bounds; [lo, 4) of them are its own
  const int64_t i0 = VEC && ib > m - 4 ? m - 4 : ib;
  const int lo = (int)(ib - i0);
  const int rows = i0 + 4 <= m ? 4 : (int)(m - i0);
  f4 xv, yv;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    xv[q] = q < rows ? x[(i0 + q) * incx] : (T)0;
    yv[q] = TWO && q < rows ? y[(i0 + q) * incy] : (T)0;
  }
  // update of one column's 4 rows (masked rows keep their value)
  auto column_scalars = [&](int64_t j, T &t1, T &t2) -> bool {
    const T c1 = y[j * incy];
    const T c2 = TWO ? x[j * incx] : (T)0;
    t1 = alpha * c1;
    t2 = alpha * c2;
    return c1 != (T)0 || (TWO && c2 != (T)0);
  };
  auto update = [&](f4 &a, T t1, T t2) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      a[q] = fma(xv[q], t1, a[q]);
      if (TWO) a[q] = fma(yv[q], t2, a[q]);
    }
  };
  // MODE: how the wave accesses A, whole vectors with no per-lane branch
  // between the stores (kVecA: non-temporal; kVecCut: in a chunk that m cuts, as
  // kVecU), or kElems for a wave with fewer
  // than 4 rows (its loads are still whole vectors where m >= 4) or a matrix with
  // fewer. A lane whose rows cross m updates the last 4 rows of its wave, as its
  // neighbours in the same instructions do: the rows they share get the same
  // values. MASK (the diagonal columns of a triangle): the same loads and
  // arithmetic, and each lane stores only its own rows inside the triangle (whole
  // vectors where all four are).
  auto walk = [&](auto mode_tag, auto mask_tag, int64_t ja, int64_t jb) {
    constexpr int MODE = decltype(mode_tag)::value;
    constexpr bool FULL = MODE != kElems;
    constexpr bool MASK = decltype(mask_tag)::value;
    auto load = [&](const T *col) -> f4 {
      if constexpr (VEC) return ld<FULL ? MODE : kVecU>(col + i0);
      f4 v;
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = col[i0 + (q < rows ? q : 0)];
      return v;
    };
    auto store = [&](T *col, const f4 &v, int64_t j) {
      if constexpr (MASK) {
        const bool all = lo == 0 && (UPLO == 1 ? i0 >= j : i0 + rows - 1 <= j);
        if (!all) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int64_t i = i0 + q;
            if (q >= lo && q < rows && (UPLO == 1 ? i >= j : i <= j)) col[i] = v[q];
          }
          return;
        }
      }
      if (FULL || (VEC && lo == 0)) {
        if constexpr (MODE == kVecA) {
          __builtin_nontemporal_store(v, reinterpret_cast<vec4u<T> *>(col + i0));
        } else if constexpr (MODE == kVecCut) {
          // all of the column's vector is loaded before any part of it is stored:
          // lanes that share rows must not read each other's results
          T a = v[0], b = v[1], c = v[2], d = v[3];
          asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d) : : "memory");
          *reinterpret_cast<vec4u<T> *>(col + i0) = f4{a, b, c, d};
        } else {
          *reinterpret_cast<vec4u<T> *>(col + i0) = v;
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (q >= lo && q < rows) col[i0 + q] = v[q];
      }
    };
    int64_t j = ja;
    for (; j + kStepG <= jb; j += kStepG) {
      T t1[kStepG], t2[kStepG];
      bool live[kStepG];
      f4 a[kStepG];
#pragma unroll
      for (int c = 0; c < kStepG; ++c) live[c] = column_scalars(j + c, t1[c], t2[c]);
#pragma unroll
      for (int c = 0; c < kStepG; ++c) a[c] = load(A + (j + c) * lda);
#pragma unroll
      for (int c = 0; c < kStepG; ++c) {
        if (live[c]) {  // uniform: the column's entries
          update(a[c], t1[c], t2[c]);
          store(A + (j + c) * lda, a[c], j + c);
        }
      }
    }
    for (; j < jb; ++j) {
      T t1, t2;
      if (column_scalars(j, t1, t2)) {
        f4 a = load(A + j * lda);
        update(a, t1, t2);
        store(A + j * lda, a, j);
      }
    }
  };
  const int64_t w0 = r0 + 256 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // the wave's 256 rows
  const bool vectors = VEC && m - w0 >= 4;
  // The blocks of a row chunk that m cuts access A through the caches: non-temporal
  // whole waves there and element stores in the crossing one took dger 768 x
  // 30000 87 us (element accesses in the whole block 71, this 58), 1001 x 30000,
  // lda 1004, 103 (93, 74), 5001^2, lda 5004, 112 (108, 107), 8191^2, lda 8192, 198
  // (192, 192).
  const bool cut = r0 + kChunkRows > m;
  auto walk_range = [&](auto mask_tag, int64_t ja, int64_t jb) {
    if (ja >= jb) return;
    if (vectors && !cut)
      walk(std::integral_constant<int, VEC>{}, mask_tag, ja, jb);
    else if (vectors)
      walk(std::integral_constant<int, VEC ? kVecCut : kElems>{}, mask_tag, ja, jb);
    else
      walk(std::integral_constant<int, kElems>{}, mask_tag, ja, jb);
  };
  // columns wholly inside the triangle for these 256 rows, and diagonal ones
  // (row i of column j is stored where i >= j (lower) or i <= j (upper))
  const int64_t da = j0 > w0 ? j0 : w0, db = j1 < w0 + 256 ? j1 : w0 + 256;
  if constexpr (UPLO == 0) {
    walk_range(std::false_type{}, j0, j1);
  } else if constexpr (UPLO == 1) {
    walk_range(std::false_type{}, j0, j1 < w0 ? j1 : w0);
    walk_range(std::true_type{}, da, db);
  } else {
    walk_range(std::true_type{}, da, db);
    walk_range(std::false_type{}, j0 > w0 + 256 ? j0 : w0 + 256, j1);
  }
  };
  if constexpr (UPLO == 0) {
    const int64_t j0 = (int64_t)blockIdx.y * cpb;
    chunk((int64_t)blockIdx.x * kChunkRows, j0, j0 + cpb < n ? j0 + cpb : n);
  } else {
    walk_triangle<UPLO == 1>(n, cpb, [&](int64_t r, int64_t c0, int64_t c1) { chunk(r * kChunkRows, c0, c1); });
  }
}

// ger (uplo 0, y given), syr (uplo 1 / 2, y == x, !two), syr2 (uplo 1 / 2,
// two): argument checks, reference BLAS's quick returns (m or n zero, alpha
// zero: A untouched, vectors unread; src/sger/sger.mjs:86, 103,
// src/ssyr/ssyr.mjs:59, 75), one launch.
template <typename T>
int rank_update(wgb_ctx *ctx, int uplo, bool two, int64_t m, int64_t n, T alpha, const T *x,
                int64_t incx, const T *y, int64_t incy, T *A, int64_t lda) {
  int st = wgb::enter(ctx);
  if (st) return st;
  if (uplo != 0 && uplo != WGB_LOWER && uplo != WGB_UPPER)
    return fail(WGB_ERR_INVALID_VALUE, "uplo must be WGB_LOWER or WGB_UPPER");
  if (m < 0 || n < 0) return fail(WGB_ERR_INVALID_VALUE, "m and n must be non-negative");
  if (lda < imax(1, m)) return fail(WGB_ERR_INVALID_VALUE, "lda must be >= max(1, rows of A)");
  if (incx <= 0 || incy <= 0) return fail(WGB_ERR_INVALID_VALUE, "incx and incy must be positive");
  if (m == 0 || n == 0 || alpha == (T)0) return WGB_OK;
  if (!A || !x || !y) return fail(WGB_ERR_INVALID_VALUE, "A, x or y is null");
  wgb::timing_begin(ctx);
  const int64_t bx = cdiv(m, 4 * kThreads);
  // column chunks: about one block per CU in all for ger (each a long run of
  // columns), at least kStepG columns each. Measured at 16384^2 on one box,
  // blocks in all against TB/s (fp32 / fp64): 128 3.5 / 3.7, 256 5.7 / 5.2,
  // 384 5.7 / 4.1, 512 5.5 / 4.9, 2048 4.8 / 4.7. Triangles: equal runs, two
  // per CU for fp32 and one for fp64 (lower, 1 / 2 / 4 runs per CU: ssyr2 8192
  // 63.7 / 52.9 / 52.9 us, 16384 211 / 207 / 205; dsyr2 8192 115 / 117 / 128,
  // 16384 453 / 479 / 484; a rectangular grid took 80, 300, 200 and 632).
  const int64_t cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  dim3 grid;
  int64_t cpb;
  if (uplo == 0) {
    int64_t chunks = cdiv(cus, bx);
    if (chunks > cdiv(n, kStepG)) chunks = cdiv(n, kStepG);
    if (chunks > 65535) chunks = 65535;
    if (chunks < 1) chunks = 1;
    cpb = cdiv(n, chunks);
    grid = dim3((unsigned)bx, (unsigned)cdiv(n, cpb));
  } else {
    const int64_t total = uplo == WGB_LOWER ? triangle_columns<true>(n) : triangle_columns<false>(n);
    cpb = cdiv(cdiv(total, (sizeof(T) == 4 ? 2 : 1) * cus), kStepG) * kStepG;
    grid = dim3((unsigned)cdiv(total, cpb));
  }
  auto launch = [&](auto kern) {
    kern<<<grid, kThreads, 0, ctx->stream>>>(m, n, alpha, x, incx, y, incy, A, lda, cpb);
  };
  auto by_form = [&](auto vec_tag) {
    constexpr int VEC = decltype(vec_tag)::value;
    if (uplo == 0)
      launch(rank_update_kernel<T, VEC, 0, false>);
    else if (uplo == WGB_LOWER)
      launch(two ? rank_update_kernel<T, VEC, 1, true> : rank_update_kernel<T, VEC, 1, false>);
    else
      launch(two ? rank_update_kernel<T, VEC, 2, true> : rank_update_kernel<T, VEC, 2, false>);
  };
  const int vec = access_of(m, A, lda);
  if (vec == kVecA)
    by_form(std::integral_constant<int, kVecA>{});
  else if (vec == kVecU)
    by_form(std::integral_constant<int, kVecU>{});
  else
    by_form(std::integral_constant<int, kElems>{});
  WGB_CHECK_LAUNCH("rank_update_kernel");
  wgb::timing_end(ctx);
  return WGB_OK;
}

// ssymv / dsymv: y <- alpha S x + beta y, S the n x n symmetric matrix whose
// uplo triangle A holds (column-major). The triangle is read once: a block
// takes a run of columns of a chunk of 1024 rows (walk_triangle; 4 rows per
// lane, their x entries in registers), 8 columns at a time with all of a
// step's loads in flight, and uses each stored element twice: A(i, j) x(j) for
// row i and, off the diagonal, A(i, j) x(i) for its mirror, row j. The row
// sums of block b over chunk r go to row slot b - (r's first block)
// (part[slot n + i]); the mirror sums of a column are folded across each wave
// (fold8) and, once at the end of the run, across the 4 waves (LDS) into column
// slot r (part[(slots + r) n + j]). symv_fold_kernel then adds, for each j,
// exactly the slots that were written for it, in a fixed order (deterministic),
// and applies alpha and beta. Every term is taken (no zero skipping, as
// reference BLAS's symv). Waves that cross the diagonal mask elements outside
// the triangle by selecting their terms away (never multiplying them).
// HBM-bound: the triangle once. Lower, rectangular 1024 x 128 blocks with a
// shuffle fold per column -> this: ssymv 16384 144 -> 89 us (6.0 TB/s), 8192 58
// -> 28, 4096 50 -> 13; dsymv 16384 339 -> 192 (5.6 TB/s), 4096 65 -> 21.
constexpr int kRunMax = 512;  // columns per block (the LDS of their sums)
constexpr int kRunMin = 32;
constexpr int64_t kSymvMaxN = (int64_t)65535 * 128;  // accepted orders
constexpr int kSymvStep = kTriStep;                  // columns per step
constexpr int kSymvFoldWaves = 8;

// Columns per block, blocks, and row slots (the most blocks that meet one
// chunk): equal runs, two per CU where they have kRunMin columns, and no more
// than kRunMax allows (lower, 1 / 2 / 4 per CU: ssymv 8192 29.3 / 27.7 / 29.3
// us, dsymv 8192 57.9 / 55.6 / 73.0, 16384 193 / 192 / 242; dsymv 4096, where
// two would be 20 columns, 21.2 against 27.0 in runs of 32).
struct SymvPlan {
  int64_t run, blocks, slots;
};
template <bool LOWER>
SymvPlan symv_plan(int64_t n, int64_t cus) {
  const int64_t total = triangle_columns<LOWER>(n);
  int64_t rounds = cdiv(total, cus * kRunMax);
  if (rounds < 2) rounds = total >= 2 * cus * kRunMin ? 2 : 1;
  int64_t run = cdiv(cdiv(total, rounds * cus), kTriStep) * kTriStep;
  if (run < kRunMin) run = kRunMin;
  SymvPlan p = {run, cdiv(total, run), 0};
  for (int64_t r = 0; r * kChunkRows < n; ++r) {
    const int64_t off = chunk_offset<LOWER>(n, r);
    const int64_t meet = (off + chunk_columns<LOWER>(n, r) - 1) / run - off / run + 1;
    if (meet > p.slots) p.slots = meet;
  }
  return p;
}

// Value of lane ^ 1, ^ 2 (quads), the mirror in 8 lanes, lane ^ 8: DPP moves,
// one VALU instruction each (two for 8-byte values).
template <int CTRL, typename T>
__device__ __forceinline__ T dpp(T v) {
  constexpr int W = sizeof(T) / 4;
  int w[W];
  __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
  for (int k = 0; k < W; ++k) w[k] = __builtin_amdgcn_mov_dpp(w[k], CTRL, 0xf, 0xf, true);
  __builtin_memcpy(&v, w, sizeof(T));
  return v;
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppRor8 = 0x128;

// permlane32_swap exchanges a's upper 32 lanes with b's lower 32, so that the
// two results' sum holds a's fold in the lower half and b's in the upper one;
// permlane16_swap does the same with odd and even rows of 16 lanes.
template <bool HALVES, typename T>
__device__ __forceinline__ T swap_add(T a, T b) {
  constexpr int W = sizeof(T) / 4;
  unsigned wa[W], wb[W];
  __builtin_memcpy(wa, &a, sizeof(T));
  __builtin_memcpy(wb, &b, sizeof(T));
#pragma unroll
  for (int k = 0; k < W; ++k) {
    if constexpr (HALVES) {
      const auto r = __builtin_amdgcn_permlane32_swap(wa[k], wb[k], false, false);
      wa[k] = r[0];
      wb[k] = r[1];
    } else {
      const auto r = __builtin_amdgcn_permlane16_swap(wa[k], wb[k], false, false);
      wa[k] = r[0];
      wb[k] = r[1];
    }
  }
  __builtin_memcpy(&a, wa, sizeof(T));
  __builtin_memcpy(&b, wb, sizeof(T));
  return a + b;
}

// Folds 8 values per lane over the wave: returns, in every lane, the sum of
// v[lane / 8] over all 64 lanes. Each exchange halves the values a lane
// still carries: 6 swaps and 4 DPP moves, against 48 LDS-routed shuffles for
// 8 folds of their own.
template <typename T>
__device__ __forceinline__ T fold8(const T (&v)[8], int lane) {
  T a[4], b[2];
#pragma unroll
  for (int c = 0; c < 4; ++c) a[c] = swap_add<true>(v[c], v[c + 4]);
#pragma unroll
  for (int c = 0; c < 2; ++c) b[c] = swap_add<false>(a[c], a[c + 2]);
  const bool odd = lane & 8;
  T s = (odd ? b[1] : b[0]) + dpp<kDppRor8>(odd ? b[0] : b[1]);
  s += dpp<kDppXor1>(s);
  s += dpp<kDppXor2>(s);
  return s + dpp<kDppHalfMirror>(s);
}

// MODE 0: symv (row and mirror sums); 1: strmv without transpose (row sums
// over the triangle, diagonal included, a column skipped where x is zero);
// 2: strmv transposed (column sums over the triangle, diagonal included, no
// skipping). UNIT: the diagonal taken as 1, its stored value never used.
// VEC not kElems (n >= 4): a lane whose rows cross n (or lie past it) reads the
// matrix's last 4 rows, in bounds, and uses only its own.
template <typename T, int VEC, int UPLO, int MODE = 0, bool UNIT = false>
__global__ __launch_bounds__(kThreads) void symv_kernel(int64_t n, int64_t run, int64_t slots,
                                                        const T *__restrict__ A, int64_t lda,
                                                        const T *__restrict__ x, int64_t incx,
                                                        T *__restrict__ part) {
  typedef vec4<T> f4;
  constexpr int S = kSymvStep;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // per-wave column sums of every step, added across the waves once at the
  // end: no barrier between steps, so a step's loads never wait on the
  // previous step's reduction
  __shared__ T red[MODE == 1 ? 1 : kRunMax / S][4][S];
  walk_triangle<UPLO == 1>(n, run, [&](const int64_t r, const int64_t c0, const int64_t cend) {
  const int64_t r0 = r * kChunkRows;
  const int64_t w0 = r0 + 256 * wave;  // the wave's 256 rows
  const int64_t ib = r0 + 4 * threadIdx.x;  // this lane's rows: those of i0 .. i0 + 3 in [ib, n)
  const int64_t i0 = VEC ? (ib <= n - 4 ? ib : n - 4) : (ib < n ? ib : 0);
  f4 xv;
  T racc[4];
  bool own[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    own[q] = i0 + q >= ib && i0 + q < n;
    xv[q] = own[q] ? x[(i0 + q) * incx] : (T)0;
    racc[q] = (T)0;
  }
  // columns [ja, jb), a whole number of steps from c0 on. WHOLE: whole steps,
  // and every lane's rows inside n or (PART) rows of other lanes taken as 0;
  // CROSS: some element outside the triangle or on the diagonal. Compiled once
  // per form: with any as a run-time test the loads sat in separate branches
  // and issued one by one.
  auto steps = [&](auto whole_tag, auto cross_tag, auto part_tag, int64_t ja, int64_t jb) {
    constexpr bool WHOLE = decltype(whole_tag)::value;
    constexpr bool PART = decltype(part_tag)::value;
    constexpr bool CROSS = decltype(cross_tag)::value;
    int step = (int)(ja - c0) / S;
    for (int64_t j = ja; j < jb; j += S, ++step) {
      const int cols = WHOLE || jb - j >= S ? S : (int)(jb - j);
      f4 a[S];
      T xc[S];
#pragma unroll
      for (int c = 0; c < S; ++c) {
        const int64_t jc = j + (c < cols ? c : 0);  // clamped: every load in bounds
        const T xj = x[jc * incx];
        xc[c] = c < cols ? xj : (T)0;
        const T *col = A + jc * lda;
        if constexpr (VEC) {
          a[c] = ld<VEC>(col + i0);
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) a[c][q] = col[i0 + q < n ? i0 + q : n - 1];
        }
      }
      T cacc[S];
      T rstep[4] = {(T)0, (T)0, (T)0, (T)0};  // the step's row sums: a chain of 8 products, then one add
      const int d = CROSS ? (int)(i0 - j) : 0;
#pragma unroll
      for (int c = 0; c < S; ++c) {
        cacc[c] = (T)0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          bool in = WHOLE || (c < cols && own[q]);  // stored element (i0 + q, j + c) of this lane
          bool mirror = in;                         // ... off the diagonal
          if constexpr (CROSS) {
            in = in && (UPLO == 1 ? d >= c - q : d <= c - q);
            mirror = in && d != c - q;
          }
          T av = a[c][q];
          if constexpr (PART) av = own[q] ? av : (T)0;
          if constexpr (UNIT && CROSS) av = d == c - q ? (T)1 : av;  // only a crossing block holds the diagonal
          if constexpr (MODE == 0) {
            rstep[q] = in ? fma(av, xc[c], rstep[q]) : rstep[q];
            cacc[c] = mirror ? fma(av, xv[q], cacc[c]) : cacc[c];
          } else if constexpr (MODE == 1) {
            // reference BLAS's column form: a zero x entry skips its column
            rstep[q] = in && xc[c] != (T)0 ? fma(av, xc[c], rstep[q]) : rstep[q];
          } else {
            cacc[c] = in ? fma(av, xv[q], cacc[c]) : cacc[c];
          }
        }
      }
      if constexpr (MODE != 2) {
#pragma unroll
        for (int q = 0; q < 4; ++q) racc[q] += rstep[q];
      }
      if constexpr (MODE != 1) {  // the step's column sums across the wave
        const T v = fold8(cacc, lane);
        if ((lane & 7) == 0) red[step][wave][lane >> 3] = v;
      }
    }
  };
  auto range = [&](auto cross_tag, int64_t ja, int64_t jb) {
    if (ja >= jb) return;
    // symv: only a run's last, partial step has run-time columns. A wave that
    // crosses n and took them for its 256 diagonal columns set the launch's time
    // (ssymv 16383 upper, lda 16384, 151 us against 89 now; lower 12000 90
    // against 51). strmv keeps them there: its shorter kernels lose 2 to 4% to
    // the form's code at orders that are multiples of 256.
    constexpr bool CROSS = decltype(cross_tag)::value;
    const bool all = w0 + 256 <= n;
    const int64_t jw = VEC && (all || !CROSS || MODE == 0) ? ja + (jb - ja) / S * S : ja;
    if (ja < jw) {
      if (all)
        steps(std::true_type{}, cross_tag, std::false_type{}, ja, jw);
      else if constexpr (!CROSS || MODE == 0)
        steps(std::true_type{}, cross_tag, std::true_type{}, ja, jw);
    }
    if (jw < jb) steps(std::false_type{}, std::true_type{}, std::false_type{}, jw, jb);
  };
  // for the wave's 256 rows: columns all inside the triangle and off the
  // diagonal, columns that cross it, and columns outside (their sums are 0)
  const int64_t lo = c0 > w0 ? c0 : w0, hi = cend < w0 + 256 ? cend : w0 + 256;
  if constexpr (UPLO == 1) {
    if (w0 < n) {
      range(std::false_type{}, c0, cend < w0 ? cend : w0);
      range(std::true_type{}, lo, hi);
    }
  } else {
    range(std::true_type{}, lo, hi);
    range(std::false_type{}, c0 > w0 + 256 ? c0 : w0 + 256, cend);
  }
  if constexpr (MODE != 1) {
    const int64_t za = UPLO == 1 && w0 < n ? (c0 > w0 + 256 ? c0 : w0 + 256) : c0;
    const int64_t zb = UPLO == 1 ? cend : (cend < w0 ? cend : w0);
    for (int64_t j = za + lane; j < zb; j += 64) red[(j - c0) / S][wave][(j - c0) % S] = (T)0;
  }
  if (MODE != 2) {
    const int64_t slot = (int64_t)blockIdx.x - chunk_offset<UPLO == 1>(n, r) / run;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (own[q]) part[slot * n + i0 + q] = racc[q];
  }
  if constexpr (MODE != 1) {
    __syncthreads();
    T *colpart = part + (slots + r) * n + c0;
    for (int t = threadIdx.x; t < cend - c0; t += kThreads) {
      const int st = t / S, c = t % S;
      colpart[t] = ((red[st][0][c] + red[st][1][c]) + red[st][2][c]) + red[st][3][c];
    }
    __syncthreads();  // the next chunk's sums take the same LDS
  }
  });
}

// y(j) <- alpha (sum of the row slots of j's chunk + sum of the column slots of
// the chunks that meet column j) + beta y(j). A block folds 64 outputs (one
// chunk's): its waves take 8 slots at a time in turn, added in wave order
// through LDS. beta == 0 never reads y.
template <typename T, int UPLO, int MODE = 0>
__global__ __launch_bounds__(64 * kSymvFoldWaves) void symv_fold_kernel(int64_t n, int64_t run, int64_t slots,
                                                                        const T *__restrict__ part, T alpha,
                                                                        T beta, T *__restrict__ y, int64_t incy) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t j = (int64_t)blockIdx.x * 64 + lane;
  const int64_t jl = j < n ? j : n - 1;  // lanes past n fold column n - 1 and store nothing
  const int64_t r = (int64_t)blockIdx.x * 64 / kChunkRows, nr = (n + kChunkRows - 1) / kChunkRows;
  const int64_t off = chunk_offset<UPLO == 1>(n, r);
  // row sums (symv, strmv without transpose), then column sums (symv's
  // mirrors, strmv transposed)
  const int rows = MODE != 2 ? (int)((off + chunk_columns<UPLO == 1>(n, r) - 1) / run - off / run + 1) : 0;
  const int64_t ra = UPLO == 1 ? r : 0;
  const int total = rows + (MODE != 1 ? (int)((UPLO == 1 ? nr : r + 1) - ra) : 0);
  T s = (T)0;
  for (int k = 8 * wave; k < total; k += 8 * kSymvFoldWaves) {
    T v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int q = k + u < total ? k + u : total - 1;
      v[u] = part[(q < rows ? q : slots + ra + q - rows) * n + jl];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) s = k + u < total ? s + v[u] : s;
  }
  __shared__ T red[kSymvFoldWaves][64];
  red[wave][lane] = s;
  __syncthreads();
  if (wave > 0 || j >= n) return;
#pragma unroll
  for (int w = 1; w < kSymvFoldWaves; ++w) s += red[w][lane];
  T v = alpha * s;
  if (beta != (T)0) v = fma(beta, y[j * incy], v);
  y[j * incy] = v;
}

template <typename T>
int symv(wgb_ctx *ctx, int uplo, int64_t n, T alpha, const T *A, int64_t lda, const T *x, int64_t incx,
         T beta, T *y, int64_t incy) {
  int st = wgb::enter(ctx);
  if (st) return st;
  if (uplo != WGB_LOWER && uplo != WGB_UPPER)
    return fail(WGB_ERR_INVALID_VALUE, "uplo must be WGB_LOWER or WGB_UPPER");
  if (n < 0) return fail(WGB_ERR_INVALID_VALUE, "n must be non-negative");
  if (lda < imax(1, n)) return fail(WGB_ERR_INVALID_VALUE, "lda must be >= max(1, n)");
  if (incx <= 0 || incy <= 0) return fail(WGB_ERR_INVALID_VALUE, "incx and incy must be positive");
  if (n == 0) return WGB_OK;
  if (alpha == (T)0 && beta == (T)1) {
    // dsymv: reference BLAS's quick return, no kernel (src/dsymv/dsymv.mjs:116);
    // ssymv runs (and times) its kernels there (src/ssymv/ssymv.mjs): an
    // empty span, y untouched
    if (sizeof(T) == 8) return WGB_OK;
    wgb::timing_begin(ctx);
    wgb::timing_end(ctx);
    return WGB_OK;
  }
  if (!y || (alpha != (T)0 && (!A || !x))) return fail(WGB_ERR_INVALID_VALUE, "A, x or y is null");
  wgb::timing_begin(ctx);
  if (alpha == (T)0) {
    scale_y_kernel<T><<<(unsigned)cdiv(n, kThreads), kThreads, 0, ctx->stream>>>(n, beta, y, incy);
    WGB_CHECK_LAUNCH("scale_y_kernel");
    wgb::timing_end(ctx);
    return WGB_OK;
  }
  if (n > kSymvMaxN) return fail(WGB_ERR_INVALID_VALUE, "n too large for one launch");
  const int64_t cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  const SymvPlan plan = uplo == WGB_LOWER ? symv_plan<true>(n, cus) : symv_plan<false>(n, cus);
  if ((st = wgb::ensure_op_workspace(ctx, (size_t)((plan.slots + cdiv(n, kChunkRows)) * n) * sizeof(T)))) return st;
  T *part = static_cast<T *>(ctx->op_ws);
  auto launch = [&](auto vec_tag) {
    constexpr int VEC = decltype(vec_tag)::value;
    auto kern = uplo == WGB_LOWER ? symv_kernel<T, VEC, 1> : symv_kernel<T, VEC, 2>;
    kern<<<(unsigned)plan.blocks, kThreads, 0, ctx->stream>>>(n, plan.run, plan.slots, A, lda, x, incx, part);
  };
  const int vec = access_of(n, A, lda);
  if (vec == kVecA)
    launch(std::integral_constant<int, kVecA>{});
  else if (vec == kVecU)
    launch(std::integral_constant<int, kVecU>{});
  else
    launch(std::integral_constant<int, kElems>{});
  WGB_CHECK_LAUNCH("symv_kernel");
  auto fold = uplo == WGB_LOWER ? symv_fold_kernel<T, 1> : symv_fold_kernel<T, 2>;
  fold<<<(unsigned)cdiv(n, 64), 64 * kSymvFoldWaves, 0, ctx->stream>>>(n, plan.run, plan.slots, part, alpha,
                                                                            beta, y, incy);
  WGB_CHECK_LAUNCH("symv_fold_kernel");
  wgb::timing_end(ctx);
  return WGB_OK;
}

// strmv / dtrmv: y <- op(T) x, T the n x n triangle (uplo) of A, unit
// diagonal taken as 1 where diag is WGB_UNIT; on symv_kernel's row sums
// (no transpose, with the column form's zero skip) or column sums
// (transpose), folded as symv's. x and y must not overlap.
template <typename T>
int trmv(wgb_ctx *ctx, int uplo, int trans, int diag, int64_t n, const T *A, int64_t lda, const T *x,
         int64_t incx, T *y, int64_t incy) {
  int st = wgb::enter(ctx);
  if (st) return st;
  if (uplo != WGB_LOWER && uplo != WGB_UPPER)
    return fail(WGB_ERR_INVALID_VALUE, "uplo must be WGB_LOWER or WGB_UPPER");
  if (trans != WGB_NO_TRANS && trans != WGB_TRANS)
    return fail(WGB_ERR_INVALID_VALUE, "trans must be WGB_NO_TRANS or WGB_TRANS");
  if (diag != WGB_NON_UNIT && diag != WGB_UNIT)
    return fail(WGB_ERR_INVALID_VALUE, "diag must be WGB_NON_UNIT or WGB_UNIT");
  if (n < 0) return fail(WGB_ERR_INVALID_VALUE, "n must be non-negative");
  if (lda < imax(1, n)) return fail(WGB_ERR_INVALID_VALUE, "lda must be >= max(1, n)");
  if (incx <= 0 || incy <= 0) return fail(WGB_ERR_INVALID_VALUE, "incx and incy must be positive");
  if (n == 0) return WGB_OK;
  if (!A || !x || !y) return fail(WGB_ERR_INVALID_VALUE, "A, x or y is null");
  if (n > kSymvMaxN) return fail(WGB_ERR_INVALID_VALUE, "n too large for one launch");
  const int64_t cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  const SymvPlan plan = uplo == WGB_LOWER ? symv_plan<true>(n, cus) : symv_plan<false>(n, cus);
  if ((st = wgb::ensure_op_workspace(ctx, (size_t)((plan.slots + cdiv(n, kChunkRows)) * n) * sizeof(T)))) return st;
  T *part = static_cast<T *>(ctx->op_ws);
  wgb::timing_begin(ctx);
  const int vec = access_of(n, A, lda);
  const bool lower = uplo == WGB_LOWER, nt = trans == WGB_NO_TRANS, unit = diag == WGB_UNIT;
  auto launch = [&](auto kern) {
    kern<<<(unsigned)plan.blocks, kThreads, 0, ctx->stream>>>(n, plan.run, plan.slots, A, lda, x, incx, part);
  };
  // one instantiation per (vector loads, uplo, form, unit)
  auto pick = [&](auto vec_tag, auto lower_tag, auto mode_tag, auto unit_tag) {
    launch(symv_kernel<T, decltype(vec_tag)::value, decltype(lower_tag)::value ? 1 : 2,
                       decltype(mode_tag)::value, decltype(unit_tag)::value>);
  };
  auto by_unit = [&](auto v, auto l, auto m) {
    if (unit)
      pick(v, l, m, std::true_type{});
    else
      pick(v, l, m, std::false_type{});
  };
  auto by_mode = [&](auto v, auto l) {
    if (nt)
      by_unit(v, l, std::integral_constant<int, 1>{});
    else
      by_unit(v, l, std::integral_constant<int, 2>{});
  };
  auto by_lower = [&](auto v) {
    if (lower)
      by_mode(v, std::true_type{});
    else
      by_mode(v, std::false_type{});
  };
  if (vec == kVecA)
    by_lower(std::integral_constant<int, kVecA>{});
  else if (vec == kVecU)
    by_lower(std::integral_constant<int, kVecU>{});
  else
    by_lower(std::integral_constant<int, kElems>{});
  WGB_CHECK_LAUNCH("symv_kernel");
  auto fold = [&](auto kern) {
    kern<<<(unsigned)cdiv(n, 64), 64 * kSymvFoldWaves, 0, ctx->stream>>>(n, plan.run, plan.slots, part, (T)1, (T)0, y,
                                                                         incy);
  };
  if (lower)
    fold(nt ? symv_fold_kernel<T, 1, 1> : symv_fold_kernel<T, 1, 2>);
  else
    fold(nt ? symv_fold_kernel<T, 2, 1> : symv_fold_kernel<T, 2, 2>);
  WGB_CHECK_LAUNCH("symv_fold_kernel");
  wgb::timing_end(ctx);
  return WGB_OK;
}

int64_t split_count(int64_t want, int64_t most) {
  if (want > most) want = most;
  if (want > 65535) want = 65535;  // grid y limit
  return want < 1 ? 1 : want;
}

// The N form's blocks: narrow (256 rows, the columns shared by kColWaves waves)
// or wide (1024 rows), how many side by side, and columns per split.
//
// Narrow: at most one block per CU where one per 256 rows is not more already
// (a few more put two on some CUs, which the rest waits for: dgemv 15000 x 4000
// in 59 x 5 blocks 127 us, in 59 x 4 94); whole steps for every wave.
//
// Either kind reads at about the same rate per CU, so the one that leaves the
// busiest CU the smaller part of A (fp64: by 1/64) is the faster one, while the wide ones are
// fewer than the CUs and hold kMinColsN columns or fewer (narrow / wide, us):
// dgemv 1024 x 57000 88 / 92, 65000 100 / 98, 964 x 61000 102 / 94, 25000 x 2304
// 100 / 91, 50000 x 768 62 / 82, 230000 x 200 70 / 66. In fp32 the CUs read narrow
// blocks faster, and a wide block of fewer rows takes as long (sgemv 15000 x 4352
// 46 / 47, 25000 x 2304 41 / 45, 800 x 65000 37 / 46): narrow ones wherever they are
// one per CU, else up to 15/16 of the wide ones' rows (205000 x 200 31 / 33,
// 255000 x 200 41 / 37) or over few columns (255000 x 32 7.7 / 8.9). Up to
// 512 rows half of a wide block's waves and more would have none (sgemv 250 x
// 70000 18 / 42, dgemv 512 x 160000 121 / 160).
struct PlanN {
  bool narrow;
  int64_t blocks, per;
};
template <typename T>
PlanN plan_n(int64_t m, int64_t n) {
  const int64_t cus = kTargetBlocksN, unit = kColWaves * kStepN;
  PlanN wide = {false, cdiv(m, 4 * kThreads), 0}, narrow = {true, cdiv(m, 256), 0};
  wide.per = cdiv(n, split_count(cdiv(cus, wide.blocks), cdiv(n, kMinColsN)));
  narrow.per = cdiv(cdiv(n, split_count(cus / narrow.blocks, cdiv(n, kMinColsNarrow))), unit) * unit;
  if (m <= 512) return narrow;
  if (wide.blocks * cdiv(n, kMinColsN) >= cus) return wide;
  const int64_t cols = narrow.per < n ? narrow.per : n;
  const int64_t rounds = cdiv(narrow.blocks * cdiv(n, narrow.per), cus);
  bool better;
  if (sizeof(T) == 8)
    better = 64 * rounds * cols * 256 < 63 * wide.per * (m < 4 * kThreads ? m : 4 * kThreads);
  else
    better = rounds == 1 || n <= kMinColsN / 2 || 16 * narrow.blocks < 15 * 4 * cus;
  return better ? narrow : wide;
}

// sgemv / dgemv on the kernels above. dgemv keeps reference BLAS's quick
// return for alpha == 0 with beta == 1 (src/dgemv/dgemv.mjs:126: no
// kernel, y untouched bit for bit); sgemv times an empty span there, as
// wgblas runs a kernel (src/sgemv/sgemv.mjs:85 returns early only for m or
// n == 0).
template <typename T>
int gemv(wgb_ctx *ctx, int trans, int64_t m, int64_t n, T alpha, const T *A, int64_t lda,
         const T *x, int64_t incx, T beta, T *y, int64_t incy) {
  int st = wgb::enter(ctx);
  if (st) return st;
  if (trans != WGB_NO_TRANS && trans != WGB_TRANS)
    return fail(WGB_ERR_INVALID_VALUE, "trans must be WGB_NO_TRANS or WGB_TRANS");
  if (m < 0 || n < 0) return fail(WGB_ERR_INVALID_VALUE, "m and n must be non-negative");
  if (lda < imax(1, m)) return fail(WGB_ERR_INVALID_VALUE, "lda must be >= max(1, m)");
  if (incx <= 0 || incy <= 0) return fail(WGB_ERR_INVALID_VALUE, "incx and incy must be positive");
  // reference BLAS quick return: nothing to do, y untouched
  if (m == 0 || n == 0) return WGB_OK;
  if (alpha == (T)0 && beta == (T)1) {
    if (sizeof(T) == 8) return WGB_OK;
    // y untouched; this call's empty span, so per-call timing reports it
    // rather than an older call
    wgb::timing_begin(ctx);
    wgb::timing_end(ctx);
    return WGB_OK;
  }
  if (!y || (alpha != (T)0 && (!A || !x))) return fail(WGB_ERR_INVALID_VALUE, "A, x or y is null");
  const bool nt = trans == WGB_NO_TRANS;
  const int64_t len = nt ? m : n;  // length of y
  wgb::timing_begin(ctx);
  if (alpha == (T)0) {
    scale_y_kernel<T><<<(unsigned)cdiv(len, kThreads), kThreads, 0, ctx->stream>>>(len, beta, y, incy);
    WGB_CHECK_LAUNCH("scale_y_kernel");
    wgb::timing_end(ctx);
    return WGB_OK;
  }
  // blocks along the output; split the contraction dimension until about
  // the target block count streams A (N: plan_n; T: >= 256
  // rows, a multiple of 256 so every split starts aligned)
  const int cpw = m <= kShortColsRows ? kColsPerWaveShort : kColsPerWave;  // T form
  const PlanN plan = nt ? plan_n<T>(m, n) : PlanN{};
  const int64_t bx = nt ? plan.blocks : cdiv(cdiv(n, cpw), kThreads / 64);
  const int64_t per = nt ? plan.per : cdiv(cdiv(m, split_count(cdiv(kTargetBlocks, bx), cdiv(m, 256))), 256) * 256;
  const int64_t splits = nt ? cdiv(n, per) : cdiv(m, per);
  T *part = nullptr;
  if (splits > 1) {
    // partials, then the fold passes' group sums after them
    const int64_t groups = cdiv(splits, kFold);
    if ((st = wgb::ensure_op_workspace(ctx, (size_t)((splits + groups) * len) * sizeof(T))))
      return st;
    part = static_cast<T *>(ctx->op_ws);
  }
  dim3 grid((unsigned)bx, (unsigned)splits);
  if (nt) {
    const int vec = access_of(m, A, lda);
    auto launch = [&](auto kern, int threads) {
      kern<<<grid, threads, 0, ctx->stream>>>(m, n, A, lda, x, incx, per, part, alpha, beta, y, incy);
    };
    if (plan.narrow)
      launch(vec == kVecA   ? gemv_n_kernel<T, kVecA, 1, kColWaves>
             : vec == kVecU ? gemv_n_kernel<T, kVecU, 1, kColWaves>
                            : gemv_n_kernel<T, kElems, 1, kColWaves>,
             64 * kColWaves);
    else
      launch(vec == kVecA   ? gemv_n_kernel<T, kVecA, 4, 1>
             : vec == kVecU ? gemv_n_kernel<T, kVecU, 4, 1>
                            : gemv_n_kernel<T, kElems, 4, 1>,
             kThreads);
    WGB_CHECK_LAUNCH("gemv_n_kernel");
  } else {
    const int vec = incx != 1 ? kElems : access_t(m, n, A, lda);
    auto launch = [&](auto vec_tag) {
      constexpr int VEC = decltype(vec_tag)::value;
      auto kern = cpw == kColsPerWaveShort ? gemv_t_kernel<T, VEC, kColsPerWaveShort> : gemv_t_kernel<T, VEC, kColsPerWave>;
      kern<<<grid, kThreads, 0, ctx->stream>>>(m, n, A, lda, x, incx, per, part, alpha, beta, y, incy);
    };
    if (vec == kVecA)
      launch(std::integral_constant<int, kVecA>{});
    else if (vec == kVecU)
      launch(std::integral_constant<int, kVecU>{});
    else
      launch(std::integral_constant<int, kElems>{});
    WGB_CHECK_LAUNCH("gemv_t_kernel");
  }
  if (part) {
    // fold passes until one group of at most kFold remains; each pass
    // alternates between the two halves of the workspace
    T *src = part, *dst = part + splits * len;
    int64_t k = splits;
    while (k > kFold) {
      const int64_t groups = cdiv(k, kFold);
      gemv_fold_kernel<T><<<dim3((unsigned)cdiv(len, kThreads), (unsigned)groups), kThreads, 0,
                         ctx->stream>>>(len, k, src, dst, alpha, beta, y, incy);
      WGB_CHECK_LAUNCH("gemv_fold_kernel");
      T *t = src;
      src = dst;
      dst = t;
      k = groups;
    }
    gemv_fold_kernel<T><<<dim3((unsigned)cdiv(len, kThreads), 1), kThreads, 0, ctx->stream>>>(
        len, k, src, nullptr, alpha, beta, y, incy);
    WGB_CHECK_LAUNCH("gemv_fold_kernel");
  }
  wgb::timing_end(ctx);
  return WGB_OK;
}

}  // namespace

extern "C" int wgb_sgemv(wgb_ctx *ctx, int trans, int64_t m, int64_t n, float alpha,
                         const float *A, int64_t lda, const float *x, int64_t incx, float beta,
                         float *y, int64_t incy) {
  return gemv<float>(ctx, trans, m, n, alpha, A, lda, x, incx, beta, y, incy);
}

extern "C" int wgb_sger(wgb_ctx *ctx, int64_t m, int64_t n, float alpha, const float *x,
                        int64_t incx, const float *y, int64_t incy, float *A, int64_t lda) {
  return rank_update<float>(ctx, 0, false, m, n, alpha, x, incx, y, incy, A, lda);
}

extern "C" int wgb_dger(wgb_ctx *ctx, int64_t m, int64_t n, double alpha, const double *x,
                        int64_t incx, const double *y, int64_t incy, double *A, int64_t lda) {
  return rank_update<double>(ctx, 0, false, m, n, alpha, x, incx, y, incy, A, lda);
}

extern "C" int wgb_ssyr(wgb_ctx *ctx, int uplo, int64_t n, float alpha, const float *x,
                        int64_t incx, float *A, int64_t lda) {
  if (uplo == 0) return fail(WGB_ERR_INVALID_VALUE, "uplo must be WGB_LOWER or WGB_UPPER");
  return rank_update<float>(ctx, uplo, false, n, n, alpha, x, incx, x, incx, A, lda);
}

extern "C" int wgb_dsyr(wgb_ctx *ctx, int uplo, int64_t n, double alpha, const double *x,
                        int64_t incx, double *A, int64_t lda) {
  if (uplo == 0) return fail(WGB_ERR_INVALID_VALUE, "uplo must be WGB_LOWER or WGB_UPPER");
  return rank_update<double>(ctx, uplo, false, n, n, alpha, x, incx, x, incx, A, lda);
}

extern "C" int wgb_ssyr2(wgb_ctx *ctx, int uplo, int64_t n, float alpha, const float *x,
                         int64_t incx, const float *y, int64_t incy, float *A, int64_t lda) {
  if (uplo == 0) return fail(WGB_ERR_INVALID_VALUE, "uplo must be WGB_LOWER or WGB_UPPER");
  return rank_update<float>(ctx, uplo, true, n, n, alpha, x, incx, y, incy, A, lda);
}

extern "C" int wgb_dsyr2(wgb_ctx *ctx, int uplo, int64_t n, double alpha, const double *x,
                         int64_t incx, const double *y, int64_t incy, double *A, int64_t lda) {
  if (uplo == 0) return fail(WGB_ERR_INVALID_VALUE, "uplo must be WGB_LOWER or WGB_UPPER");
  return rank_update<double>(ctx, uplo, true, n, n, alpha, x, incx, y, incy, A, lda);
}

extern "C" int wgb_ssymv(wgb_ctx *ctx, int uplo, int64_t n, float alpha, const float *A,
                         int64_t lda, const float *x, int64_t incx, float beta, float *y,
                         int64_t incy) {
  return symv<float>(ctx, uplo, n, alpha, A, lda, x, incx, beta, y, incy);
}

extern "C" int wgb_dsymv(wgb_ctx *ctx, int uplo, int64_t n, double alpha, const double *A,
                         int64_t lda, const double *x, int64_t incx, double beta, double *y,
                         int64_t incy) {
  return symv<double>(ctx, uplo, n, alpha, A, lda, x, incx, beta, y, incy);
}

extern "C" int wgb_strmv(wgb_ctx *ctx, int uplo, int trans, int diag, int64_t n, const float *A,
                         int64_t lda, const float *x, int64_t incx, float *y, int64_t incy) {
  return trmv<float>(ctx, uplo, trans, diag, n, A, lda, x, incx, y, incy);
}

extern "C" int wgb_dtrmv(wgb_ctx *ctx, int uplo, int trans, int diag, int64_t n, const double *A,
                         int64_t lda, const double *x, int64_t incx, double *y, int64_t incy) {
  return trmv<double>(ctx, uplo, trans, diag, n, A, lda, x, incx, y, incy);
}

extern "C" int wgb_dgemv(wgb_ctx *ctx, int trans, int64_t m, int64_t n, double alpha,
                         const double *A, int64_t lda, const double *x, int64_t incx, double beta,
                         double *y, int64_t incy) {
  return gemv<double>(ctx, trans, m, n, alpha, A, lda, x, incx, beta, y, incy);
}

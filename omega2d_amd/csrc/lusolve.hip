// lusolve.hip - solves with the kept LU factors (lu.hip's layout), for src/BEM.h:169-234.
//
// A library triangular solve of one right-hand side runs as a chain on one workgroup: 0.37 ms
// (L) and 0.55 ms (U) at order 2049, where the factors are 34 MB, 7 us of memory traffic. Here the
// chain is one launch per kSB rows: every workgroup of a launch forms the block's solution from
// the inverse of its diagonal block (kSB x kSB, prepared once per factorisation) and takes it off
// its own rows of what is left, so a launch spreads its column panel over the chip and the
// launches' own latency (2 x 33 at order 2049, 4 us each) is what remains: 0.92 -> 0.27 ms a solve,
// after 0.017 ms for the diagonal blocks.
// Row interchanges are applied to the right-hand side as a gather by the permutation that the
// factorisation composed block by block.
//
// With the explicit inverse a solve is one matrix-vector product, split over columns so that the
// read is spread over the chip, partial sums added in order: 83 -> 12.5 us at order 2049; up to order
// kOnceMax in one launch.
#include <algorithm>

#include "nbody.h"
#include "o2d_runtime.h"

namespace o2d {

namespace {

constexpr int kSB = 64;     // rows per block of a triangular solve
constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kChunk = 32;  // columns per workgroup of the matrix-vector product
constexpr int kOnceT = 1024, kOnceMax = 256;  // threads and largest order of its form in one launch
static_assert(kSB == 64, "a lane per row of a block");

// The inverses of the diagonal blocks of L (unit lower; blockIdx.y = 0) and U (upper; 1), padded
// with the identity past n: dinv[((y nblk) + block) kSB^2 + k kSB + i] = inverse(i, k). Each wave inverts
// one of the four diagonal kSub x kSub blocks by substitution, four lanes to a column; then, twice,
// pairs of inverted blocks X11, X22 are joined over the block M21 between them: X21 = -X22 (M21 X11).
// Bound by the latency of its chain: substitution over all 64 rows took 38 us at any order, this takes
// 17 (the factorisation of order 50 with one solve 178 and 157).
constexpr int kSub = 16;

// x[h + i][k] = -sum_l X22[i][l] (M21 X11)[l][k] for the kH x kH block below and left of the middle of the
// 2 kH rows from r on; the sum's first product stands in x's own place in between. PAIRS of them at a time.
template <int kH, int PAIRS>
__device__ void join_blocks(const double (*m)[kSB + 1], double (*x)[kSB + 1]) {
  constexpr int kEach = PAIRS * kH * kH / kBlock;
  static_assert(PAIRS * 2 * kH == kSB && kEach >= 1, "all rows, whole shares");
  double v[kEach];
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
    for (int u = 0; u < kEach; ++u) {
      const int e = threadIdx.x + u * kBlock;
      const int r = e / (kH * kH) * 2 * kH, i = e / kH % kH, k = e % kH;
      double s = 0.0;
#pragma unroll 8
      for (int l = 0; l < kH; ++l)
        s = pass == 0 ? __builtin_fma(m[r + kH + i][r + l], x[r + l][r + k], s)
                      : __builtin_fma(-x[r + kH + i][r + kH + l], x[r + kH + l][r + k], s);
      v[u] = s;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kEach; ++u) {
      const int e = threadIdx.x + u * kBlock;
      x[e / (kH * kH) * 2 * kH + kH + e / kH % kH][e / (kH * kH) * 2 * kH + e % kH] = v[u];
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(kBlock) void lu_diag_inverse_kernel(int n, int nblk,
                                                                 const double* __restrict__ lu,
                                                                 double* __restrict__ dinv) {
  static_assert(kSB == kWaves * kSub && 64 == 4 * kSub, "a wave per block, four lanes per column");
  __shared__ double m[kSB][kSB + 1];  // m[r][c]: the block; of U, its mirror
  __shared__ double x[kSB][kSB + 1];  // x[i][k]
  const int t = threadIdx.x, b = blockIdx.x, r0 = b * kSB;
  const bool upper = blockIdx.y != 0;
  // U is solved as the lower triangle that reversing rows and columns makes of it
#pragma unroll 4
  for (int e = t; e < kSB * kSB; e += kBlock) {
    const int r = e % kSB, c = e / kSB;
    const bool in = r0 + r < n && r0 + c < n;
    double v = in ? lu[(int64_t)(r0 + c) * n + r0 + r] : 0.0;
    if (upper ? r > c : r < c) v = 0.0;
    if (r == c && (!upper || !in)) v = 1.0;
    if (upper) m[kSB - 1 - r][kSB - 1 - c] = v;
    else m[r][c] = v;
    x[r][c] = 0.0;
  }
  __syncthreads();
  {
    const int o = t / 64 * kSub, k = t % 64 / 4, q = t % 4;  // rows of this wave's block, column, lane
    double mine[kSub / 4];  // x[q + 4 l][k]
#pragma unroll
    for (int i = 0; i < kSub; ++i) {
      double s = 0.0;
#pragma unroll
      for (int l = 0; 4 * l < i; ++l)
        if (q + 4 * l < i) s = __builtin_fma(-m[o + i][o + q + 4 * l], mine[l], s);
      s += __shfl_xor(s, 1, 64);
      s += __shfl_xor(s, 2, 64);
      s += k == i ? 1.0 : 0.0;
      if (upper) s /= m[o + i][o + i];
      if (q == i % 4) {
        mine[i / 4] = s;
        x[o + i][o + k] = s;
      }
    }
  }
  __syncthreads();
  join_blocks<kSub, 2>(m, x);
  join_blocks<2 * kSub, 1>(m, x);
  double* out = dinv + ((int64_t)blockIdx.y * nblk + b) * kSB * kSB;
#pragma unroll 4
  for (int e = t; e < kSB * kSB; e += kBlock) {
    const int i = e % kSB, c = e / kSB;
    out[e] = upper ? x[kSB - 1 - i][kSB - 1 - c] : x[i][c];
  }
}

// r = P b (perm[i]: the row of A that row i of the factors is)
__global__ __launch_bounds__(kBlock) void lu_permute_kernel(int n, const int* __restrict__ perm,
                                                            const double* __restrict__ b,
                                                            double* __restrict__ r) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) r[i] = b[perm[i]];
}

// One block step: y = D^-1 r for the rows [c0, c0 + 64) (by every workgroup; the first writes it
// to out), then r[row] -= sum_k A[row, c0 + k] y_k for the workgroup's 64 rows from first on. r
// of the block's own rows is only read and out is another array, so no workgroup waits for
// another. Four waves share the columns.
__global__ __launch_bounds__(kBlock) void lu_step_kernel(int n, const double* __restrict__ lu,
                                                         const double* __restrict__ dinv, int c0,
                                                         int first, int rows,
                                                         double* __restrict__ r,
                                                         double* __restrict__ out) {
  constexpr int kCols = kSB / kWaves;
  __shared__ double part[kWaves][kSB];
  __shared__ double y[kSB];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = first + blockIdx.x * kSB + lane;
  const bool mine = row < first + rows;
  // the update's column entries, on their way while the block is solved
  double a[kCols];
#pragma unroll
  for (int k = 0; k < kCols; ++k) {
    const int c = c0 + wave * kCols + k;
    a[k] = mine && c < n ? lu[(int64_t)c * n + row] : 0.0;
  }
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < kCols; ++k) {
    const int c = wave * kCols + k;
    s = __builtin_fma(dinv[c * kSB + lane], c0 + c < n ? r[c0 + c] : 0.0, s);
  }
  part[wave][lane] = s;
  __syncthreads();
  if (wave == 0) {
    s = part[0][lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) s += part[w][lane];
    y[lane] = s;
    if (blockIdx.x == 0 && c0 + lane < n) out[c0 + lane] = s;
  }
  __syncthreads();
  s = 0.0;
#pragma unroll
  for (int k = 0; k < kCols; ++k) s = __builtin_fma(a[k], y[wave * kCols + k], s);
  part[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && mine) {
    s = part[0][lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) s += part[w][lane];
    r[row] -= s;
  }
}

// part[chunk n + row] = sum over the chunk's columns of a[row, c] b[c] (a column-major)
__global__ __launch_bounds__(kBlock) void matvec_kernel(int n, const double* __restrict__ a,
                                                        const double* __restrict__ b,
                                                        double* __restrict__ part) {
  const int row = blockIdx.x * kBlock + threadIdx.x;
  const int c0 = blockIdx.y * kChunk, c1 = c0 + kChunk < n ? c0 + kChunk : n;
  if (row >= n) return;
  double s = 0.0;
#pragma unroll 8
  for (int c = c0; c < c1; ++c) s = __builtin_fma(a[(int64_t)c * n + row], b[c], s);
  part[(int64_t)blockIdx.y * n + row] = s;
}

// x[row] = sum over the chunks of part, in order; four waves share the chunks of 64 rows
__global__ __launch_bounds__(kBlock) void matvec_sum_kernel(int n, int nchunk,
                                                            const double* __restrict__ part,
                                                            double* __restrict__ x) {
  __shared__ double sm[kWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = blockIdx.x * 64 + lane;
  double s = 0.0;
  if (row < n) {
#pragma unroll 8
    for (int c = wave; c < nchunk; c += kWaves) s += part[(int64_t)c * n + row];
  }
  sm[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && row < n) x[row] = ((sm[0][lane] + sm[1][lane]) + sm[2][lane]) + sm[3][lane];
}

// x = a b in one launch, for small orders: a workgroup takes 64 rows, its 16 waves every 16th column, added
// in wave order. Order 50 2.1 us, 3.3 in two launches, 200 4.2 and 4.3, 300 5.6 and 4.7 (in a graph; a call
// by itself, which waits for its launches, 6.9 and 9.3)
__global__ __launch_bounds__(kOnceT) void matvec_once_kernel(int n, const double* __restrict__ a,
                                                             const double* b, double* x) {
  constexpr int kW = kOnceT / 64;
  __shared__ double sm[kW][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = blockIdx.x * 64 + lane;
  double s = 0.0;
  if (row < n) {
#pragma unroll 8
    for (int c = wave; c < n; c += kW) s = __builtin_fma(a[(int64_t)c * n + row], b[c], s);
  }
  sm[wave][lane] = s;
  __syncthreads();
  if (wave != 0 || row >= n) return;
#pragma unroll
  for (int w = 1; w < kW; ++w) s += sm[w][lane];
  x[row] = s;
}

inline int blocks_of(int64_t n) { return (int)((n + kSB - 1) / kSB); }

}  // namespace

// two vectors for the block substitution, one per chunk of columns for the product; the same for both,
// so that the slot stays where it is from one solve to the next (a captured solve keeps its address)
size_t solve_scratch(int64_t n) {
  return sizeof(double) * std::max<int64_t>(2, (n + kChunk - 1) / kChunk) * n;
}

// the diagonal inverses of the factors lu (n x n, leading dimension n), into the kLuDinv slot
int lu_prepare_solve(Device* d, hipStream_t s, int n, const double* lu) {
  const int nblk = blocks_of(n);
  void* p;
  O2D_TRY(slot(d, kLuDinv, sizeof(double) * 2 * nblk * kSB * kSB, s, &p));
  lu_diag_inverse_kernel<<<dim3(nblk, 2), kBlock, 0, s>>>(n, nblk, lu, static_cast<double*>(p));
  O2D_LAUNCH_CHECK();
  return 0;
}

// x = (LU)^-1 P b with the diagonal inverses prepared (x may alias b)
int lu_solve_dev(Device* d, hipStream_t s, int n, const double* lu, const int* perm,
                 const double* b, double* x) {
  const int nblk = blocks_of(n);
  void* p;
  O2D_TRY(slot(d, kSolveTmp, solve_scratch(n), s, &p));
  double *r = static_cast<double*>(p), *y = r + n;
  const double* dl = static_cast<const double*>(d->buf[kLuDinv]);
  const double* du = dl + (int64_t)nblk * kSB * kSB;
  lu_permute_kernel<<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(n, perm, b, r);
  O2D_LAUNCH_CHECK();
  for (int i = 0; i < nblk; ++i) {
    const int c0 = i * kSB, first = c0 + kSB, rows = std::max(0, n - first);
    lu_step_kernel<<<std::max(1, blocks_of(rows)), kBlock, 0, s>>>(
        n, lu, dl + (int64_t)i * kSB * kSB, c0, first, rows, r, y);
    O2D_LAUNCH_CHECK();
  }
  for (int i = nblk - 1; i >= 0; --i) {
    const int c0 = i * kSB;
    lu_step_kernel<<<std::max(1, blocks_of(c0)), kBlock, 0, s>>>(
        n, lu, du + (int64_t)i * kSB * kSB, c0, 0, c0, y, x);
    O2D_LAUNCH_CHECK();
  }
  return 0;
}

// x = A b, A n x n column-major (x may alias b)
int matvec_dev(Device* d, hipStream_t s, int n, const double* a, const double* b, double* x) {
  if (n <= kOnceMax && (x != b || n <= 64)) {  // (in place, another workgroup could still read b)
    matvec_once_kernel<<<blocks_of(n), kOnceT, 0, s>>>(n, a, b, x);
    O2D_LAUNCH_CHECK();
    return 0;
  }
  const int nchunk = (n + kChunk - 1) / kChunk;
  void* p;
  O2D_TRY(slot(d, kSolveTmp, solve_scratch(n), s, &p));
  double* part = static_cast<double*>(p);
  matvec_kernel<<<dim3((n + kBlock - 1) / kBlock, nchunk), kBlock, 0, s>>>(n, a, b, part);
  O2D_LAUNCH_CHECK();
  matvec_sum_kernel<<<blocks_of(n), kBlock, 0, s>>>(n, nchunk, part, x);
  O2D_LAUNCH_CHECK();
  return 0;
}

}  // namespace o2d

// vorticity.hip - Gaussian vorticity of particles at targets, points_affect_points_vorticity
// (src/InfluenceVort.h:47-126, the x86 loop :103-117):
//   tw_i += sum_j 2 s_j exp(-d_ij^2 / r_j^2) / r_j^2      (unscaled; finalize_vels adds 1/2pi)
// in fp64. A pair with d^2/r^2 > 746 contributes exactly +-0 (exp underflows to 0 in double), so
// its exponential is skipped without changing the sum. The exponential is a table-driven exp(-x) on
// [0, 746).
//
// Sources and targets go in Morton order, and a group of 16 targets meets only the boxes of 32 sources
// that its own box can reach. The order is fixed, so sums are reproducible. (A kernel without boxes, two
// targets a lane, in orders from 4,096 sources and 1,024 targets on, took 50 us at 1,000 particles against
// 26, 64 at 4,000 against 47, 262 for 200,000 on 50 points against 111 and 322 for 3,000 on 200,000 against
// 79. Where the radii reach across the whole domain the boxes leave nothing out, and a call that it did
// not order pays for its orders: 3,000 on 200,000 461 against 516, 1,000 on 200,000 184 against 204;
// 50,000 on themselves 1,957 against 1,994. Radii are known on the device only.)
//
// A NaN position or radius adds NaN, as in the reference (its tile and its targets' group are never
// skipped); a non-finite strength or a zero radius beyond the bound adds nothing, where the
// reference's inf*0 gives NaN.
#include <algorithm>

#include "nbody.h"
#include "o2d_runtime.h"

namespace o2d {

namespace {

constexpr int kBlock = 256;
constexpr int kTile = 256;
constexpr double kUnderflow = 746.0;  // exp(-x) == 0 in double for every x above this
constexpr int kSub = 32;                   // sources per box of a tile
constexpr int kSubs = kTile / kSub;
constexpr int kGroup = 16;                 // targets per wave of vort_near_kernel
constexpr int kNearT = 256;                // its threads
constexpr int kNearTargets = 32;           // its targets: two groups, two waves each
constexpr int kPer = 2;                    // targets a lane holds
// rows of tiles that its grid is cut into: kNearWgs workgroups per CU, and at least kNearRows (the
// workgroups of dense regions last longest, and without rows the launch waits for them): 200,000 wake
// particles take 394 us a call with one row, 347 with two, 330 with four; 100,000 209, 173 (two)
// and 148 (three); 20,000 51 with 12 workgroups per CU and 65 with 48
constexpr int64_t kNearWgs = 12, kNearRows = 3;
// as long as a row keeps kRowTiles tiles: with fewer the rows' own work is most of it (3,000 particles on
// 200,000 points 106 us with three rows, 76 with one; 12,000 152 and 141)
constexpr int64_t kRowTiles = 32;
constexpr int64_t kPartialBytes = int64_t(1) << 30;  // the cap on the rows' partial sums

struct alignas(16) VSrc {
  double x, y, rr, c;  // position, 1/r^2, 2 s / r^2
};

// 2^(j/64), j = 0..63, each the double nearest to the exact value
__constant__ double kExp2Tab[64] = {
    0x1.0000000000000p+0, 0x1.02c9a3e778061p+0, 0x1.059b0d3158574p+0, 0x1.0874518759bc8p+0,
    0x1.0b5586cf9890fp+0, 0x1.0e3ec32d3d1a2p+0, 0x1.11301d0125b51p+0, 0x1.1429aaea92de0p+0,
    0x1.172b83c7d517bp+0, 0x1.1a35beb6fcb75p+0, 0x1.1d4873168b9aap+0, 0x1.2063b88628cd6p+0,
    0x1.2387a6e756238p+0, 0x1.26b4565e27cddp+0, 0x1.29e9df51fdee1p+0, 0x1.2d285a6e4030bp+0,
    0x1.306fe0a31b715p+0, 0x1.33c08b26416ffp+0, 0x1.371a7373aa9cbp+0, 0x1.3a7db34e59ff7p+0,
    0x1.3dea64c123422p+0, 0x1.4160a21f72e2ap+0, 0x1.44e086061892dp+0, 0x1.486a2b5c13cd0p+0,
    0x1.4bfdad5362a27p+0, 0x1.4f9b2769d2ca7p+0, 0x1.5342b569d4f82p+0, 0x1.56f4736b527dap+0,
    0x1.5ab07dd485429p+0, 0x1.5e76f15ad2148p+0, 0x1.6247eb03a5585p+0, 0x1.6623882552225p+0,
    0x1.6a09e667f3bcdp+0, 0x1.6dfb23c651a2fp+0, 0x1.71f75e8ec5f74p+0, 0x1.75feb564267c9p+0,
    0x1.7a11473eb0187p+0, 0x1.7e2f336cf4e62p+0, 0x1.82589994cce13p+0, 0x1.868d99b4492edp+0,
    0x1.8ace5422aa0dbp+0, 0x1.8f1ae99157736p+0, 0x1.93737b0cdc5e5p+0, 0x1.97d829fde4e50p+0,
    0x1.9c49182a3f090p+0, 0x1.a0c667b5de565p+0, 0x1.a5503b23e255dp+0, 0x1.a9e6b5579fdbfp+0,
    0x1.ae89f995ad3adp+0, 0x1.b33a2b84f15fbp+0, 0x1.b7f76f2fb5e47p+0, 0x1.bcc1e904bc1d2p+0,
    0x1.c199bdd85529cp+0, 0x1.c67f12e57d14bp+0, 0x1.cb720dcef9069p+0, 0x1.d072d4a07897cp+0,
    0x1.d5818dcfba487p+0, 0x1.da9e603db3285p+0, 0x1.dfc97337b9b5fp+0, 0x1.e502ee78b3ff6p+0,
    0x1.ea4afa2a490dap+0, 0x1.efa1bee615a27p+0, 0x1.f50765b6e4540p+0, 0x1.fa7c1819e90d8p+0,
};

// exp(-x) for 0 <= x < 746 (NaN for NaN), by Tang's table-driven method (P. T. P. Tang,
// ACM TOMS 15(2), 1989): -x = n ln2/64 + r with n = rint(-64 x/ln2) and |r| <= ln2/128, taken
// as r = (-x - n L1) - n L2 with ln2/64 = L1 + L2 and L1 of 30 bits, so n L1 and the first
// difference are exact; then exp(-x) = 2^m 2^(j/64) (1 + q(r)), n = 64 m + j, with q the
// degree-6 Taylor polynomial of e^r - 1 (remainder below 2^-60 relative). tab holds kExp2Tab.
// Checked against long double expl on 40 million points of the range: within 1.01 ulp, and
// within 1 unit of 2^-1074 where the result is subnormal.
__device__ __forceinline__ double exp_neg(double x, const double* tab) {
  const double y = -x;
  const double n = rint(y * 0x1.71547652b82fep+6);
  double r = fma(-n, 0x1.62e42ffp-7, y);
  r = fma(-n, -0x1.718432a1b0e26p-41, r);
  const int ni = (int)n;
  const int j = ni & 63;
  const int m = ni >> 6;  // floor(n / 64): n = 64 m + j
  double q = fma(r, 1.0 / 720.0, 1.0 / 120.0);
  q = fma(r, q, 1.0 / 24.0);
  q = fma(r, q, 1.0 / 6.0);
  q = fma(r, q, 0.5);
  q = fma(r, q, 1.0);
  q *= r;
  const double t = tab[j];
  return ldexp(fma(t, q, t), m);
}

// the staged record of a source
__device__ __forceinline__ VSrc vsrc_of(double x, double y, double s, double r) {
  const double r2 = r * r;
  const double rr = 1.0 / r2;
  return VSrc{x, y, rr, 2.0 * s * rr};
}

// the smallest and largest of v over aligned groups of 32 lanes
__device__ __forceinline__ double min32(double v) {
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ double max32(double v) { return -min32(-v); }

// LDS writes of this wave visible to its own later reads, and no compiler reordering across
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A box of source positions with their smallest 1/r^2. A NaN position or radius makes it unbounded.
struct VBox {
  double x0, x1, y0, y1, rr;
};

// the sources in the order sorder as staged records, the box of every kSub of them (sub) and of
// every tile of kTile (tile), padded to whole tiles with the last source at zero strength. One
// workgroup per tile.
__global__ __launch_bounds__(kBlock) void vort_gather_kernel(int64_t ns, const double* __restrict__ sx,
                                                             const double* __restrict__ sy,
                                                             const double* __restrict__ ss,
                                                             const double* __restrict__ sr,
                                                             const uint32_t* __restrict__ sorder,
                                                             VSrc* __restrict__ vs,
                                                             VBox* __restrict__ sub,
                                                             VBox* __restrict__ tile) {
  static_assert(kTile == kBlock && kSub == 32, "a tile per workgroup, two boxes per wave");
  __shared__ VBox sm[kSubs];
  const int t = threadIdx.x;
  const int64_t g = (int64_t)blockIdx.x * kBlock + t;
  const int64_t j = sorder[g < ns ? g : ns - 1];
  VSrc q = vsrc_of(sx[j], sy[j], ss[j], sr[j]);
  if (g >= ns) q.c = 0.0;
  vs[g] = q;
  const bool bad = !(q.x == q.x) || !(q.y == q.y) || !(q.rr == q.rr);
  VBox b;
  b.x0 = min32(bad ? -INFINITY : q.x);
  b.x1 = max32(bad ? INFINITY : q.x);
  b.y0 = min32(bad ? -INFINITY : q.y);
  b.y1 = max32(bad ? INFINITY : q.y);
  b.rr = min32(bad ? 0.0 : q.rr);
  if ((t & (kSub - 1)) == 0) {
    sm[t / kSub] = b;
    sub[(int64_t)blockIdx.x * kSubs + t / kSub] = b;
  }
  __syncthreads();
  if (t != 0) return;
  for (int k = 1; k < kSubs; ++k) {
    b.x0 = fmin(b.x0, sm[k].x0);
    b.x1 = fmax(b.x1, sm[k].x1);
    b.y0 = fmin(b.y0, sm[k].y0);
    b.y1 = fmax(b.y1, sm[k].y1);
    b.rr = fmin(b.rr, sm[k].rr);
  }
  tile[blockIdx.x] = b;
}

// true unless every pair of source box b and target box (x0, x1, y0, y1) lies beyond the underflow
// bound, by a relative margin of 2^-40, far above the rounding of this test and of a pair's own
__device__ __forceinline__ bool box_near(const VBox& b, double x0, double x1, double y0, double y1) {
  const double dx = fmax(0.0, fmax(b.x0 - x1, x0 - b.x1));
  const double dy = fmax(0.0, fmax(b.y0 - y1, y0 - b.y1));
  return !((dx * dx + dy * dy) * b.rr * (1.0 - 0x1p-40) > kUnderflow);
}

// Targets and sources in Morton order. Bound by the fp64 vector units: an exponential is 20 of a
// pair's 26 operations, and the boxes decide how many pairs that add exactly 0 are met. A workgroup
// takes 32 targets; wave w holds group w % 2 of 16 of them, two a lane, each in eight lanes that take every
// eighth source, and the two waves of a group take the even and the odd boxes. The source tiles that
// the workgroup's box reaches are listed 256 at a time (in order), and a wave takes the boxes of 32
// sources in them that its own 16 targets reach, without waiting for the others. For 200,000 wake
// particles (radius 0.005, 1.65e8 pairs within the bound) that is 4.0e8 pairs; 64 targets against tiles
// of 256 were 9.7e8. 735 us and 40 for the sum over chunks -> 306 us and 8. Staging whole tiles between
// barriers took 548 us, exponentials without the branch around them 60% longer. One target a lane reads
// LDS twice as often for a pair, which shows where most pairs are near: 50,000 particles that all are
// 2,050 us a call, two 1,990, 200,000 of radius 0.02 6,340 and 6,070, 200,000 wake particles 334 and 322; six
// waves a SIMD, without spills, where registers alone would leave five.
//
// blockIdx.y takes the listed tiles y, y + gridDim.y, ...; out: tw by torder when gridDim.y is 1, else
// the partial sums part[y nt + p] of the target at position p.
__global__ __launch_bounds__(kNearT, 6) void vort_near_kernel(int64_t nt, const double* __restrict__ tx,
                                                           const double* __restrict__ ty,
                                                           const uint32_t* __restrict__ torder,
                                                           int64_t ntiles, const VSrc* __restrict__ vs,
                                                           const VBox* __restrict__ sub,
                                                           const VBox* __restrict__ tbox,
                                                           double* __restrict__ tw,
                                                           double* __restrict__ part) {
  constexpr int kWaves = kNearT / 64, kGroups = kNearTargets / kGroup;
  constexpr int kSpan = kGroup / kPer, kLanes = 64 / kSpan;
  static_assert(kWaves == 2 * kGroups && kSub % kLanes == 0, "two waves a group, whole shares");
  static_assert(sizeof(VSrc) * kSub == 64 * sizeof(double2), "a box's sources are one load a lane");
  __shared__ VSrc staged[kWaves][kSub];
  __shared__ double e2t[64];  // kExp2Tab
  __shared__ double gb[kWaves][4];
  __shared__ uint32_t list[kNearT], found[kWaves];
  __shared__ double sum[kGroups][kGroup];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, group = wave % kGroups;
  const int half = wave / kGroups, share = lane / kSpan;
  VSrc* mine = staged[wave];
  if (t < 64) e2t[t] = kExp2Tab[t];
  const int64_t p0 = (int64_t)blockIdx.x * kNearTargets + group * kGroup + lane % kSpan;
  uint32_t o[kPer];
  double px[kPer], py[kPer], acc[kPer];
  // the group's box, and the workgroup's (a NaN position: unbounded)
  double x0 = INFINITY, x1 = -INFINITY, y0 = INFINITY, y1 = -INFINITY;
#pragma unroll
  for (int e = 0; e < kPer; ++e) {
    const int64_t p = p0 + e * kSpan;
    o[e] = torder[p < nt ? p : nt - 1];
    px[e] = tx[o[e]];
    py[e] = ty[o[e]];
    acc[e] = 0.0;
    const bool bad = !(px[e] == px[e]) || !(py[e] == py[e]);
    x0 = fmin(x0, bad ? -INFINITY : px[e]);
    x1 = fmax(x1, bad ? INFINITY : px[e]);
    y0 = fmin(y0, bad ? -INFINITY : py[e]);
    y1 = fmax(y1, bad ? INFINITY : py[e]);
  }
#pragma unroll
  for (int s = kSpan / 2; s > 0; s >>= 1) {
    x0 = fmin(x0, __shfl_xor(x0, s, 64));
    x1 = fmax(x1, __shfl_xor(x1, s, 64));
    y0 = fmin(y0, __shfl_xor(y0, s, 64));
    y1 = fmax(y1, __shfl_xor(y1, s, 64));
  }
  if (lane == 0) {
    gb[wave][0] = x0;
    gb[wave][1] = x1;
    gb[wave][2] = y0;
    gb[wave][3] = y1;
  }
  __syncthreads();
  double wx0 = gb[0][0], wx1 = gb[0][1], wy0 = gb[0][2], wy1 = gb[0][3];
  for (int k = 1; k < kGroups; ++k) {
    wx0 = fmin(wx0, gb[k][0]);
    wx1 = fmax(wx1, gb[k][1]);
    wy0 = fmin(wy0, gb[k][2]);
    wy1 = fmax(wy1, gb[k][3]);
  }
  for (int64_t base = 0; base < ntiles; base += (int64_t)kNearT * gridDim.y) {
    // the next kNearT of this row's tiles
    const int64_t it = base + (int64_t)t * gridDim.y + blockIdx.y;
    bool near = it < ntiles;
    if (near) near = box_near(tbox[it], wx0, wx1, wy0, wy1);
    const unsigned long long m = __ballot(near);
    if (lane == 0) found[wave] = __popcll(m);
    __syncthreads();
    uint32_t at = 0, total = 0;
    for (int w = 0; w < kWaves; ++w) {
      at += w < wave ? found[w] : 0u;
      total += found[w];
    }
    if (near) list[at + __popcll(m & ((1ull << lane) - 1ull))] = (uint32_t)it;
    __syncthreads();
    // 64 boxes of eight listed tiles at a time; the two waves of a group take the even and the odd
    // ones. A box's sources pass through this wave's piece of LDS, the next box's loads under way.
    for (uint32_t l0 = 0; l0 < total; l0 += 64 / kSubs) {
      const uint32_t l = l0 + lane / kSubs;
      uint32_t e = 0;
      bool reach = false;
      if (l < total && (lane & 1) == half) {
        e = list[l] * kSubs + lane % kSubs;
        reach = box_near(sub[e], x0, x1, y0, y1);
      }
      unsigned long long todo = __ballot(reach);
      double2 next = make_double2(0.0, 0.0);
      if (todo) {
        const uint32_t f = __builtin_amdgcn_readlane(e, __builtin_ctzll(todo));
        next = reinterpret_cast<const double2*>(vs + (int64_t)f * kSub)[lane];
      }
      while (todo) {
        todo &= todo - 1;
        wave_sync();
        reinterpret_cast<double2*>(mine)[lane] = next;
        wave_sync();
        if (todo) {
          const uint32_t f = __builtin_amdgcn_readlane(e, __builtin_ctzll(todo));
          next = reinterpret_cast<const double2*>(vs + (int64_t)f * kSub)[lane];
        }
#pragma unroll
        for (int k = 0; k < kSub / kLanes; ++k) {
          const VSrc c = mine[k * kLanes + share];
#pragma unroll
          for (int e = 0; e < kPer; ++e) {
            const double dx = px[e] - c.x, dy = py[e] - c.y;
            const double x = (dx * dx + dy * dy) * c.rr;
            if (!(x >= kUnderflow)) acc[e] += c.c * exp_neg(x, e2t);  // a NaN exponent adds NaN
          }
        }
      }
    }
    __syncthreads();  // before the list changes
  }
  // a target's lanes, then its two waves
#pragma unroll
  for (int e = 0; e < kPer; ++e) {
#pragma unroll
    for (int s = kSpan; s < 64; s <<= 1) acc[e] += __shfl_xor(acc[e], s, 64);
    if (half == 1 && share == 0) sum[group][e * kSpan + lane] = acc[e];
  }
  __syncthreads();
  if (half != 0 || share != 0) return;
#pragma unroll
  for (int e = 0; e < kPer; ++e) {
    const int64_t p = p0 + e * kSpan;
    if (p >= nt) continue;
    const double s = acc[e] + sum[group][e * kSpan + lane];
    if (part)
      part[(int64_t)blockIdx.y * nt + p] = s;
    else
      tw[o[e]] += s;
  }
}

// tw[torder[p]] += the sum over rows of part[row nt + p], in row order
__global__ __launch_bounds__(kBlock) void vort_reduce_kernel(int64_t rows, int64_t nt,
                                                             const double* __restrict__ part,
                                                             const uint32_t* __restrict__ torder,
                                                             double* __restrict__ tw) {
  const int64_t p = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (p >= nt) return;
  double s = 0.0;
#pragma unroll 4
  for (int64_t r = 0; r < rows; ++r) s += part[r * nt + p];
  tw[torder[p]] += s;
}

}  // namespace

int vorticity_dev(Device* d, hipStream_t s, int64_t ns, const double* sx, const double* sy,
                  const double* ss, const double* sr, int64_t nt, const double* tx,
                  const double* ty, double* tw) {
  if (ns == 0 || nt == 0) return 0;
  const int64_t ntiles = (ns + kTile - 1) / kTile;
  const uint32_t *sorder = nullptr, *torder = nullptr;
  O2D_TRY(morton_order16(d, s, ns, sx, sy, &sorder));
  void* vp;
  O2D_TRY(slot(d, kVortSrc, (sizeof(VSrc) * kTile + sizeof(VBox) * (kSubs + 1)) * (size_t)ntiles, s,
               &vp));
  VSrc* vs = static_cast<VSrc*>(vp);
  VBox* sub = reinterpret_cast<VBox*>(vs + kTile * ntiles);
  VBox* tbox = sub + kSubs * ntiles;
  vort_gather_kernel<<<(unsigned)ntiles, kBlock, 0, s>>>(ns, sx, sy, ss, sr, sorder, vs, sub, tbox);
  O2D_LAUNCH_CHECK();
  torder = sorder;  // the sources themselves, or another order in the same slot: vs holds the sources
  if (!(tx == sx && ty == sy && nt == ns)) O2D_TRY(morton_order16(d, s, nt, tx, ty, &torder));
  const int64_t twgs = (nt + kNearTargets - 1) / kNearTargets;
  const int64_t want = kNearWgs * (int64_t)d->num_cu;
  int64_t rows = std::max((want + twgs - 1) / twgs, std::min(kNearRows, ntiles / kRowTiles));
  rows = std::min({rows, ntiles, kPartialBytes / ((int64_t)sizeof(double) * nt)});
  rows = std::max<int64_t>(rows, 1);
  void* part = nullptr;
  if (rows > 1) O2D_TRY(slot(d, kPartials, sizeof(double) * rows * nt, s, &part));
  KernelTimer kt(O2D_KT_VORT, s);
  vort_near_kernel<<<dim3((unsigned)twgs, (unsigned)rows), kNearT, 0, s>>>(
      nt, tx, ty, torder, ntiles, vs, sub, tbox, tw, static_cast<double*>(part));
  kt.stop();
  O2D_LAUNCH_CHECK();
  if (rows > 1) {
    vort_reduce_kernel<<<(unsigned)((nt + kBlock - 1) / kBlock), kBlock, 0, s>>>(
        rows, nt, static_cast<const double*>(part), torder, tw);
    O2D_LAUNCH_CHECK();
  }
  return 0;
}

}  // namespace o2d

using namespace o2d;

extern "C" {

static int check_vort(const o2d_env* env, int64_t ns, const void* sx, const void* sy,
                      const void* ss, const void* sr, int64_t nt, const void* tx,
                      const void* ty, const void* tw) {
  O2D_TRY(check_env(env));  // any precision form: the sum is always fp64
  if (ns < 0 || nt < 0) return fail(O2D_ERR_SIZE, "negative count");
  if (ns > 0x7fffffffLL || nt > 0x7fffffffLL) return fail(O2D_ERR_SIZE, "count too large");
  if (ns > 0 && (!sx || !sy || !ss || !sr)) return fail(O2D_ERR_ARG, "NULL source array");
  if (nt > 0 && (!tx || !ty || !tw)) return fail(O2D_ERR_ARG, "NULL target array");
  return 0;
}

int o2d_hip_points_vorticity_dev_d(const o2d_env* env, int64_t ns, const double* sx,
                                   const double* sy, const double* sstr, const double* srad,
                                   int64_t nt, const double* tx, const double* ty, double* tw) {
  clear_error();
  O2D_TRY(check_vort(env, ns, sx, sy, sstr, srad, nt, tx, ty, tw));
  if (ns == 0 || nt == 0) return 0;
  Device* d;
  O2D_TRY(device(env->device, &d));
  return vorticity_dev(d, dev_stream(env), ns, sx, sy, sstr, srad, nt, tx, ty, tw);
}

int o2d_hip_points_vorticity_d(const o2d_env* env, int64_t ns, const double* sx,
                               const double* sy, const double* sstr, const double* srad,
                               int64_t nt, const double* tx, const double* ty, double* tw) {
  clear_error();
  O2D_TRY(check_vort(env, ns, sx, sy, sstr, srad, nt, tx, ty, tw));
  if (ns == 0 || nt == 0) return 0;
  Device* d;
  O2D_TRY(device(env->device, &d));
  hipStream_t s = stream_of(env, d);
  double *dsx, *dsy, *dss, *dsr, *dtx, *dty, *dtw;
  O2D_TRY(upload<double>(d, kSrcX, sx, ns, s, &dsx));
  O2D_TRY(upload<double>(d, kSrcY, sy, ns, s, &dsy));
  O2D_TRY(upload<double>(d, kSrcS, sstr, ns, s, &dss));
  O2D_TRY(upload<double>(d, kSrcR, srad, ns, s, &dsr));
  O2D_TRY(upload<double>(d, kTrgX, tx, nt, s, &dtx));
  O2D_TRY(upload<double>(d, kTrgY, ty, nt, s, &dty));
  O2D_TRY(upload<double>(d, kOutW, tw, nt, s, &dtw));
  O2D_TRY(vorticity_dev(d, s, ns, dsx, dsy, dss, dsr, nt, dtx, dty, dtw));
  O2D_TRY(download<double>(tw, dtw, nt, s));
  O2D_HIP(hipStreamSynchronize(s));
  return 0;
}

}  // extern "C"

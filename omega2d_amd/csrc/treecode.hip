// treecode.hip - O(N log N) particle sums: the summation the reference reserves as summation_t
// barneshut (src/ExecEnv.h:26-31) behind the same operator as the direct sum, and, at an
// acceptance where the remainder is below rounding, the fp64 Gaussian velocity sum and its
// adjoint beyond the compact cutoff, where K = 1/d^2 exactly (src/CoreFunc.h:120-122).
//
// With q_j the charge of source j (its strength; gv - i gu for the adjoint, whose sources are the
// probes), far sources act on a target z through S = sum_j q_j / (z - z_j), and for the adjoint
// also S2 = sum_j q_j / (z - z_j)^2 = -dS/dz. The unscaled velocity is u - i v = -i S.
//
// Tree: sources in Morton order, cut into leaves of kLeaf consecutive sources; each coarser
// level groups kFan consecutive cells, so every cell is one contiguous Morton range. Per cell: box
// centre c, radius r (covers every source), largest radius term, and the moments
// M_k = sum_j q_j ((z_j - c) / r)^k, k < p, in fp64 (scaled by the radius, so that no power
// overflows or vanishes). Parents shift their children's. A cell with a charge or radius that
// is not finite gets r = inf, is never used through its moments, and reaches the sum pair by pair.
//
// Evaluation, from the largest clusters of targets to the smallest:
//   super groups   one workgroup per kSuper Morton-ordered targets opens the tree from the root,
//                  every cell of a round tested by its own thread. Cells that are far for all the
//                  targets become one local expansion about the targets' centre, L_l =
//                  sum_j q_j / ..., (z - c_T)^l; cells no larger than half the super group that
//                  are not far form its frontier;
//   groups         one wave per 64 targets (one per lane) starts at the frontier. 64 cells are
//                  tested at a time, one per lane, against the box of the wave's targets: far
//                  cells are evaluated through their moments by every lane, leaves that are not
//                  far pair by pair in fp64 with the exact core, the rest is opened.
// A cell of radius r is far from targets at distance D or more from its centre when r <= theta D
// and the core equals 1/d^2 for every pair within core_tol, from d_min = D - r: exactly beyond the
// Gaussian's compact cutoff (d^2 > 16 w); for the other cores through the bound on |K d^2 - 1|
// (RM w/d^2, WL w^2/d^4, V2 w/(2 d^4), V3 w/(3 d^6)). A local expansion of radius R at distance d
// from the cell's centre also needs R <= theta (d - r).
//
// What bounds it: issue of the near pairs and of the moment sums. One wave that popped one cell
// at a time from its own stack spent most of its time waiting for that cell's record and moments;
// testing 64 cells at once takes a handful of dependent loads per wave, a far cell's moments and a
// leaf's sources come through LDS, and the far cells of 1,024 targets are summed once, not sixteen
// times. The group kernel is held to 128 registers, four waves per SIMD (the Gaussian's then spills 12
// to 14 of them, the adjoint's 40 to 43). 1M blob particles on themselves plus 65,536 tracers (theta
// 0.6, order 28): 7.6 -> 3.2 ms, of which the particles' groups 2.1, the tracers' 0.58, the super groups
// 0.2, the trees and orders 0.5.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "nbody.h"
#include "o2d_math.h"
#include "o2d_runtime.h"

namespace o2d {

namespace {

constexpr int kLeaf = 32;       // sources per leaf
constexpr int kFan = 4;         // children per cell
constexpr int kMaxP = 32;       // largest expansion order; cells store this many moments
constexpr int kMaxLevels = 16;  // 2^31 sources make 14 levels
constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kGroupWaves = 1, kGroupBlock = 64 * kGroupWaves;  // a wave ends by itself
constexpr int kSuper = 1024;    // targets per super group
constexpr int kSuperBlock = 512;
constexpr int kSuperWaves = kSuperBlock / 64;
constexpr int kQueue = 1024;    // cells of one round of a super group
constexpr int kFront = 512;     // frontier cells of a super group
constexpr int kStack = 512;     // cells a group's wave has still to test
constexpr int kStackSpare = 3 * kMaxLevels;  // what opening one cell at a time can add
// acceptance at which the remainder of kMaxP moments is below rounding: a far cell's is at most
// 3^-kMaxP = 5e-16 of sum |q_j| / D. (0.3 took 2.0 ms instead of 1.73 for 262,147 blob particles
// on themselves and 9,973 tracers, 0.36, whose remainder is 6e-15, 1.59 ms; the error against 64
// bits did not move, 5e-16, a quarter of the pair by pair sum's.)
constexpr double kExactTheta = 1.0 / 3.0;
// The remainder of a cell at distance d is (r / d)^p of its contribution, at most theta^p. A sum takes
// many cells near the limit, and truncates some in more than one way, so each way keeps to a share of
// theta^p: the moments of cells at the limit of groups of 64 targets and of 16 (smaller, so that more of
// their targets are near it), the orders left out of cells further away, and local expansions. From
// kShareOrder on a share is kept by taking cells from a little further than theta says; below, where
// that little is much, cells near the limit use up to kSpareOrders more than p. The exact sums, whose
// remainders are below rounding, take the wider shares (their error is 4.6e-16 with either).
constexpr double kShare64 = 0.275, kShare16 = 0.08, kShareTail = 0.02, kShareLocal = 0.0105;
constexpr double kExactShare16 = 0.275, kExactShareTail = 0.05;
constexpr int kShareOrder = 28, kSpareOrders = 6;
inline int kept_orders(int p) {
  return p + std::max(0, std::min(kSpareOrders, kShareOrder - p));
}
// Groups of 16 targets where targets are much sparser than the sources, else of 64: a box of 64 would
// hold many leaves that few of its targets are near. 1M sources, targets a 64th, 16th, 12th, 8th and 5th
// as many: 564, 722, 822, 876 and 1,009 us in groups of 16, 714, 766, 804, 872 and 999 of 64; at theta
// 1/3 804, 1,191, 1,410, 1,578 and 1,964 against 1,003, 1,142, 1,233, 1,417 and 1,727. In the adjoint,
// whose targets are the particles: 50,000 among 200,000 probes 887 and 756, 10,000 among 100,000 486 and
// 457, 781 among 50,000 219 and 244, 1,000 among 1M 788 and 1,094.
constexpr int64_t kSparse = 12, kSparseAdjoint = 64;
// waves per CU the group kernel aims for by sharing a group's cells and leaves out: every share
// opens the same cells, so more of them cost more (1M particles: 32 and 64 equal), unless they no
// longer fit the chip at once (16 per CU do): 20,000 particles take 163 us at 16 or just below and 175
// at 32, 100,000 and 8,000 targets in groups of 16 214 at or just below 16 and 222 just above. From
// kEvenGroups groups on a second round of waves costs less than groups of unequal work (30,000 targets of
// which many are within the cores 394 and 418 us, 40,000 635 and 660, 262,144 1,437 and 1,698). (Opening
// the same cells in every share is also why small theta gains nothing over the earlier form, whose shares
// began at different cells, where targets are few: 200,000 sources on 12,500 at theta 0.3 404 us against
// 412, 0.2 555 and 474, 0.1 1,090 and 560.)
constexpr int kWaves64 = 32, kWavesOnce = 16;
constexpr int64_t kEvenGroups = 400;
// Fewer super groups than this leave most of the chip idle for longer than they save: us with and without,
// 40,000 blob particles on themselves (40 of them) 237 and 225, 90,000 339 and 325, 110,000 382 and 373,
// 130,000 412 and 417, 262,144 717 and 743, 524,288 1,220 and 1,325; the adjoint of 30,000 particles 301 and
// 281, 64,000 317 and 313, 80,000 348 and 352, 200,000 422 and 475
constexpr int64_t kMinSupers = 120, kMinSupersAdjoint = 72;

// When the fp64 Gaussian sums go by clusters. In units of a pair of the pair by pair form, whose work is
// sources times targets filled up to its tiles: what building and walking the tree costs besides, which
// grows more slowly than the sources, and (up to a most) with targets that share few cells.
// Velocity, us by clusters and pair by pair (blobs): 10,000 on themselves 137 and 101, 16,000 184 and 206,
// 20,000 182 and 259; 50,000 on 6,000 points 243 and 225; 100,000 on 3,000 and 4,000 266 and 274 against 227
// and 273; 262,144 on 2,000 and 3,000 382 and 383 against 345 and 492; 1M on 300, 700 and 1,000 618, 627
// and 655 against 419, 653 and 656; 2M on 100 883 and 756; 4M on 100 1,155 and 1,362; 10,000 on 30,000
// 203 and 230; 1,000 on 200,000 and 350,000 193 and 262 against 183 and 282.
constexpr double kClusterPairs = 1.2e8, kClusterSources = 9e5, kClusterTarget = 300, kClusterTargets = 2e8;
// The adjoint: 10,000 on themselves 182 and 203, 16,000 247 and 315; 60,000 particles and 4,000 probes 241
// and 256; 100,000 and 2,200 and 3,000 254 and 279 against 231 and 316; 250,000 and 1,000 and 1,500 313 and
// 352 against 259 and 375; 1M and 500 574 and 499; 4M and 100 and 700 1,258 and 2,633 against 902 and 2,915;
// 10,000 and 25,000 265 and 257; 3,000 and 50,000 and 150,000 297 and 426 against 172 and 443; 2,000 and
// 300,000 493 and 601; 1,000 and 500,000 and 1M 578 and 797 against 537 and 1,022; 100 and 4M 1,836 and
// 1,951, but 2,677 with a pair in the cutoff sampled; 40 and 10M 3,324 and 4,528.
constexpr double kAdjointPairs = 2e8, kAdjointParticle = 500, kAdjointProbe = 400, kAdjointFew = 1000,
                 kAdjointFewMost = 2.5e8;

// Clusters gain nothing on pairs nearer than the cutoff, and where few targets share the chip their walk is
// far slower there than the pair by pair loops. A sample of kSampleS sources and kSampleT targets says
// which part of the pairs that is; past a limit the call sums pair by pair (8 us more than pairs alone,
// and the tree for nothing). The limit, the targets from which it is whole (with fewer: times the
// square of their part) and those from which nothing is sampled, because clusters are about as fast as
// pairs at any radius. us by clusters and pair by pair; velocity: 262,144 on 10,000 with 8% of the pairs
// near 2,274 and 3,949, 28% 4,990 and 4,961, 74% 9,834 and 6,487; 20,000 on themselves 19% 471 and 471, 99%
// 1,064 and 777; 100,000 on 4,000 0.5% 330 and 406, 8% 728 and 571; 1M on 1,000 0.5% 1,418 and 1,184, 75%
// 17,020 and 2,729; 10,000 on 100,000 78% 2,003 and 2,482. Adjoint: 10,000 particles and 100,000 probes 0.5%
// 557 and 1,018, 8% 1,282 and 1,373, 77% 4,786 and 3,025; 1,000 and 1M 0 792 and 1,022, 0.5% 1,381 and
// 1,186, 77% 28,915 and 3,433; 30,000 and 12,000 100% 1,619 and 1,199; 100,000 and 8,000 75% 2,545 and 2,284.
constexpr int kSampleS = 256, kSampleT = 64;
constexpr double kNearLimit = 0.3, kNearTargets = 1e4, kNearMany = 5e4;
constexpr double kNearLimitAdjoint = 0.4, kNearTargetsAdjoint = 2e4, kNearManyAdjoint = 7e4;

// A cell: head = (centre x, y, radius, largest radius term), kids = (first child, children); a
// leaf has no children, and its first child is its index among the leaves. (As one struct the
// records went through scratch memory wherever they were read ahead.)

struct Levels {
  int n;                      // number of levels (level 0 = leaves, n - 1 = root)
  int64_t off[kMaxLevels];    // first cell of each level in the cell array
  int64_t cnt[kMaxLevels];    // cells per level
};

// a source as the pair loops read it: position, then strength and radius term (velocity) or the
// two upstream gradients (adjoint)
struct alignas(16) Src {
  double x, y, a, b;
};

// a target: position, strength, then its radius term (velocity) or radius (adjoint). A collection
// acting on itself reads its sources' records as its targets'.
struct alignas(16) Trg {
  double x, y, s, w;
};
static_assert(sizeof(Src) == sizeof(Trg), "one array serves both");

// C(n + m, m) for n, m < kMaxP, rounded once from the exact integers
struct Binomials {
  double v[kMaxP * kMaxP];
};
constexpr Binomials make_binomials() {
  Binomials b{};
  unsigned long long row[kMaxP] = {};
  for (int m = 0; m < kMaxP; ++m) row[m] = 1;
  for (int n = 0; n < kMaxP; ++n) {
    for (int m = 0; m < kMaxP; ++m) {
      if (n > 0 && m > 0) row[m] += row[m - 1];  // C(n+m, m) = C(n-1+m, m) + C(n+m-1, m-1)
      b.v[n * kMaxP + m] = (double)row[m];
    }
  }
  return b;
}
__constant__ Binomials kBinomials = make_binomials();

__device__ __forceinline__ double rterm_any(int core, double r) {
  return core == O2D_CORE_V2   ? rterm<O2D_CORE_V2>(r)
         : core == O2D_CORE_V3 ? rterm<O2D_CORE_V3>(r)
                               : rterm<O2D_CORE_RM>(r);
}

// LDS writes of this wave visible to its own later reads, and no compiler reordering across
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// lane l's x, in every lane
__device__ __forceinline__ double lane_f64(double x, int l) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)b, l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// reductions over lanes that differ in the bits below `width`
template <int width>
__device__ __forceinline__ double lanes_min(double v) {
#pragma unroll
  for (int m = width / 2; m >= 1; m >>= 1) v = fmin(v, __shfl_xor(v, m));
  return v;
}
template <int width>
__device__ __forceinline__ double lanes_max(double v) {
#pragma unroll
  for (int m = width / 2; m >= 1; m >>= 1) v = fmax(v, __shfl_xor(v, m));
  return v;
}

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(__builtin_fma(a.x, b.x, -a.y * b.y), __builtin_fma(a.x, b.y, a.y * b.x));
}
// f = f z + m
__device__ __forceinline__ void horner(double2& f, double2 z, double2 m) {
  const double fx = __builtin_fma(f.x, z.x, __builtin_fma(-f.y, z.y, m.x));
  f.y = __builtin_fma(f.x, z.y, __builtin_fma(f.y, z.x, m.y));
  f.x = fx;
}
// z^k, k < kMaxP
__device__ __forceinline__ double2 cpow(double2 z, int k) {
  double2 r = make_double2(1.0, 0.0);
#pragma unroll
  for (int b = 1; b < kMaxP; b <<= 1) {
    const double2 t = cmul(r, z);
    const bool set = (k & b) != 0;  // component by component: as structs they go through memory
    r.x = set ? t.x : r.x;
    r.y = set ? t.y : r.y;
    if (2 * b < kMaxP) z = cmul(z, z);
  }
  return r;
}
// 1 / (x + i y)
__device__ __forceinline__ double2 cinv(double x, double y) {
  const double q = rcp64(__builtin_fma(x, x, y * y));
  return make_double2(x * q, -y * q);
}

// ---------------------------------------------------------------------------- the tree

// What a call samples: its targets (tr null: no radii), and the part of the pairs within the Gaussian's
// cutoff from which *gate is set
struct Sample {
  int64_t nt;
  const double *tx, *ty, *tr;
  double limit;
  int* gate;
};

// *gate = more than the limit of kSampleS x kSampleT pairs, spread evenly over the arrays, are within the
// cutoff (one workgroup; sr: the sources' radii, in the adjoint only the targets' count; lds: three
// arrays of kSampleT and a count per wave). Pairs with a NaN are not.
template <bool ADJ>
__device__ void sample_near(int64_t ns, const double* x, const double* y, const double* sr,
                            const Sample& m, double* lds) {
  double *tx = lds, *ty = lds + kSampleT, *tw = lds + 2 * kSampleT;
  int* near = reinterpret_cast<int*>(lds + 3 * kSampleT);
  const int t = threadIdx.x;
  static_assert(kSampleS == kBlock, "a source per thread");
  if (t < kSampleT) {
    const int64_t i = m.nt * t / kSampleT;
    tx[t] = m.tx[i];
    ty[t] = m.ty[i];
    tw[t] = m.tr ? m.tr[i] * m.tr[i] : 0.0;
  }
  const int64_t j = ns * t / kSampleS;
  const double px = x[j], py = y[j], w = ADJ ? 0.0 : sr[j] * sr[j];
  __syncthreads();
  int n = 0;
  for (int i = 0; i < kSampleT; ++i) {
    const double dx = px - tx[i], dy = py - ty[i];
    n += dx * dx + dy * dy < kGaussFar * (w + tw[i]) ? 1 : 0;
  }
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
  if ((t & 63) == 0) near[t >> 6] = n;
  __syncthreads();
  if (t != 0) return;
  for (int w = 1; w < kWaves; ++w) n += near[w];
  *m.gate = (double)n > m.limit * (kSampleS * kSampleT) ? 1 : 0;
}

// One wave per 64 sources in Morton order (kLeafs leaves): gathers their records (padding a
// short last leaf with charges of 0 at its last source) and forms each leaf's cell, box and
// moments. The powers of eight orders at a time pass through LDS, and each (leaf, order) sum is
// taken by a few lanes: a wave sum per order through shuffles took 130 us for 1M sources.
// ADJ: a is gv's and b gu's array, and radii play no part. The last workgroup samples instead, where
// there is a gate to set.
template <bool ADJ>
__global__ __launch_bounds__(kBlock) void tree_leaf_kernel(
    int64_t ns, int64_t nleaf, int p, const uint32_t* __restrict__ order,
    const double* __restrict__ x, const double* __restrict__ y, const double* __restrict__ a,
    const double* __restrict__ b, int core, Src* __restrict__ src, double4* __restrict__ head,
    uint2* __restrict__ kids, double4* __restrict__ box, double2* __restrict__ mom, Sample sample) {
  constexpr int kLeafs = 64 / kLeaf, kChunk = 8;
  constexpr int kShare = 64 / (kLeafs * kChunk);  // lanes per (leaf, order)
  static_assert(kShare >= 1 && kLeaf % kShare == 0, "whole shares");
  __shared__ double2 buf[kWaves][kChunk][64 + 1];
  if (sample.gate && blockIdx.x == gridDim.x - 1) {
    sample_near<ADJ>(ns, x, y, b, sample, reinterpret_cast<double*>(buf));
    return;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t first = ((int64_t)blockIdx.x * kWaves + wave) * 64;
  if (first >= nleaf * kLeaf) return;  // whole waves; no workgroup barrier below
  const int64_t i = first + lane;
  const bool in = i < ns;
  const uint32_t o = order[in ? i : ns - 1];
  Src q;
  q.x = x[o];
  q.y = y[o];
  q.a = in ? a[o] : 0.0;
  if constexpr (ADJ) q.b = in ? b[o] : 0.0;
  else q.b = in ? rterm_any(core, b[o]) : 1.0;
  if (i < nleaf * kLeaf) src[i] = q;
  const double x0 = lanes_min<kLeaf>(in ? q.x : INFINITY), x1 = lanes_max<kLeaf>(in ? q.x : -INFINITY);
  const double y0 = lanes_min<kLeaf>(in ? q.y : INFINITY), y1 = lanes_max<kLeaf>(in ? q.y : -INFINITY);
  const double wm = ADJ ? 0.0 : lanes_max<kLeaf>(in ? q.b : 0.0);
  const double cx = 0.5 * (x0 + x1), cy = 0.5 * (y0 + y1);
  const double dx = q.x - cx, dy = q.y - cy;
  // a charge that is not finite (its product with 0 is not 0) makes r infinite; an infinite radius
  // term keeps the cell from being far by itself, and a NaN one reaches the pairs near it, as in
  // the pair by pair sum, whose tiles beyond the largest finite term do not look at it
  const bool odd = in && !(q.a * 0.0 + (ADJ ? q.b * 0.0 : 0.0) == 0.0);
  const double r2 = lanes_max<kLeaf>(odd ? INFINITY : (in ? dx * dx + dy * dy : 0.0));
  // rounding of the offsets: a relative margin keeps r an upper bound
  const double r = sqrt(r2) * (1.0 + 1e-12);
  const double inv = r > 0.0 ? 1.0 / r : 0.0;
  const double2 d = make_double2(dx * inv, dy * inv);
  double2 pw = ADJ ? make_double2(q.a, -q.b) : make_double2(q.a, 0.0);
  if (!in) pw = make_double2(0.0, 0.0);
  const int64_t leaf = first / kLeaf + lane / kLeaf;
  if ((lane & (kLeaf - 1)) == 0 && leaf < nleaf) {
    head[leaf] = make_double4(cx, cy, r, wm);
    kids[leaf] = make_uint2((uint32_t)leaf, 0);
    box[leaf] = make_double4(x0, y0, x1, y1);
  }
  // lane = ((share * kLeafs) + lf) * kChunk + k
  const int k = lane % kChunk, lf = (lane / kChunk) % kLeafs, share = lane / (kChunk * kLeafs);
  for (int k0 = 0; k0 < kMaxP; k0 += kChunk) {
#pragma unroll
    for (int e = 0; e < kChunk; ++e) {
      buf[wave][e][lane] = pw;
      pw = cmul(pw, d);
    }
    wave_sync();
    double2 m = make_double2(0.0, 0.0);
#pragma unroll
    for (int j = 0; j < kLeaf / kShare; ++j) {
      const double2 t = buf[wave][k][lf * kLeaf + share * (kLeaf / kShare) + j];
      m.x += t.x;
      m.y += t.y;
    }
#pragma unroll
    for (int s = kChunk * kLeafs; s < 64; s <<= 1) {
      m.x += __shfl_xor(m.x, s);
      m.y += __shfl_xor(m.y, s);
    }
    const int64_t c = first / kLeaf + lf;
    if (share == 0 && c < nleaf)
      mom[c * kMaxP + k0 + k] = k0 + k < p ? m : make_double2(0.0, 0.0);
    wave_sync();
  }
}

// One cell from its children (global cells child0 .. child0 + nch - 1), by one wave: the union of
// the boxes, a covering radius (of the children's circles or of the box, whichever is smaller),
// and the moments, M'_k = sum_children sum_{l <= k} C(k, l) (r_c / r)^l M_l ((c_c - c) / r)^(k - l).
// Half-waves take a child each, lane k its order k; sa, sd: the wave's 2 x kMaxP scratch entries.
__device__ __forceinline__ void tree_parent(uint32_t self, uint32_t child0, int nch, int p,
                                            const double* __restrict__ binom, double2* sa,
                                            double2* sd, double4* head, uint2* kids,
                                            double4* box, double2* mom) {
  const int lane = threadIdx.x & 63, k = lane & (kMaxP - 1), h = lane / kMaxP;
  double4 b = box[child0];
  double wm = head[child0].w;
  for (int c = 1; c < nch; ++c) {
    const double4 e = box[child0 + c];
    b.x = fmin(b.x, e.x);
    b.y = fmin(b.y, e.y);
    b.z = fmax(b.z, e.z);
    b.w = fmax(b.w, e.w);
    wm = fmax(wm, head[child0 + c].w);
  }
  const double cx = 0.5 * (b.x + b.z), cy = 0.5 * (b.y + b.w);
  double r = 0.0;
  bool odd = false;
  for (int c = 0; c < nch; ++c) {
    const double4 q = head[child0 + c];
    const double dx = q.x - cx, dy = q.y - cy;
    r = fmax(r, sqrt(dx * dx + dy * dy) + q.z);
    odd = odd || !(q.z < INFINITY);
  }
  const double ex = b.z - cx, ey = b.w - cy;
  r = odd ? INFINITY : fmin(r, sqrt(ex * ex + ey * ey)) * (1.0 + 1e-12);
  const double inv = r > 0.0 ? 1.0 / r : 0.0;
  double2 acc = make_double2(0.0, 0.0);
  for (int c0 = 0; c0 < kFan; c0 += 2) {
    const int c = c0 + h;
    double2 a = make_double2(0.0, 0.0), d = a;
    if (c < nch) {
      const double4 q = head[child0 + c];
      const double2 m = mom[(int64_t)(child0 + c) * kMaxP + k];
      const double ratio = cpow(make_double2(q.z * inv, 0.0), k).x;
      a = make_double2(m.x * ratio, m.y * ratio);
      d = cpow(make_double2((q.x - cx) * inv, (q.y - cy) * inv), k);
    }
    wave_sync();
    sa[lane] = a;
    sd[lane] = d;
    wave_sync();
#pragma unroll 4
    for (int l = 0; l < kMaxP; ++l) {
      if (l <= k) {
        const double2 al = sa[h * kMaxP + l], dl = sd[h * kMaxP + k - l];
        const double bn = binom[l * kMaxP + k - l];
        const double2 t = make_double2(al.x * bn, al.y * bn);
        acc.x = __builtin_fma(t.x, dl.x, __builtin_fma(-t.y, dl.y, acc.x));
        acc.y = __builtin_fma(t.x, dl.y, __builtin_fma(t.y, dl.x, acc.y));
      }
    }
  }
  acc.x += __shfl_xor(acc.x, kMaxP);
  acc.y += __shfl_xor(acc.y, kMaxP);
  if (h == 0) mom[(int64_t)self * kMaxP + k] = k < p ? acc : make_double2(0.0, 0.0);
  if (lane == 0) {
    head[self] = make_double4(cx, cy, r, wm);
    kids[self] = make_uint2(child0, (uint32_t)nch);
    box[self] = b;
  }
}

// Two coarser levels per launch: a workgroup's four waves form four cells of level l + 1, then
// its first wave their parent of level l + 2 (when there is one: cnt2 > 0)
__global__ __launch_bounds__(kBlock) void tree_up_kernel(uint32_t off0, uint32_t cnt0, uint32_t off1,
                                                         uint32_t cnt1, uint32_t off2,
                                                         uint32_t cnt2, int p, double4* head,
                                                         uint2* kids, double4* box,
                                                         double2* mom) {
  __shared__ double binom[kMaxP * kMaxP];
  __shared__ double2 sa[kWaves][64], sd[kWaves][64];
  static_assert(kWaves == kFan, "a workgroup forms the children of one cell");
  const int wave = threadIdx.x >> 6;
  for (int e = threadIdx.x; e < kMaxP * kMaxP; e += kBlock) binom[e] = kBinomials.v[e];
  __syncthreads();
  const uint32_t c1 = blockIdx.x * kFan + wave;
  if (c1 < cnt1) {
    const uint32_t k0 = c1 * kFan;
    const int nch = (int)(k0 + kFan < cnt0 ? kFan : cnt0 - k0);
    tree_parent(off1 + c1, off0 + k0, nch, p, binom, sa[wave], sd[wave], head, kids, box,
                mom);
  }
  if (cnt2 == 0) return;  // uniform
  __threadfence_block();
  __syncthreads();
  if (wave != 0) return;
  const uint32_t k0 = blockIdx.x * kFan;
  const int nch = (int)(k0 + kFan < cnt1 ? kFan : cnt1 - k0);
  tree_parent(off2 + blockIdx.x, off1 + k0, nch, p, binom, sa[0], sd[0], head, kids, box, mom);
}

// the targets in Morton order
template <bool ADJ>
__global__ __launch_bounds__(kBlock) void tree_targets_kernel(int64_t n, const uint32_t* __restrict__ order,
                                                              const double* __restrict__ x,
                                                              const double* __restrict__ y,
                                                              const double* __restrict__ r,
                                                              const double* __restrict__ s,
                                                              int core, Trg* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const uint32_t o = order[i];
  Trg t;
  t.x = x[o];
  t.y = y[o];
  if constexpr (ADJ) {
    t.w = r[o];
    t.s = s[o];
  } else {
    t.w = r ? rterm_any(core, r[o]) : 0.0;
    t.s = 0.0;
  }
  out[i] = t;
}

// ---------------------------------------------------------------------------- far tests

// the pair distance from which the core equals 1/d^2 to within tol (exactly for the Gaussian) for
// radius terms up to w, with a margin far above the rounding of the tests that use it
template <int CORE>
__device__ __forceinline__ double core_reach(double w, double tol) {
  if constexpr (CORE == O2D_CORE_GAUSSIAN) {
    return 4.0 * sqrt(w) * (1.0 + 1e-12);
  } else if constexpr (CORE == O2D_CORE_RM) {
    return sqrt(w / tol) * (1.0 + 1e-12);
  } else if constexpr (CORE == O2D_CORE_WL) {
    return sqrt(w / sqrt(tol)) * (1.0 + 1e-12);
  } else if constexpr (CORE == O2D_CORE_V2) {
    return sqrt(sqrt(w / (2.0 * tol))) * (1.0 + 1e-12);
  } else {
    return cbrt(sqrt(w / (3.0 * tol))) * (1.0 + 1e-12);
  }
}

// a radius as the largest radius term of the pairs' targets: the adjoint's targets carry radii
template <int CORE, bool ADJ>
__device__ __forceinline__ double target_term(const Trg& t) {
  return ADJ ? rterm<CORE>(t.w) : t.w;
}

// ---------------------------------------------------------------------------- super groups

struct Super {
  double cx, cy, r;  // the local expansion's centre and the radius that scales it
  int64_t nfront;    // frontier cells, or -1: the groups start from the root, without the expansion
};

// One workgroup per kSuper targets. Cells of a round are tested by one thread each; accepted
// ones are dealt to the waves, whose local expansions are added in wave order at the end, so
// nothing depends on scheduling. A wave takes a cell's moments into lanes 0..kMaxP-1, a_k =
// M_k (r / D)^k with D = c_T - c, and its lanes form sum_k C(k + l, l) a_k, half of the k each;
// the upper half-wave scales by (-R / D)^l / D and keeps the sums.
template <int CORE, bool ADJ>
__global__ __launch_bounds__(kSuperBlock) void tree_super_kernel(
    int64_t nt, const Trg* __restrict__ trg, const double4* __restrict__ head,
    const uint2* __restrict__ kids, const double2* __restrict__ mom, uint32_t root, double theta, double tol,
    Super* __restrict__ super, double2* __restrict__ local, uint32_t* __restrict__ front,
    const int* __restrict__ gate) {
  if (gate && *gate != 0) return;
  __shared__ double binom[kMaxP * kMaxP];
  __shared__ uint32_t queue[2][kQueue], taken[kSuperBlock];
  __shared__ int counts[kSuperWaves][3];
  __shared__ double2 am[kSuperWaves][kMaxP];
  __shared__ double2 sums[kSuperWaves][kMaxP];
  __shared__ double red[kSuperWaves][5];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int k = lane & (kMaxP - 1), h = lane / kMaxP;
  for (int e = t; e < kMaxP * kMaxP; e += kSuperBlock) binom[e] = kBinomials.v[e];
  // the targets' box, its centre and the radius that covers them (NaN positions are left out:
  // those targets' sums are NaN whatever is done with the cells)
  const int64_t t0 = (int64_t)blockIdx.x * kSuper;
  double x0 = INFINITY, x1 = -INFINITY, y0 = INFINITY, y1 = -INFINITY, wt = 0.0;
  double px[kSuper / kSuperBlock], py[kSuper / kSuperBlock];
  bool odd = false;
#pragma unroll
  for (int e = 0; e < kSuper / kSuperBlock; ++e) {
    const int64_t i = t0 + e * kSuperBlock + t;
    const Trg q = trg[i < nt ? i : nt - 1];
    const double w = target_term<CORE, ADJ>(q);
    px[e] = q.x;
    py[e] = q.y;
    x0 = fmin(x0, q.x);
    x1 = fmax(x1, q.x);
    y0 = fmin(y0, q.y);
    y1 = fmax(y1, q.y);
    wt = fmax(wt, w);
    odd = odd || !(w < INFINITY);
  }
  if (odd) wt = INFINITY;  // nothing is far from a target whose radius is not finite
  x0 = lanes_min<64>(x0);
  x1 = lanes_max<64>(x1);
  y0 = lanes_min<64>(y0);
  y1 = lanes_max<64>(y1);
  wt = lanes_max<64>(wt);
  if (lane == 0) {
    red[wave][0] = x0;
    red[wave][1] = x1;
    red[wave][2] = y0;
    red[wave][3] = y1;
    red[wave][4] = wt;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kSuperWaves; ++w) {
    x0 = fmin(x0, red[w][0]);
    x1 = fmax(x1, red[w][1]);
    y0 = fmin(y0, red[w][2]);
    y1 = fmax(y1, red[w][3]);
    wt = fmax(wt, red[w][4]);
  }
  const double cx = 0.5 * (x0 + x1), cy = 0.5 * (y0 + y1);
  double r2 = 0.0;
#pragma unroll
  for (int e = 0; e < kSuper / kSuperBlock; ++e) {
    const double dx = px[e] - cx, dy = py[e] - cy;
    r2 = fmax(r2, dx * dx + dy * dy);
  }
  r2 = lanes_max<64>(r2);
  __syncthreads();
  if (lane == 0) red[wave][0] = r2;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kSuperWaves; ++w) r2 = fmax(r2, red[w][0]);
  const double R = sqrt(r2) * (1.0 + 1e-12);

  uint32_t* fr = front + (int64_t)blockIdx.x * kFront;
  int nf = 0, nq = 1, cur = 0;
  bool over = !(R < INFINITY);  // a target at infinity must not reach the others
  if (t == 0) queue[0][0] = root;
  double2 acc = make_double2(0.0, 0.0);  // lane kMaxP + l: L_l
  __syncthreads();
  while (nq > 0 && !over) {
    int nnext = 0;
    for (int base = 0; base < nq && !over; base += kSuperBlock) {
      const bool live = base + t < nq;
      const uint32_t ci = live ? queue[cur][base + t] : root;
      const double4 c = head[ci];
      const uint2 kd = kids[ci];
      const double dx = cx - c.x, dy = cy - c.y;
      const double d = sqrt(dx * dx + dy * dy);
      const double near = d - R;  // the nearest a target can be to the cell's centre
      const bool far = live && near > c.z + core_reach<CORE>(c.w + wt, tol) &&
                       c.z <= theta * near && R <= theta * (d - c.z);
      const bool keep = live && !far && (kd.y == 0 || c.z <= 0.5 * R);
      const int nc = live && !far && !keep ? (int)kd.y : 0;
      // places in the three lists: ballots within the wave, the waves' counts before it
      const unsigned long long below = (1ull << lane) - 1ull;
      const unsigned long long mf = __ballot(far), mk = __ballot(keep);
      const unsigned long long b0 = __ballot(nc & 1), b1 = __ballot(nc & 2), b2 = __ballot(nc & 4);
      int pf = __popcll(mf & below), pk = __popcll(mk & below);
      int pc = __popcll(b0 & below) + 2 * __popcll(b1 & below) + 4 * __popcll(b2 & below);
      if (lane == 0) {
        counts[wave][0] = __popcll(mf);
        counts[wave][1] = __popcll(mk);
        counts[wave][2] = __popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2);
      }
      __syncthreads();
      int nfar = 0, nkeep = 0, nchild = 0;
#pragma unroll
      for (int w = 0; w < kSuperWaves; ++w) {
        pf += w < wave ? counts[w][0] : 0;
        pk += w < wave ? counts[w][1] : 0;
        pc += w < wave ? counts[w][2] : 0;
        nfar += counts[w][0];
        nkeep += counts[w][1];
        nchild += counts[w][2];
      }
      if (nf + nkeep > kFront || nnext + nchild > kQueue) {
        over = true;  // uniform
      } else {
        if (far) taken[pf] = ci;
        if (keep) fr[nf + pk] = ci;
        for (int e = 0; e < nc; ++e) queue[cur ^ 1][nnext + pc + e] = kd.x + e;
      }
      nf += nkeep;
      nnext += nchild;
      __syncthreads();
      if (over) break;
      // the accepted cells, dealt to the waves; the next one's record and moments are on their
      // way while one is shifted
      int j = wave;
      double4 nxt = make_double4(0.0, 0.0, 0.0, 0.0);
      double2 nm = make_double2(0.0, 0.0);
      if (j < nfar) {
        const uint32_t cj = taken[j];
        nxt = head[cj];
        nm = mom[(int64_t)cj * kMaxP + k];
      }
      while (j < nfar) {
        const double4 q = nxt;
        const double2 m = nm;
        j += kSuperWaves;
        if (j < nfar) {
          const uint32_t cj = taken[j];
          nxt = head[cj];
          nm = mom[(int64_t)cj * kMaxP + k];
        }
        const double2 id = cinv(cx - q.x, cy - q.y);  // 1 / D
        const double sc = h == 0 ? q.z : -R;
        const double2 pw = cpow(make_double2(sc * id.x, sc * id.y), k);
        const double2 a = cmul(m, pw);
        wave_sync();
        if (h == 0) am[wave][k] = a;
        wave_sync();
        double2 s = make_double2(0.0, 0.0);
#pragma unroll 8
        for (int e = 0; e < kMaxP / 2; ++e) {
          const int kk = h * (kMaxP / 2) + e;
          const double bn = binom[kk * kMaxP + k];
          const double2 ak = am[wave][kk];
          s.x = __builtin_fma(bn, ak.x, s.x);
          s.y = __builtin_fma(bn, ak.y, s.y);
        }
        s.x += __shfl_xor(s.x, kMaxP);
        s.y += __shfl_xor(s.y, kMaxP);
        const double2 f = cmul(cmul(pw, id), s);
        acc.x += f.x;
        acc.y += f.y;
      }
      __syncthreads();
    }
    cur ^= 1;
    nq = nnext;
  }
  if (h == 1) sums[wave][k] = acc;
  __syncthreads();
  if (t < kMaxP) {
    double2 s = sums[0][t];
    for (int w = 1; w < kSuperWaves; ++w) {
      s.x += sums[w][t].x;
      s.y += sums[w][t].y;
    }
    local[(int64_t)blockIdx.x * kMaxP + t] = s;
  }
  if (t == 0) super[blockIdx.x] = Super{cx, cy, R, over ? -1 : nf};
}

// ---------------------------------------------------------------------------- groups

struct GroupArgs {
  int64_t nt;
  int g;           // targets per wave
  int p;           // moments used, and terms of the local expansion
  int ksplit;      // waves per group: wave k takes every ksplit-th far cell and leaf
  uint32_t start;  // starting cells when there are no super groups (or one gave up): start ..
  uint32_t nstart; // start + nstart - 1, all of one level
  double theta;    // cells are far from radius / theta on
  float logtail;   // twice the logarithm (base 2) of the remainder that cells further away keep to
  double tol;
  const int* gate;  // set (or null): nothing is done
};

// One wave per G targets and share (blockIdx.y) of their far cells and leaves; every share opens
// the same cells. The wave's 64 / G slices
// hold the same targets and take different cells and leaves; their sums are added in slice order.
// ou..: the outputs in the targets' input order, or (part != null) partial sums by position,
// [component][ksplit][nt].
template <int CORE, bool ADJ, int G>
__global__ __launch_bounds__(kGroupBlock, 4) void tree_group_kernel(
    GroupArgs a, const Trg* __restrict__ trg, const uint32_t* __restrict__ torder,
    const double4* __restrict__ head, const uint2* __restrict__ kids,
    const double2* __restrict__ mom, const Src* __restrict__ src,
    const Super* __restrict__ super, const double2* __restrict__ local,
    const uint32_t* __restrict__ front, double* __restrict__ o0, double* __restrict__ o1,
    double* __restrict__ o2, double* __restrict__ o3, double* __restrict__ part) {
  constexpr int kSlices = 64 / G;
  constexpr int kItem = 2 * kLeaf;  // double2 elements of a leaf's records
  static_assert(kMaxP <= kItem && kItem % G == 0 && kMaxP % (G < kMaxP ? G : kMaxP) == 0,
                "whole loads per slice");
  __shared__ uint32_t stacks[kGroupWaves][kStack];
  // per slice the moments or the sources being worked on (rows apart by other than a multiple of
  // the banks, so that the slices' reads do not meet)
  __shared__ double2 buffers[kGroupWaves][kSlices][kItem + (kSlices > 1 ? 1 : 0)];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int slice = lane / G, mine = lane % G;
  const int64_t group = (int64_t)blockIdx.x * kGroupWaves + wave;
  if (group * G >= a.nt) return;  // whole waves; no workgroup barrier below
  if (a.gate && *a.gate != 0) return;
  uint32_t* st = stacks[wave];
  double2* data = buffers[wave][slice];
  const int64_t i = group * G + mine;
  const Trg tg = trg[i < a.nt ? i : a.nt - 1];
  const double x = tg.x, y = tg.y;
  const double wmine = target_term<CORE, ADJ>(tg);
  const double x0 = lanes_min<G>(x), x1 = lanes_max<G>(x);
  const double y0 = lanes_min<G>(y), y1 = lanes_max<G>(y);
  const double wt = __any(!(wmine < INFINITY)) ? INFINITY : lanes_max<G>(wmine);
  const double itheta = 1.0 / a.theta;
  const int p = a.p;
  // pairs: velocity u, v; adjoint dJ/ds, dJ/dx, dJ/dy, dJ/dr (the last three over the strength)
  double n0 = 0.0, n1 = 0.0, n2 = 0.0, n3 = 0.0;
  double2 S = make_double2(0.0, 0.0), S2 = S;  // far cells: S, and for the adjoint S2

  const uint32_t* init = nullptr;
  int64_t ninit = a.nstart;
  if (super) {
    const int64_t sg = group * G / kSuper;
    const Super sp = super[sg];
    if (sp.nfront >= 0) {
      init = front + sg * kFront;
      ninit = sp.nfront;
      if (blockIdx.y == 0) {  // the super group's local expansion at this target (slice 0's sums)
        double2* L = buffers[wave][0];
        if (lane < kMaxP) L[lane] = local[sg * kMaxP + lane];
        wave_sync();
        const double ir = sp.r > 0.0 ? 1.0 / sp.r : 0.0;
        const double2 z = make_double2((x - sp.cx) * ir, (y - sp.cy) * ir);
        double2 f = L[p - 1], g = make_double2(0.0, 0.0);
#pragma unroll 4
        for (int l = p - 2; l >= 0; --l) {
          if constexpr (ADJ) horner(g, z, f);
          horner(f, z, L[l]);
        }
        if (slice != 0) f = g = make_double2(0.0, 0.0);
        S = f;
        if constexpr (ADJ) S2 = make_double2(-g.x * ir, -g.y * ir);  // -dS/dz
      }
    }
  }
  // the next set bit of `bits` for every slice: this lane's in `from` (-1 when there is none
  // left), the lowest bits to the lowest slices
  auto deal = [&](unsigned long long& bits, int& from) {
    from = -1;
#pragma unroll
    for (int q = 0; q < kSlices; ++q) {
      const int b = bits ? __builtin_ctzll(bits) : -1;
      bits = bits ? bits & (bits - 1) : bits;
      from = slice == q ? b : from;
    }
  };
  // lane l's value (l the same in every lane of the wave when there is one slice)
  auto lane_of = [&](double v, int l) {
    if constexpr (kSlices == 1) return lane_f64(v, l);
    else return __shfl(v, l < 0 ? 0 : l, 64);
  };
  auto int_of = [&](int v, int l) {
    if constexpr (kSlices == 1) return __builtin_amdgcn_readlane(v, l);
    else return __shfl(v, l < 0 ? 0 : l, 64);
  };
  int sp = 0;
  int64_t next = 0;  // the next starting cell
  // this share's far cells and leaves: every ksplit-th of each kind
  unsigned nfar = 0, nleaf = 0;
  auto share = [&](unsigned long long bits, unsigned& seen) {
    if (a.ksplit == 1) return bits;
    const unsigned at = seen + __popcll(bits & ((1ull << lane) - 1ull));
    seen += __popcll(bits);
    return bits & __ballot(at % (unsigned)a.ksplit == blockIdx.y);
  };
  for (;;) {
    if (sp < 64 && next < ninit) {
      const int64_t at = next + lane;
      if (at < ninit) st[sp + lane] = init ? init[at] : a.start + (uint32_t)at;
      sp += ninit - next < 64 ? (int)(ninit - next) : 64;
      next += 64;
      wave_sync();
    }
    if (sp == 0) break;
    // as many of the top cells as the stack has room to open
    int m = (kStack - kStackSpare - sp) / 3;
    m = m < 1 ? 1 : (m < 64 ? m : 64);
    m = m < sp ? m : sp;
    sp -= m;
    const bool live = lane < m;
    const uint32_t ci = st[sp + (live ? lane : 0)];
    const double4 c = head[ci];
    const uint2 kd = kids[ci];
    const uint32_t first = kd.x, nkids = kd.y;
    // squared distances to the centre from which the core is 1/d^2 for every pair, and from which
    // the cell is far
    const double reach = c.z + core_reach<CORE>(c.w + wt, a.tol), open = c.z * itheta;
    const double rcore = reach * reach, rfar = fmax(rcore, open * open);
    // the box's squared distance, a little low so that no target is nearer
    const double bx = fmax(fmax(x0 - c.x, c.x - x1), 0.0);
    const double by = fmax(fmax(y0 - c.y, c.y - y1), 0.0);
    const double b2d = (bx * bx + by * by) * (1.0 - 1e-12);
    unsigned long long fbits = __ballot(live && b2d >= rfar);
    unsigned long long cbits = CORE == O2D_CORE_GAUSSIAN ? __ballot(live && b2d >= rcore) : 0ull;
    // cells too near the box may still be far from every target (a box that spans a jump of the
    // curve is mostly empty): target by target
    for (unsigned long long bits = __ballot(live) & ~fbits; bits;) {
      int from;
      deal(bits, from);
      const double ex = x - lane_of(c.x, from), ey = y - lane_of(c.y, from);
      const double e2 = __builtin_fma(ex, ex, ey * ey) * (1.0 - 1e-12);
      const double tfar = lane_of(rfar, from), tcore = lane_of(rcore, from);  // by every lane
      const unsigned long long mf = __ballot(from >= 0 && e2 >= tfar);
      const unsigned long long mc =
          CORE == O2D_CORE_GAUSSIAN ? __ballot(from >= 0 && e2 >= tcore) : 0ull;
      constexpr unsigned long long kAll = G == 64 ? ~0ull : (1ull << (G & 63)) - 1ull;
#pragma unroll
      for (int q = 0; q < kSlices; ++q) {
        const int f = __builtin_amdgcn_readlane(from, q * G);
        if (((mf >> (q * G)) & kAll) == kAll) fbits |= 1ull << f;
        if (((mc >> (q * G)) & kAll) == kAll) cbits |= 1ull << f;
      }
    }
    const bool far = (fbits >> lane) & 1ull;
    // orders that this cell needs at its distance: (r / d)^terms <= kShareTail theta^p, so that cells
    // nearer the limit keep all p and the others stay well below its truncation
    int terms = p;
    if (far && b2d >= rfar) {
      // the quotient in fp64: either square alone can leave the range of a float
      const float ratio =
          __builtin_amdgcn_logf((float)(c.z * c.z * __builtin_amdgcn_rcp(b2d)));
      const float need = __builtin_ceilf(a.logtail / ratio);
      terms = need < (float)p ? (need > 2.0f ? (int)need : 2) : p;
      terms = terms < p ? terms : p;
    }
    const bool leaf = live && !far && nkids == 0;
    const int nc = live && !far && !leaf ? (int)nkids : 0;
    const unsigned long long below = (1ull << lane) - 1ull;
    const unsigned long long b0 = __ballot(nc & 1), b1 = __ballot(nc & 2), b2 = __ballot(nc & 4);
    const int pc = __popcll(b0 & below) + 2 * __popcll(b1 & below) + 4 * __popcll(b2 & below);
    wave_sync();  // the popped entries have been read
    for (int e = 0; e < nc; ++e) st[sp + pc + e] = first + e;
    sp += __popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2);
    wave_sync();

    // The batch's far cells, then its leaves beyond the core, then the others, one a slice at a
    // time. Moments and records are loaded, an element per lane and load, while those before are
    // worked on, and go through LDS, which the slice's lanes read as broadcasts (as scalar loads
    // they arrive a few at a time: 18 ms, against 10, before the cells were tested by target)
    const uint32_t item = far ? ci : first;  // the cell, or the leaf
    const unsigned long long lbits = share(__ballot(leaf), nleaf);
    const unsigned long long mine_far = share(fbits, nfar);
    constexpr int kMomLoads = kMaxP > G ? kMaxP / G : 1, kLeafLoads = kItem / G;
    double2 nxt[kLeafLoads];
    auto load_mom = [&](int from) {
      const uint32_t id = __shfl(item, from < 0 ? 0 : from, 64);
      const double2* m = mom + (int64_t)id * kMaxP;
      if (from >= 0) {
#pragma unroll
        for (int e = 0; e < kMomLoads; ++e) nxt[e] = m[(e * G + mine) & (kMaxP - 1)];
      }
    };
    auto load_leaf = [&](int from) {
      const uint32_t id = __shfl(item, from < 0 ? 0 : from, 64);
      const double2* m = reinterpret_cast<const double2*>(src) + (int64_t)id * kItem;
      if (from >= 0) {
#pragma unroll
        for (int e = 0; e < kLeafLoads; ++e) nxt[e] = m[e * G + mine];
      }
    };
    {
      unsigned long long bits = mine_far;
      int from = -1, then = -1;
      if (bits) {
        deal(bits, then);
        load_mom(then);
      }
      for (bool more = mine_far != 0ull; more;) {
        from = then;
        wave_sync();  // the cells before have been read
#pragma unroll
        for (int e = 0; e < kMomLoads; ++e)
          if (e * G + mine < kMaxP) data[e * G + mine] = nxt[e];
        more = bits != 0ull;
        if (more) {
          deal(bits, then);
          load_mom(then);
        }
        wave_sync();
        // through its moments: t = r / (z - c), S += sum_k M_k t^k / (z - c)
        const double qr = lane_of(c.z, from), qx = lane_of(c.x, from), qy = lane_of(c.y, from);
        const int np = int_of(terms, from);
        if (from >= 0) {
          const double2 id = cinv(x - qx, y - qy);
          const double2 z = make_double2(qr * id.x, qr * id.y);
          double2 f = data[np - 1], g = make_double2(0.0, 0.0);
#pragma unroll 4
          for (int k = np - 2; k >= 0; --k) {
            if constexpr (ADJ) horner(g, z, f);
            horner(f, z, data[k]);
          }
          const double2 s1 = cmul(f, id);
          S.x += s1.x;
          S.y += s1.y;
          if constexpr (ADJ) {  // S2 = (f + t f') / (z - c)^2
            const double2 fz = cmul(g, z);
            const double2 s2 = cmul(make_double2(f.x + fz.x, f.y + fz.y), cmul(id, id));
            S2.x += s2.x;
            S2.y += s2.y;
          }
        }
      }
    }
    // leaves pair by pair: first those beyond the Gaussian's cutoff for every pair, without the
    // test per pair
    auto leaves = [&](unsigned long long bits, auto inner) {
      int from = -1, then = -1;
      if (!bits) return;
      deal(bits, then);
      load_leaf(then);
      for (bool more = true; more;) {
        from = then;
        wave_sync();
#pragma unroll
        for (int e = 0; e < kLeafLoads; ++e) data[e * G + mine] = nxt[e];
        more = bits != 0ull;
        if (more) {
          deal(bits, then);
          load_leaf(then);
        }
        wave_sync();
        if (from >= 0) inner(reinterpret_cast<const Src*>(data));
      }
    };
    if constexpr (CORE == O2D_CORE_GAUSSIAN) {
      leaves(lbits & cbits, [&](const Src* ls) {
#pragma unroll 8
        for (int k = 0; k < kLeaf; ++k) {
          const Src q = ls[k];
          if constexpr (ADJ) {
            const double dx = q.x - x, dy = q.y - y;
            const double kk = rcp64(__builtin_fma(dx, dx, dy * dy));
            const double tr = dx * kk, ti = -dy * kk;
            n0 = __builtin_fma(q.a, tr, __builtin_fma(q.b, ti, n0));
            const double sr2 = __builtin_fma(tr, tr, -ti * ti), si2 = 2.0 * tr * ti;
            n1 = __builtin_fma(q.a, sr2, __builtin_fma(q.b, si2, n1));
            n2 = __builtin_fma(q.b, sr2, __builtin_fma(-q.a, si2, n2));
          } else {
            const double ex = x - q.x, ey = y - q.y;
            const double g = q.a * rcp64(__builtin_fma(ex, ex, ey * ey));
            n0 = __builtin_fma(-g, ey, n0);
            n1 = __builtin_fma(g, ex, n1);
          }
        }
      });
    }
    leaves(lbits & ~cbits, [&](const Src* ls) {
#pragma unroll 4
      for (int k = 0; k < kLeaf; ++k) {
        const Src q = ls[k];
        if constexpr (ADJ) {
          const double dx = q.x - x, dy = q.y - y;
          const double d2 = __builtin_fma(dx, dx, dy * dy);
          double kk, bbb, dks;
          core_adj64<CORE>(dx, dy, d2, tg.w, kk, bbb, dks);
          const double w = __builtin_fma(q.a, dx, -q.b * dy);
          n0 = __builtin_fma(kk, w, n0);
          n3 = __builtin_fma(dks, w, n3);
          const double bxy = bbb * dx * dy;
          n1 += __builtin_fma(q.b, bxy, -q.a * __builtin_fma(bbb, dx * dx, kk));
          n2 += __builtin_fma(q.b, __builtin_fma(bbb, dy * dy, kk), -q.a * bxy);
        } else {
          const double ex = x - q.x, ey = y - q.y;
          const double e2 = __builtin_fma(ex, ex, ey * ey);
          const double w = wsum(q.b, tg.w);
          double k0;
          if constexpr (CORE == O2D_CORE_GAUSSIAN)  // near leaves hold most of the pairs inside cores
            k0 = e2 > kGaussFar * (1.0 + kCutMargin) * w ? rcp64(e2) : gauss_inside64(ex, ey, e2, w);
          else
            k0 = core_k64<CORE>(ex, ey, e2, w);
          const double g = q.a * k0;
          n0 = __builtin_fma(-g, ey, n0);
          n1 = __builtin_fma(g, ex, n1);
        }
      }
    });
    wave_sync();
  }
#pragma unroll
  for (int o = G; o < 64; o <<= 1) {  // the slices' sums
    n0 += __shfl_xor(n0, o, 64);
    n1 += __shfl_xor(n1, o, 64);
    S.x += __shfl_xor(S.x, o, 64);
    S.y += __shfl_xor(S.y, o, 64);
    if constexpr (ADJ) {
      n2 += __shfl_xor(n2, o, 64);
      n3 += __shfl_xor(n3, o, 64);
      S2.x += __shfl_xor(S2.x, o, 64);
      S2.y += __shfl_xor(S2.y, o, 64);
    }
  }
  if (slice != 0) return;
  if (i >= a.nt) return;
  if constexpr (ADJ) {
    // t = 1/(z_probe - z) = -1/(z - z_probe): sum G t = -S, sum G t^2 = S2
    n0 -= S.x;
    n1 = tg.s * (n1 + S2.x);
    n2 = tg.s * (n2 - S2.y);
    n3 *= tg.s;
  } else {
    n0 += S.y;
    n1 += S.x;
  }
  if (part) {
    const int64_t stride = (int64_t)a.ksplit * a.nt, at = (int64_t)blockIdx.y * a.nt + i;
    part[at] = n0;
    part[stride + at] = n1;
    if constexpr (ADJ) {
      part[2 * stride + at] = n2;
      part[3 * stride + at] = n3;
    }
  } else {
    const uint32_t o = torder[i];
    o0[o] += n0;
    o1[o] += n1;
    if constexpr (ADJ) {
      o2[o] += n2;
      o3[o] += n3;
    }
  }
}

inline unsigned blocks(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

struct Problem {
  int core;
  int order;  // the remainder of a far cell stays below theta^order
  int p;      // orders kept of a cell and of a local expansion
  double theta, tol;
  double share16, tail;  // of theta^order, for groups of 16 and for orders left out
  // sources, and their charges: strength and radius (velocity) or gv and gu (adjoint)
  int64_t ns;
  const double *sx, *sy, *sa, *sb;
  // targets: radius (may be null for the velocity) and strength (adjoint)
  int64_t nt;
  const double *tx, *ty, *tr, *ts;
  double *o0, *o1, *o2, *o3;
  int timed;  // kernel class of the evaluation
  // part of the pairs within the cutoff, as sampled, past which the sum goes pair by pair (0: never)
  double near_limit;
};

// log2 of the given share of theta^order
inline double remainder(const Problem& q, double share) {
  return q.order * std::log2(q.theta) + std::log2(share) * std::max(1.0, (double)q.order / kShareOrder);
}
// the r / d at which q.p orders leave that, at most theta
inline double limit(const Problem& q, double share) {
  return std::min(q.theta, std::exp2(remainder(q, share) / q.p));
}

template <int CORE, bool ADJ>
void launch_eval(const Problem& q, hipStream_t s, int64_t nsuper, const GroupArgs& ga,
                 const Trg* trg, const uint32_t* torder, const double4* head, const uint2* kids,
                 const double2* mom, const Src* src, uint32_t root, Super* super, double2* local, uint32_t* front,
                 double* part) {
  if (nsuper)
    tree_super_kernel<CORE, ADJ><<<(unsigned)nsuper, kSuperBlock, 0, s>>>(
        q.nt, trg, head, kids, mom, root, limit(q, kShareLocal), q.tol, super, local, front, ga.gate);
  const int64_t groups = (q.nt + ga.g - 1) / ga.g;
  const dim3 grid((unsigned)((groups + kGroupWaves - 1) / kGroupWaves), (unsigned)ga.ksplit);
  auto* sup = nsuper ? super : nullptr;
  if (ga.g == 16)
    tree_group_kernel<CORE, ADJ, 16><<<grid, kGroupBlock, 0, s>>>(
        ga, trg, torder, head, kids, mom, src, sup, local, front, q.o0, q.o1, q.o2, q.o3, part);
  else
    tree_group_kernel<CORE, ADJ, 64><<<grid, kGroupBlock, 0, s>>>(
        ga, trg, torder, head, kids, mom, src, sup, local, front, q.o0, q.o1, q.o2, q.o3, part);
}

template <bool ADJ>
int tree_run(Device* d, hipStream_t s, const Problem& q) {
  const int64_t ns = q.ns, nt = q.nt;
  Levels lv{};
  int64_t cnt = (ns + kLeaf - 1) / kLeaf, total = 0;
  for (;;) {
    if (lv.n == kMaxLevels) return fail(O2D_ERR_SIZE, "too many sources for the tree");
    lv.off[lv.n] = total;
    lv.cnt[lv.n] = cnt;
    total += cnt;
    ++lv.n;
    if (cnt == 1) break;
    cnt = (cnt + kFan - 1) / kFan;
  }
  const bool self = !ADJ && q.tx == q.sx && q.ty == q.sy && nt == ns;
  const bool same = self && q.tr == q.sb;  // sources and targets have the same records
  const int64_t nsrc = lv.cnt[0] * kLeaf;
  void *kb, *ko, *to, *sb, *cb, *bb, *mb;
  O2D_TRY(slot(d, kTreeKeys, sizeof(uint32_t) * std::max(ns, nt), s, &kb));
  O2D_TRY(slot(d, kTreeOrder, sizeof(uint32_t) * ns, s, &ko));
  O2D_TRY(slot(d, kTreeSrc, sizeof(Src) * nsrc, s, &sb));
  O2D_TRY(slot(d, kTreeCells, (sizeof(double4) + sizeof(uint2)) * total, s, &cb));
  O2D_TRY(slot(d, kTreeBox, sizeof(double4) * total, s, &bb));
  O2D_TRY(slot(d, kTreeMom, sizeof(double2) * kMaxP * total, s, &mb));
  uint32_t* sorder = static_cast<uint32_t*>(ko);
  Src* src = static_cast<Src*>(sb);
  double4* head = static_cast<double4*>(cb);
  uint2* kids = reinterpret_cast<uint2*>(head + total);
  double4* box = static_cast<double4*>(bb);
  double2* mom = static_cast<double2*>(mb);
  const uint32_t* torder = sorder;
  const Trg* trg;
  int* gate = nullptr;
  if (q.near_limit > 0.0) {
    void* gp;
    O2D_TRY(slot(d, kTreeGate, sizeof(int), s, &gp));
    gate = static_cast<int*>(gp);
  }
  {
    KernelTimer kt(O2D_KT_TREE_BUILD, s);
    O2D_TRY(morton_order(d, s, ns, q.sx, q.sy, true, 0.0, 0.0, 0.0, static_cast<uint32_t*>(kb),
                         sorder, nullptr, false));
    const int64_t lwaves = (nsrc + 63) / 64;
    tree_leaf_kernel<ADJ><<<(unsigned)((lwaves + kWaves - 1) / kWaves + (gate ? 1 : 0)), kBlock, 0, s>>>(
        ns, lv.cnt[0], q.p, sorder, q.sx, q.sy, q.sa, q.sb, q.core, src, head, kids, box, mom,
        Sample{nt, q.tx, q.ty, q.tr, q.near_limit, gate});
    O2D_LAUNCH_CHECK();
    for (int l = 0; l + 1 < lv.n; l += 2) {
      const bool two = l + 2 < lv.n;
      tree_up_kernel<<<(unsigned)((lv.cnt[l + 1] + kFan - 1) / kFan), kBlock, 0, s>>>(
          (uint32_t)lv.off[l], (uint32_t)lv.cnt[l], (uint32_t)lv.off[l + 1],
          (uint32_t)lv.cnt[l + 1], two ? (uint32_t)lv.off[l + 2] : 0u,
          two ? (uint32_t)lv.cnt[l + 2] : 0u, q.p, head, kids, box, mom);
      O2D_LAUNCH_CHECK();
    }
    if (!self) {
      O2D_TRY(slot(d, kTreeTOrder, sizeof(uint32_t) * nt, s, &to));
      O2D_TRY(morton_order(d, s, nt, q.tx, q.ty, true, 0.0, 0.0, 0.0, static_cast<uint32_t*>(kb),
                           static_cast<uint32_t*>(to), nullptr, false));
      torder = static_cast<const uint32_t*>(to);
    }
    if (same) {
      trg = reinterpret_cast<const Trg*>(src);
    } else {
      void* tb;
      O2D_TRY(slot(d, kTreeTrg, sizeof(Trg) * nt, s, &tb));
      tree_targets_kernel<ADJ><<<blocks(nt), kBlock, 0, s>>>(nt, torder, q.tx, q.ty, q.tr, q.ts,
                                                             q.core, static_cast<Trg*>(tb));
      O2D_LAUNCH_CHECK();
      trg = static_cast<const Trg*>(tb);
    }
    kt.stop();
  }
  GroupArgs ga{};
  ga.nt = nt;
  ga.p = q.p;
  ga.tol = q.tol;
  const int64_t nsup = (nt + kSuper - 1) / kSuper;
  const int64_t nsuper = nsup >= (ADJ ? kMinSupersAdjoint : kMinSupers) ? nsup : 0;
  ga.gate = gate;
  ga.g = nt < ns / (ADJ ? kSparseAdjoint : kSparse) ? 16 : 64;
  ga.theta = limit(q, ga.g == 64 ? kShare64 : q.share16);
  ga.logtail = (float)(2.0 * remainder(q, q.tail));
  const int64_t groups = (nt + ga.g - 1) / ga.g;
  const int64_t once = (int64_t)kWavesOnce * d->num_cu, most = (int64_t)kWaves64 * d->num_cu;
  ga.ksplit = (int)std::min<int64_t>(32, ga.g == 64 && groups > kEvenGroups
                                             ? (most + groups - 1) / groups
                                             : std::max<int64_t>(1, once / groups));
  // starting cells without a frontier: the lowest level that is tested in one go
  int sl = lv.n - 1;
  while (sl > 0 && lv.cnt[sl - 1] <= 64) --sl;
  ga.start = (uint32_t)lv.off[sl];
  ga.nstart = (uint32_t)lv.cnt[sl];
  KernelTimer kt(q.timed, s);
  // before the shares' partial sums are taken: both are the kPartials slot, which may move when it grows
  if (gate) {
    if constexpr (ADJ)
      O2D_TRY(adjoint_pairs_dev(d, s, q.core, nt, q.tx, q.ty, q.ts, q.tr, ns, q.sx, q.sy, q.sb, q.sa,
                                q.o1, q.o2, q.o0, q.o3, gate));
    else
      O2D_TRY(gauss_pairs_gated(d, s, ns, src, nt, trg, q.tr != nullptr, torder, q.o0, q.o1, gate));
  }
  const int nf = ADJ ? 4 : 2;
  double* part = nullptr;
  if (ga.ksplit > 1) {
    void* pp;
    O2D_TRY(slot(d, kPartials, sizeof(double) * nf * ga.ksplit * nt, s, &pp));
    part = static_cast<double*>(pp);
  }
  Super* super = nullptr;
  double2* local = nullptr;
  uint32_t* front = nullptr;
  if (nsuper) {
    void* up;
    O2D_TRY(slot(d, kTreeSuper,
                 (sizeof(Super) + sizeof(double2) * kMaxP + sizeof(uint32_t) * kFront) * nsuper, s,
                 &up));
    local = static_cast<double2*>(up);
    super = reinterpret_cast<Super*>(local + kMaxP * nsuper);
    front = reinterpret_cast<uint32_t*>(super + nsuper);
  }
  const uint32_t root = (uint32_t)lv.off[lv.n - 1];
#define O2D_EVAL(C) \
  launch_eval<C, ADJ>(q, s, nsuper, ga, trg, torder, head, kids, mom, src, root, super, local, front, part)
  switch (q.core) {
    case O2D_CORE_GAUSSIAN: O2D_EVAL(O2D_CORE_GAUSSIAN); break;
    default:
      if constexpr (!ADJ) {
        if (q.core == O2D_CORE_RM) O2D_EVAL(O2D_CORE_RM);
        else if (q.core == O2D_CORE_WL) O2D_EVAL(O2D_CORE_WL);
        else if (q.core == O2D_CORE_V2) O2D_EVAL(O2D_CORE_V2);
        else O2D_EVAL(O2D_CORE_V3);
      }
      break;
  }
#undef O2D_EVAL
  kt.stop();
  O2D_LAUNCH_CHECK();
  if (part) {
    O2D_TRY(reduce_chunks(s, ga.ksplit, nt, torder, nf, part, q.o0, q.o1, q.o2, q.o3, gate, 0));
  }
  return 0;
}

}  // namespace

int tree_dev(Device* d, hipStream_t s, int core, double theta, int p, double tol, int64_t ns,
             const double* sx, const double* sy, const double* ss, const double* sr, int64_t nt,
             const double* tx, const double* ty, const double* tr, double* tu, double* tv) {
  if (ns == 0 || nt == 0) return 0;
  const Problem q{core, p, kept_orders(p), theta, tol, kShare16, kShareTail, ns, sx, sy, ss, sr, nt, tx, ty, tr, nullptr,
                  tu, tv, nullptr, nullptr, O2D_KT_TREE_EVAL, 0.0};
  return tree_run<false>(d, s, q);
}

namespace {
// the sampled part of near pairs past which n targets are summed pair by pair (0: never)
inline double near_limit(double n, double limit, double whole, double many) {
  const double part = std::min(1.0, n / whole);
  return n < many ? limit * part * part : 0.0;
}
inline double filled(int64_t n, int64_t tile) { return (double)((n + tile - 1) / tile * tile); }
}  // namespace

bool gauss_clusters(const Device* d, int64_t ns, int64_t nt) {
  return (double)ns * filled(nt, sum64_targets(d, ns, nt)) >=
         kClusterPairs + kClusterSources * std::sqrt((double)ns) +
             std::min(kClusterTarget * nt, kClusterTargets);
}

bool gauss_adjoint_clusters(int64_t ns, int64_t nt) {
  return filled(ns, kAdjointTileS) * filled(nt, kAdjointTileT) >=
         kAdjointPairs + kAdjointParticle * ns + kAdjointProbe * nt +
             std::min(kAdjointFew * nt, kAdjointFewMost);
}

int gauss_tree_dev(Device* d, hipStream_t s, int64_t ns, const double* sx, const double* sy,
                   const double* ss, const double* sr, int64_t nt, const double* tx,
                   const double* ty, const double* tr, double* tu, double* tv) {
  const Problem q{O2D_CORE_GAUSSIAN, kMaxP, kMaxP, kExactTheta, 0.0, kExactShare16, kExactShareTail, ns, sx, sy, ss, sr, nt,
                  tx, ty, tr, nullptr, tu, tv, nullptr, nullptr,
                  tr ? O2D_KT_NBODY_PLAIN : O2D_KT_NBODY_PLAIN_PT,
                  near_limit((double)nt, kNearLimit, kNearTargets, kNearMany)};
  return tree_run<false>(d, s, q);
}

int gauss_adjoint_tree_dev(Device* d, hipStream_t s, int64_t ns, const double* sx,
                           const double* sy, const double* ss, const double* sr, int64_t nt,
                           const double* tx, const double* ty, const double* gu,
                           const double* gv, double* gx, double* gy, double* gs, double* gr) {
  const Problem q{O2D_CORE_GAUSSIAN, kMaxP, kMaxP, kExactTheta, 0.0, kExactShare16, kExactShareTail, nt, tx, ty, gv, gu, ns,
                  sx, sy, sr, ss, gs, gx, gy, gr, O2D_KT_ADJOINT,
                  near_limit((double)ns, kNearLimitAdjoint, kNearTargetsAdjoint, kNearManyAdjoint)};
  return tree_run<true>(d, s, q);
}

}  // namespace o2d

using namespace o2d;

extern "C" {

static int check_tree(const o2d_env* env, const o2d_tree_opts* opt, int64_t ns, const void* sx,
                      const void* sy, const void* ss, const void* sr, int64_t nt,
                      const void* tx, const void* ty, const void* tu, const void* tv) {
  O2D_TRY(check_env(env));
  if (env->results != O2D_VELONLY)
    return fail(O2D_ERR_RESULTS, "the treecode computes velocity only (results=%d)",
                env->results);
  if (!opt) return fail(O2D_ERR_ARG, "tree options are NULL");
  if (!(opt->theta > 0.0 && opt->theta < 1.0))
    return fail(O2D_ERR_ARG, "theta must lie in (0, 1) (got %g)", opt->theta);
  if (opt->order < 1 || opt->order > kMaxP)
    return fail(O2D_ERR_ARG, "expansion order must be 1..%d (got %d)", kMaxP, (int)opt->order);
  if (!(opt->core_tol >= 0.0)) return fail(O2D_ERR_ARG, "core_tol must be >= 0");
  if (ns < 0 || nt < 0) return fail(O2D_ERR_SIZE, "negative count");
  if (ns > 0x7fffffffLL || nt > 0x7fffffffLL) return fail(O2D_ERR_SIZE, "count too large");
  if (ns > 0 && (!sx || !sy || !ss || !sr)) return fail(O2D_ERR_ARG, "NULL source array");
  if (nt > 0 && (!tx || !ty || !tu || !tv)) return fail(O2D_ERR_ARG, "NULL target array");
  return 0;
}

int o2d_hip_points_on_points_tree_dev_d(const o2d_env* env, const o2d_tree_opts* opt,
                                        int64_t ns, const double* sx, const double* sy,
                                        const double* sstr, const double* srad, int64_t nt,
                                        const double* tx, const double* ty, const double* trad,
                                        double* tu, double* tv) {
  clear_error();
  O2D_TRY(check_tree(env, opt, ns, sx, sy, sstr, srad, nt, tx, ty, tu, tv));
  if (ns == 0 || nt == 0) return 0;
  Device* d;
  O2D_TRY(device(env->device, &d));
  return tree_dev(d, dev_stream(env), env->core, opt->theta, opt->order, opt->core_tol, ns, sx,
                  sy, sstr, srad, nt, tx, ty, trad, tu, tv);
}

int o2d_hip_points_on_points_tree_d(const o2d_env* env, const o2d_tree_opts* opt, int64_t ns,
                                    const double* sx, const double* sy, const double* sstr,
                                    const double* srad, int64_t nt, const double* tx,
                                    const double* ty, const double* trad, double* tu,
                                    double* tv) {
  clear_error();
  O2D_TRY(check_tree(env, opt, ns, sx, sy, sstr, srad, nt, tx, ty, tu, tv));
  if (ns == 0 || nt == 0) return 0;
  Device* d;
  O2D_TRY(device(env->device, &d));
  hipStream_t s = stream_of(env, d);
  double *dsx, *dsy, *dss, *dsr, *dtx, *dty, *dtr = nullptr, *du, *dv;
  O2D_TRY(upload<double>(d, kSrcX, sx, ns, s, &dsx));
  O2D_TRY(upload<double>(d, kSrcY, sy, ns, s, &dsy));
  O2D_TRY(upload<double>(d, kSrcS, sstr, ns, s, &dss));
  O2D_TRY(upload<double>(d, kSrcR, srad, ns, s, &dsr));
  O2D_TRY(upload<double>(d, kTrgX, tx, nt, s, &dtx));
  O2D_TRY(upload<double>(d, kTrgY, ty, nt, s, &dty));
  if (trad) O2D_TRY(upload<double>(d, kTrgR, trad, nt, s, &dtr));
  O2D_TRY(upload<double>(d, kOutU, tu, nt, s, &du));
  O2D_TRY(upload<double>(d, kOutV, tv, nt, s, &dv));
  O2D_TRY(tree_dev(d, s, env->core, opt->theta, opt->order, opt->core_tol, ns, dsx, dsy, dss,
                   dsr, nt, dtx, dty, dtr, du, dv));
  O2D_TRY(download<double>(tu, du, nt, s));
  O2D_TRY(download<double>(tv, dv, nt, s));
  O2D_HIP(hipStreamSynchronize(s));
  return 0;
}

}  // extern "C"

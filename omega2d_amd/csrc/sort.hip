// sort.hip - stable order of 32-bit keys made from the points themselves: Morton keys (32 or 16
// bits) of points on their own box or on a given one, and panel ends keyed by node. Every
// sorted path starts with one of these, and most of its cost is launches: a library radix sort
// of pairs ran as a merge sort at these sizes (a block sort and up to sixteen merge launches,
// 110 us for 200k or 1M points, 45 us for 10k), after three or four launches that made the keys.
//
// Up to kRankMax keys one launch does everything, box included, by counting for each key the keys that
// go before it (rank_kernel). Beyond, least significant digits first, 8 bits a pass: the box (one
// launch), the keys with the first digit's tile histograms (one launch), then one launch per digit. A
// scatter launch sums the histogram rows of the tiles before its own (every tile reads all rows from
// cache), ranks its keys within the tile by wave-wide digit matches (stable: a wave's keys are
// consecutive), and, in small tiles, counts the next digit of each key it places into the row of the
// tile it places it in, so no launch only counts. Counting uses integer atomics: sums do not depend on
// their order, and neither does the result.
// Arrays past kTiledMax keys go to the library sort, whose cost is then bandwidth: 2,000,000 keys take
// 148 us tiled and 157 by the library, 1,048,577 114 and 144, but 3,000,000 224 and 171. (With the next
// digit's count compiled into the large tiles' launches, where it is never taken, 16 keys a thread
// spilled: 250 us at 2,000,000.)
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cfloat>

#include "nbody.h"
#include "o2d_runtime.h"
#include "sort.h"

namespace o2d {

namespace {

constexpr int kBoxBlock = 256;
constexpr int kBoxBlocks = 256;  // partial boxes
constexpr int kST = 512;         // threads of a key or scatter workgroup
constexpr int kSW = kST / 64;
constexpr int kDigits = 256;
constexpr int64_t kTiledMax = 1 << 21;
constexpr int kCountItems = 2;   // keys per thread up to which a pass counts the next digit
constexpr int kRankT = 1024;     // threads of a rank workgroup
constexpr int kRankW = kRankT / 64;
constexpr int kRankMax = 12 * kRankT;

__device__ __forceinline__ uint32_t spread16(uint32_t v) {  // bits of v to the even positions
  v &= 0xFFFFu;
  v = (v | (v << 8)) & 0x00FF00FFu;
  v = (v | (v << 4)) & 0x0F0F0F0Fu;
  v = (v | (v << 2)) & 0x33333333u;
  v = (v | (v << 1)) & 0x55555555u;
  return v;
}

// q = clamp(floor(((v - x0) * inv) * 65536), 0, 65535) with unfused IEEE operations
__device__ __forceinline__ uint32_t quant16(double v, double v0, double inv) {
#pragma clang fp contract(off)
  double q = floor(__dmul_rn(__dmul_rn(__dsub_rn(v, v0), inv), 65536.0));
  q = q < 0.0 ? 0.0 : (q > 65535.0 ? 65535.0 : q);
  return (uint32_t)q;
}

struct Box {
  double x0, y0, x1, y1;  // smallest and largest coordinates (NaN left out)
};

// the key of point or panel end i. kMorton32: 16 bits per axis on the square box of the larger
// extent (x0, y0, inv given, or from the box); kMorton16: 8 bits per axis on the box itself
// (non-finite values only spoil the order); kNode: the end's node, clamped to the last one
template <int KIND>
__device__ __forceinline__ uint32_t make_key(const KeyGen& g, const Box& b, double x0, double y0,
                                             double inv, int64_t i) {
  if constexpr (KIND == kNode) {
    const uint32_t k = g.idx[i];
    return k < g.nnodes ? k : g.nnodes - 1;
  } else if constexpr (KIND == kMorton32) {
    return spread16(quant16(g.x[i], x0, inv)) | (spread16(quant16(g.y[i], y0, inv)) << 1);
  } else {
    double qx = (g.x[i] - b.x0) / (b.x1 - b.x0) * 255.0;
    double qy = (g.y[i] - b.y0) / (b.y1 - b.y0) * 255.0;
    qx = qx > 0.0 ? (qx < 255.0 ? qx : 255.0) : 0.0;  // NaN to 0
    qy = qy > 0.0 ? (qy < 255.0 ? qy : 255.0) : 0.0;
    return spread16((uint32_t)qx) | (spread16((uint32_t)qy) << 1);
  }
}

// origin and scale of the 32-bit keys: the given ones, or those of the points' square box
template <int KIND>
__device__ __forceinline__ void key_frame(const KeyGen& g, const Box& b, double& x0, double& y0,
                                          double& inv) {
  x0 = g.x0;
  y0 = g.y0;
  inv = g.inv;
  if (KIND == kMorton32 && g.bbox) {
    const double ext = fmax(b.x1 - b.x0, b.y1 - b.y0);
    x0 = b.x0;
    y0 = b.y0;
    inv = ext > 0.0 ? 1.0 / ext : 0.0;
  }
}

__device__ __forceinline__ Box empty_box() {
  return Box{INFINITY, INFINITY, -INFINITY, -INFINITY};
}
__device__ __forceinline__ void grow(Box& b, double x0, double y0, double x1, double y1) {
  b.x0 = fmin(b.x0, x0);
  b.y0 = fmin(b.y0, y0);
  b.x1 = fmax(b.x1, x1);
  b.y1 = fmax(b.y1, y1);
}

// the block's box in every thread (min and max are exact, so the order does not matter)
template <int WAVES>
__device__ __forceinline__ Box block_box(Box b, Box* sm) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    grow(b, __shfl_xor(b.x0, o, 64), __shfl_xor(b.y0, o, 64), __shfl_xor(b.x1, o, 64),
         __shfl_xor(b.y1, o, 64));
  if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = b;
  __syncthreads();
  b = sm[0];
#pragma unroll
  for (int w = 1; w < WAVES; ++w) grow(b, sm[w].x0, sm[w].y0, sm[w].x1, sm[w].y1);
  return b;
}

// part[b] = the box of points b kBoxBlock + t, striding by the grid
__global__ __launch_bounds__(kBoxBlock) void box_kernel(int64_t n, const double* __restrict__ x,
                                                        const double* __restrict__ y,
                                                        Box* __restrict__ part) {
  __shared__ Box sm[kBoxBlock / 64];
  Box b = empty_box();
  for (int64_t i = (int64_t)blockIdx.x * kBoxBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBoxBlock)
    grow(b, x[i], y[i], x[i], y[i]);
  b = block_box<kBoxBlock / 64>(b, sm);
  if (threadIdx.x == 0) part[blockIdx.x] = b;
}

// the keys of one tile of kST * ITEMS points, the tile's row of the first digit's histogram
// (tab[tile * kDigits + digit]), and zeros in its rows of the other digits' (rest: npass - 1
// tables of ntiles rows)
template <int KIND, int ITEMS>
__global__ __launch_bounds__(kST) void key_kernel(KeyGen g, int64_t n, const Box* __restrict__ part,
                                                  int npart, uint32_t* __restrict__ keys,
                                                  uint32_t* __restrict__ tab, int ntiles,
                                                  int npass) {
  __shared__ Box sm[kSW];
  __shared__ uint32_t hist[kDigits];
  const int t = threadIdx.x;
  if (t < kDigits) hist[t] = 0;
  Box b = empty_box();
  if (KIND != kNode && g.bbox) {
    for (int p = t; p < npart; p += kST) grow(b, part[p].x0, part[p].y0, part[p].x1, part[p].y1);
    b = block_box<kSW>(b, sm);
  }
  double x0, y0, inv;
  key_frame<KIND>(g, b, x0, y0, inv);
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * (kST * ITEMS);
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const int64_t i = base + k * kST + t;
    if (i < n) {
      const uint32_t key = make_key<KIND>(g, b, x0, y0, inv, i);
      keys[i] = key;
      atomicAdd(&hist[key & (kDigits - 1)], 1u);
    }
  }
  __syncthreads();
  if (t < kDigits) {
    tab[(int64_t)blockIdx.x * kDigits + t] = hist[t];
    for (int p = 1; p < npass; ++p) tab[((int64_t)p * ntiles + blockIdx.x) * kDigits + t] = 0;
  }
}

// LDS writes of this wave visible to its own later reads, and no compiler reordering across
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the lanes of `among` whose 8-bit digit equals this lane's
__device__ __forceinline__ unsigned long long match8(uint32_t digit, unsigned long long among) {
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const bool bit = (digit >> b) & 1u;
    const unsigned long long set = __ballot(bit);
    among &= bit ? set : ~set;
  }
  return among;
}

// exclusive prefix sums of v over the first kDigits threads of the workgroup (the others pass
// anything and get nothing); part: four partial sums in LDS
__device__ __forceinline__ uint32_t digit_scan(uint32_t v, uint32_t* part) {
  const int t = threadIdx.x, lane = t & 63;
  uint32_t inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t u = __shfl_up(inc, o, 64);
    if (lane >= o) inc += u;
  }
  if (t < kDigits && lane == 63) part[t >> 6] = inc;
  __syncthreads();
  uint32_t before = 0;
  for (int w = 0; w < kDigits / 64; ++w) before += (t >> 6) > w ? part[w] : 0u;
  return before + inc - v;
}

// the tile rows of one digit, for the passes whose counts are not taken by the pass before
template <int ITEMS>
__global__ __launch_bounds__(kST) void hist_kernel(int64_t n, int shift,
                                                   const uint32_t* __restrict__ keys,
                                                   uint32_t* __restrict__ tab) {
  __shared__ uint32_t hist[kDigits];
  const int t = threadIdx.x;
  if (t < kDigits) hist[t] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * (kST * ITEMS);
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const int64_t i = base + k * kST + t;
    if (i < n) atomicAdd(&hist[(keys[i] >> shift) & (kDigits - 1)], 1u);
  }
  __syncthreads();
  if (t < kDigits) tab[(int64_t)blockIdx.x * kDigits + t] = hist[t];
}

// one digit pass of a tile: keys (and their values; FIRST: the value is the index) to their
// places by digit (key >> shift) & 255; tab holds this digit's rows, next (unless null) takes
// the next digit's counts (up to kCountItems keys a thread). keys_out null: the keys are not needed any
// more.
template <int ITEMS, bool FIRST>
__global__ __launch_bounds__(kST) void scatter_kernel(int64_t n, int ntiles, int shift,
                                                      const uint32_t* __restrict__ keys_in,
                                                      const uint32_t* __restrict__ vals_in,
                                                      const uint32_t* __restrict__ tab,
                                                      uint32_t* __restrict__ next,
                                                      uint32_t* __restrict__ keys_out,
                                                      uint32_t* __restrict__ vals_out) {
  constexpr int kTile = kST * ITEMS;
  __shared__ uint32_t cnt[kSW][kDigits];  // per wave: counts, then offsets
  __shared__ uint4 rows[2][kSW][kDigits / 4];  // per wave: its rows' sums, all and before
  __shared__ uint32_t base[kDigits];
  __shared__ uint32_t part[kDigits / 64];
  static_assert(kDigits == 4 * 64, "a wave reads a row, four digits a lane");
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  for (int d = lane; d < kDigits; d += 64) cnt[wave][d] = 0;
  const int64_t first = (int64_t)blockIdx.x * kTile + wave * (64 * ITEMS) + lane;
  uint32_t key[ITEMS], val[ITEMS], rank[ITEMS];
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const int64_t i = first + 64 * k;
    key[k] = i < n ? keys_in[i] : 0u;
    val[k] = FIRST ? (uint32_t)i : (i < n ? vals_in[i] : 0u);
  }
  // the keys of every digit in all tiles and in those before this one: the waves share the rows
  uint4 all = make_uint4(0, 0, 0, 0), before = all;
  const uint4* tab4 = reinterpret_cast<const uint4*>(tab);
#pragma unroll 8
  for (int r = wave; r < ntiles; r += kSW) {
    const uint4 c = tab4[(int64_t)r * (kDigits / 4) + lane];
    all.x += c.x;
    all.y += c.y;
    all.z += c.z;
    all.w += c.w;
    if (r < (int)blockIdx.x) {
      before.x += c.x;
      before.y += c.y;
      before.z += c.z;
      before.w += c.w;
    }
  }
  rows[0][wave][lane] = all;
  rows[1][wave][lane] = before;
  wave_sync();
  const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const bool valid = first + 64 * k < n;
    const uint32_t d = (key[k] >> shift) & (kDigits - 1);
    const unsigned long long m = match8(d, __ballot(valid));
    const uint32_t had = cnt[wave][d];
    rank[k] = had + __popcll(m & below);
    wave_sync();
    if (valid && (m & below) == 0) cnt[wave][d] = had + __popcll(m);
    wave_sync();
  }
  __syncthreads();
  uint32_t total = 0, prior = 0;
  if (t < kDigits) {
#pragma unroll
    for (int w = 0; w < kSW; ++w) {
      total += reinterpret_cast<const uint32_t*>(rows[0][w])[t];
      prior += reinterpret_cast<const uint32_t*>(rows[1][w])[t];
    }
  }
  const uint32_t start = digit_scan(total, part);
  if (t < kDigits) {
    base[t] = start + prior;
    uint32_t run = 0;
#pragma unroll
    for (int w = 0; w < kSW; ++w) {
      const uint32_t c = cnt[w][t];
      cnt[w][t] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const bool valid = first + 64 * k < n;
    const uint32_t d = (key[k] >> shift) & (kDigits - 1);
    const uint32_t dst = base[d] + cnt[wave][d] + rank[k];
    if (valid) {
      if (keys_out) keys_out[dst] = key[k];
      vals_out[dst] = val[k];
    }
    if (ITEMS <= kCountItems && next) {
      // lanes with equal digits go to consecutive places; those that also share the next digit
      // and the destination tile count with one atomic (keys of clustered points share their
      // high digits)
      const uint32_t nd = (key[k] >> (shift + 8)) & (kDigits - 1);
      const unsigned long long live = __ballot(valid);
      const unsigned long long m = match8(nd, match8(d, live));
      if (valid) {
        const uint32_t tile = dst / kTile;
        const int last = 63 - __clzll(m), lead = __ffsll(m) - 1;
        const uint32_t tile_lead = __shfl(tile, lead, 64), tile_last = __shfl(tile, last, 64);
        uint32_t* slot = next + (int64_t)tile * kDigits + nd;
        if (tile_lead != tile_last)
          atomicAdd(slot, 1u);
        else if (lane == lead)
          atomicAdd(slot, (uint32_t)__popcll(m));
      }
    }
  }
}

// the whole order in one launch, n <= ITEMS * kRankT, by the place of each key: the keys below it,
// and the equal ones before it. Every workgroup makes all keys in LDS and places EACH of them, one to
// a lane; its waves share the blocks of 64 keys to compare with, and the 64 / EACH lanes with the same
// key share a block. Bound by latency up to 4,096 keys (7 us is the launch, two dependent passes over
// the points and their box), beyond by the integer units and LDS together: 8.4 us at 1,531 keys, 11.9
// at 4,096, 18.3 at 8,192, 25.3 at 10,000 and 28.9 at 12,288. A one-workgroup radix sort in LDS took
// 15.4 us at 1,531 (four digits, three barriers each), the six launches of the tiled passes 30 us and
// their gaps at 10,000; here 16,384 keys take 37 us, and n^2 comparisons no longer pay. Comparing 64
// keys with one scalar key and counting the mask's bits took 40 us at 10,000 (scalar registers), two
// keys a lane 28.
template <int KIND, int ITEMS, int EACH>
__global__ __launch_bounds__(kRankT) void rank_kernel(KeyGen g, int n,
                                                      uint32_t* __restrict__ keys_out,
                                                      uint32_t* __restrict__ vals_out) {
  __shared__ __align__(16) uint32_t sk[kRankT * ITEMS];
  __shared__ uint32_t cnt[kRankW][64];
  __shared__ Box sm[kRankW];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  Box b = empty_box();
  if (KIND != kNode && g.bbox) {
#pragma unroll 4
    for (int k = 0; k < ITEMS; ++k) {
      const int i = t + k * kRankT;
      if (i < n) grow(b, g.x[i], g.y[i], g.x[i], g.y[i]);
    }
    b = block_box<kRankW>(b, sm);
  }
  double x0, y0, inv;
  key_frame<KIND>(g, b, x0, y0, inv);
#pragma unroll 4
  for (int k = 0; k < ITEMS; ++k) {
    const int i = t + k * kRankT;
    // the padding goes after every key: it is only compared with keys before it, by <
    sk[i] = i < n ? make_key<KIND>(g, b, x0, y0, inv, i) : 0xFFFFFFFFu;
  }
  __syncthreads();
  const int i = blockIdx.x * EACH + lane % EACH, nblk = (n + 63) / 64;
  const int own = (blockIdx.x * EACH) / 64, part = (lane / EACH) * EACH;  // own: the keys' block
  const uint32_t mine = sk[i];
  uint32_t c = 0;
  for (int blk = wave; blk < nblk; blk += kRankW) {
    const int first = blk * 64 + part;
    const uint4* q = reinterpret_cast<const uint4*>(sk + first);
    if (blk < own) {
#pragma unroll
      for (int k = 0; k < EACH / 4; ++k) {
        const uint4 o = q[k];
        c += (o.x <= mine) + (o.y <= mine) + (o.z <= mine) + (o.w <= mine);
      }
    } else if (blk > own) {
#pragma unroll
      for (int k = 0; k < EACH / 4; ++k) {
        const uint4 o = q[k];
        c += (o.x < mine) + (o.y < mine) + (o.z < mine) + (o.w < mine);
      }
    } else {
#pragma unroll 4
      for (int k = 0; k < EACH; ++k) {
        const uint32_t o = sk[first + k];
        c += o < mine || (o == mine && first + k < i);
      }
    }
  }
  cnt[wave][lane] = c;
  __syncthreads();
  if (t >= EACH || i >= n) return;
  c = 0;
#pragma unroll
  for (int w = 0; w < kRankW; ++w)
#pragma unroll
    for (int p = 0; p < 64; p += EACH) c += cnt[w][lane + p];
  if (keys_out) keys_out[c] = mine;
  vals_out[c] = (uint32_t)i;
}

// the keys and their indices, for the library sort
template <int KIND>
__global__ __launch_bounds__(kBoxBlock) void pair_kernel(KeyGen g, int64_t n,
                                                         const Box* __restrict__ part, int npart,
                                                         uint32_t* __restrict__ keys,
                                                         uint32_t* __restrict__ vals) {
  __shared__ Box sm[kBoxBlock / 64];
  Box b = empty_box();
  if (KIND != kNode && g.bbox) {
    for (int p = threadIdx.x; p < npart; p += kBoxBlock)
      grow(b, part[p].x0, part[p].y0, part[p].x1, part[p].y1);
    b = block_box<kBoxBlock / 64>(b, sm);
  }
  double x0, y0, inv;
  key_frame<KIND>(g, b, x0, y0, inv);
  for (int64_t i = (int64_t)blockIdx.x * kBoxBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBoxBlock) {
    keys[i] = make_key<KIND>(g, b, x0, y0, inv, i);
    vals[i] = (uint32_t)i;
  }
}

// 16 keys a workgroup while that leaves no more than one for each of 256 compute units, then 32 or 64
// (each workgroup makes all keys: at 8,192 keys 16 took 25.5 us and 32 take 18.3)
template <int KIND>
void launch_rank(hipStream_t s, const KeyGen& g, int n, uint32_t* ko, uint32_t* vo) {
  if (n <= 2 * kRankT)
    rank_kernel<KIND, 2, 16><<<(n + 15) / 16, kRankT, 0, s>>>(g, n, ko, vo);
  else if (n <= 4 * kRankT)
    rank_kernel<KIND, 4, 16><<<(n + 15) / 16, kRankT, 0, s>>>(g, n, ko, vo);
  else if (n <= 8 * kRankT)
    rank_kernel<KIND, 8, 32><<<(n + 31) / 32, kRankT, 0, s>>>(g, n, ko, vo);
  else
    rank_kernel<KIND, 12, 64><<<(n + 63) / 64, kRankT, 0, s>>>(g, n, ko, vo);
}

template <int ITEMS>
void launch_keys(hipStream_t s, const KeyGen& g, int64_t n, int ntiles, int npass,
                 const Box* part, int npart, uint32_t* keys, uint32_t* tab) {
  switch (g.kind) {
    case kMorton32:
      key_kernel<kMorton32, ITEMS><<<ntiles, kST, 0, s>>>(g, n, part, npart, keys, tab, ntiles, npass);
      break;
    case kMorton16:
      key_kernel<kMorton16, ITEMS><<<ntiles, kST, 0, s>>>(g, n, part, npart, keys, tab, ntiles, npass);
      break;
    default:
      key_kernel<kNode, ITEMS><<<ntiles, kST, 0, s>>>(g, n, part, npart, keys, tab, ntiles, npass);
      break;
  }
}

// keys in kf, then the passes, alternating between the pairs (kf, vf) and (kb, vb); the last
// one ends in the caller's arrays
template <int ITEMS>
int sort_tiles(hipStream_t s, const KeyGen& g, int64_t n, int npass, const Box* part, int npart,
               uint32_t* keys_out, uint32_t* vals_out, uint32_t* kt, uint32_t* vt, uint32_t* tab,
               bool want_keys) {
  const int ntiles = (int)((n + kST * ITEMS - 1) / (kST * ITEMS));
  // pass p writes the caller's arrays when (npass - 1 - p) is even
  uint32_t* kin = npass % 2 == 0 ? keys_out : kt;
  const uint32_t* vin = nullptr;
  launch_keys<ITEMS>(s, g, n, ntiles, npass, part, npart, kin, tab);
  O2D_LAUNCH_CHECK();
  const bool count_next = ITEMS <= kCountItems;
  for (int p = 0; p < npass; ++p) {
    const bool to_out = (npass - 1 - p) % 2 == 0, last = p == npass - 1;
    uint32_t* ko = to_out ? keys_out : kt;
    uint32_t* vo = to_out ? vals_out : vt;
    const uint32_t* row = tab + (int64_t)p * ntiles * kDigits;
    uint32_t* next = last || !count_next ? nullptr : tab + (int64_t)(p + 1) * ntiles * kDigits;
    if (p > 0 && !count_next) {
      hist_kernel<ITEMS><<<ntiles, kST, 0, s>>>(n, 8 * p, kin, tab + (int64_t)p * ntiles * kDigits);
      O2D_LAUNCH_CHECK();
    }
    uint32_t* kw = last && !want_keys ? nullptr : ko;
    if (p == 0)
      scatter_kernel<ITEMS, true><<<ntiles, kST, 0, s>>>(n, ntiles, 8 * p, kin, vin, row, next, kw, vo);
    else
      scatter_kernel<ITEMS, false><<<ntiles, kST, 0, s>>>(n, ntiles, 8 * p, kin, vin, row, next, kw, vo);
    O2D_LAUNCH_CHECK();
    kin = ko;
    vin = vo;
  }
  return 0;
}

}  // namespace

int sort_order(Device* d, hipStream_t s, Workspace* ws, int64_t n, const KeyGen& g, int bits,
               uint32_t* keys_out, uint32_t* order_out, bool want_keys) {
  if (n <= 0) return 0;
  const int npass = (bits + 7) / 8;
  if (n <= kRankMax) {
    uint32_t* ko = want_keys ? keys_out : nullptr;
    switch (g.kind) {
      case kMorton32: launch_rank<kMorton32>(s, g, (int)n, ko, order_out); break;
      case kMorton16: launch_rank<kMorton16>(s, g, (int)n, ko, order_out); break;
      default: launch_rank<kNode>(s, g, (int)n, ko, order_out); break;
    }
    O2D_LAUNCH_CHECK();
    return 0;
  }
  void *kt, *vt, *tab = nullptr, *bp = nullptr;
  O2D_TRY(take(d, ws, kKeysA, n * sizeof(uint32_t), s, &kt));
  O2D_TRY(take(d, ws, kOrderA, n * sizeof(uint32_t), s, &vt));
  int npart = 0;
  if (g.bbox) {
    npart = (int)std::min<int64_t>((n + kBoxBlock - 1) / kBoxBlock, kBoxBlocks);
    O2D_TRY(take(d, ws, kBBox, sizeof(Box) * kBoxBlocks, s, &bp));
    box_kernel<<<npart, kBoxBlock, 0, s>>>(n, g.x, g.y, static_cast<Box*>(bp));
    O2D_LAUNCH_CHECK();
  }
  const Box* part = static_cast<const Box*>(bp);
  uint32_t* k0 = static_cast<uint32_t*>(kt);
  uint32_t* v0 = static_cast<uint32_t*>(vt);
  if (n <= kTiledMax) {
    // tiles of 1,024 to 8,192 keys: enough of them to spread a pass over the chip, few enough (256)
    // that every tile can sum the rows of all
    const int items = n <= (1 << 16) ? 2 : (n <= (1 << 18) ? 4 : (n <= (1 << 20) ? 8 : 16));
    const int64_t ntiles = (n + (int64_t)kST * items - 1) / ((int64_t)kST * items);
    O2D_TRY(take(d, ws, kSortTab, sizeof(uint32_t) * kDigits * (size_t)ntiles * (size_t)npass, s, &tab));
    uint32_t* tb = static_cast<uint32_t*>(tab);
    if (items == 2) return sort_tiles<2>(s, g, n, npass, part, npart, keys_out, order_out, k0, v0, tb, want_keys);
    if (items == 4) return sort_tiles<4>(s, g, n, npass, part, npart, keys_out, order_out, k0, v0, tb, want_keys);
    if (items == 8) return sort_tiles<8>(s, g, n, npass, part, npart, keys_out, order_out, k0, v0, tb, want_keys);
    return sort_tiles<16>(s, g, n, npass, part, npart, keys_out, order_out, k0, v0, tb, want_keys);
  }
  const unsigned blocks = 4096;
  switch (g.kind) {
    case kMorton32: pair_kernel<kMorton32><<<blocks, kBoxBlock, 0, s>>>(g, n, part, npart, k0, v0); break;
    case kMorton16: pair_kernel<kMorton16><<<blocks, kBoxBlock, 0, s>>>(g, n, part, npart, k0, v0); break;
    default: pair_kernel<kNode><<<blocks, kBoxBlock, 0, s>>>(g, n, part, npart, k0, v0); break;
  }
  O2D_LAUNCH_CHECK();
  size_t tbytes = 0;
  O2D_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tbytes, k0, keys_out, v0, order_out, (int)n,
                                             0, bits, s));
  void* tmp;
  O2D_TRY(take(d, ws, kSortTemp, tbytes, s, &tmp));
  O2D_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tbytes, k0, keys_out, v0, order_out, (int)n, 0,
                                             bits, s));
  return 0;
}

// Morton keys and the stable key order; bbox == true derives the box from the data on device.
int morton_order(Device* d, hipStream_t s, int64_t n, const double* x, const double* y,
                 bool bbox, double x0, double y0, double inv, uint32_t* keys_out,
                 uint32_t* order_out, Workspace* ws, bool want_keys) {
  KeyGen g{};
  g.kind = kMorton32;
  g.bbox = bbox;
  g.x = x;
  g.y = y;
  g.x0 = x0;
  g.y0 = y0;
  g.inv = inv;
  return sort_order(d, s, ws, n, g, 32, keys_out, order_out, want_keys);
}

int morton_order16(Device* d, hipStream_t s, int64_t n, const double* x, const double* y,
                   const uint32_t** order) {
  void *kB, *vB;
  O2D_TRY(slot(d, kKeysB, n * sizeof(uint32_t), s, &kB));
  O2D_TRY(slot(d, kOrderB, n * sizeof(uint32_t), s, &vB));
  KeyGen g{};
  g.kind = kMorton16;
  g.bbox = true;
  g.x = x;
  g.y = y;
  O2D_TRY(sort_order(d, s, nullptr, n, g, 16, static_cast<uint32_t*>(kB),
                     static_cast<uint32_t*>(vB), false));
  *order = static_cast<const uint32_t*>(vB);
  return 0;
}

}  // namespace o2d

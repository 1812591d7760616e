// The spatial order of the pruned passes, on the device: each range of points
// is split at a tile boundary near its middle along its widest feature, until
// each range is one tile, and tiles into their waves' 32 rows (down to the tile
// the behaviour of reference src/spatial.cuh:48-91, which does it on the host).
// Ties between equal weights always break by original index, so results do
// not depend on the order; it only decides how much a pass can skip.
//
// One level at a time, every range of the level together: a wave per range
// finds the widest feature of a sample, every point's key is (range, value of
// that feature quantised to 16 bits; fewer above some ten million points), and
// one stable radix sort of the keys splits all ranges at their middles. Far
// values (missing entries coded as 1e9, say) must not take the steps from those
// around the middle, which alone count: with steps over the whole sample's spread
// the walks over 30,000 points of 4 features, 3% of the rows at 1e6 in each,
// computed 24% of the tiles, now 9%, and 5% without those values. A range is
// named by its path (a bit per level), which orders ranges as they lie and needs
// no more bits than there are levels.
// Bound by launches up to some 10^5 points, then by the sorts' passes. With the
// order made on the host (16 threads; points on the device were copied there
// first) whole calls took: single linkage, manhattan, 50,021 x 10, 18.9 ms, now
// 13.6; HDBSCAN of 100,000 x 8 (two orders) 48.3, now 42.5; of 10^6 x 8 611, now
// 551. On these inputs the quantised splits cost the passes up to 6% (fused core
// pass of the 100,000 points 10.9 to 11.6 ms).
#include "mst.hpp"

#include "primitives.hpp"

#include <algorithm>

namespace cuhc {

namespace {

constexpr int kTilePoints = 128;
constexpr int kUnitPoints = 32; // a wave's rows of a tile: the finest ranges
constexpr int kTileUnits = kTilePoints / kUnitPoints;
constexpr int kSample = 64;      // sampled points per range: one per lane
constexpr int kMaxValueBits = 16;

// Where the units [lo, hi) split: between tiles while there is more than one,
// then between units; a single unit has an empty right half.
DEV int middleOf(int lo, int hi) {
  const int units = hi - lo;
  if (units > kTileUnits)
    return lo + (units + kTileUnits - 1) / kTileUnits / 2 * kTileUnits;
  return units > 1 ? lo + (units + 1) / 2 : hi;
}

// Units [lo, hi) of a range of the level, from its path.
DEV void rangeOfPath(unsigned int path, int level, int units, int &lo, int &hi) {
  lo = 0;
  hi = units;
  for (int l = level - 1; l >= 0; --l) {
    const int mid = middleOf(lo, hi);
    if (path >> l & 1)
      lo = mid;
    else
      hi = mid;
  }
}

DEV unsigned int pathOfUnit(int unit, int level, int units) {
  int lo = 0, hi = units;
  unsigned int path = 0;
  for (int l = 0; l < level; ++l) {
    const int mid = middleOf(lo, hi);
    const bool right = unit >= mid;
    path = path << 1 | (right ? 1u : 0u);
    if (right)
      lo = mid;
    else
      hi = mid;
  }
  return path;
}

// How a range's points are quantised: 0 below low, the highest step above high,
// between them evenly, or (byBits) evenly in the order of the floats' bits.
struct Split {
  int feature; // -1: a single unit, all points 0
  float low, high, scale;
  int shift; // byBits: steps of 2^shift; else -1
};

DEV unsigned int orderOf(float v) {
  const unsigned int b = __float_as_uint(v + 0.0f); // -0 as 0
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// The steps for a sample (v: a value per lane) with far values, to split at rank
// r: over the three quarters of the sample about it, evenly or, where the values
// next to the split would still share few steps (more than an eighth is far), by
// the bits, 128 steps or more for values from x to 2 x.
DEV void splitFarValues(float v, int r, int valueBits, Split &split) {
  auto of = [&](int lane) { // uniform lane
    return __uint_as_float((unsigned int)__builtin_amdgcn_readlane((int)__float_as_uint(v), lane));
  };
  int rank = 0;
#pragma unroll 8
  for (int j = 0; j < kSample; ++j) {
    const float other = of(j);
    rank += other < v || (other == v && j < (int)threadIdx.x);
  }
  auto ranked = [&](int at) {
    return of(__ffsll((long long)__ballot(rank == min(max(at, 0), kSample - 1))) - 1);
  };
  split.low = ranked(r - 3 * kSample / 8);
  split.high = ranked(r + 3 * kSample / 8);
  const float spread = split.high - split.low;
  const float near = ranked(r + kSample / 16) - ranked(r - kSample / 16);
  if (spread < INFINITY && spread <= near * 256.0f) {
    split.scale = spread > 0.0f ? (float)((1 << valueBits) - 3) / spread : 0.0f;
  } else {
    const unsigned int range = orderOf(split.high) - orderOf(split.low);
    split.shift = max(0, 32 - __clz((int)range) - (valueBits - 1));
  }
}

__global__ void __launch_bounds__(64)
    splitsKernel(const float *__restrict__ X, int d, const int *__restrict__ order, int count,
                 int level, int units, int valueBits, Split *__restrict__ splits) {
  int lo, hi;
  rangeOfPath(blockIdx.x, level, units, lo, hi);
  Split best{-1, 0.0f, 0.0f, 0.0f, -1};
  if (hi - lo > 1) {
    const int begin = lo * kUnitPoints, end = min(count, hi * kUnitPoints);
    const long long at = begin + (long long)(end - begin) * threadIdx.x / kSample;
    const float *row = X + (size_t)order[at] * d;
    float widest = -1.0f;
    for (int f = 0; f < d; ++f) {
      float low = row[f], high = low;
#pragma unroll
      for (int m = 32; m > 0; m >>= 1) {
        low = fminf(low, __shfl_xor(low, m, 64));
        high = fmaxf(high, __shfl_xor(high, m, 64));
      }
      if (high - low > widest) {
        widest = high - low;
        best.feature = f;
        best.low = low;
        best.high = high;
      }
    }
    // Steps evenly over the sample's spread, unless more than half of it shares a
    // 64th of them: eight of its values are looked at, one in 256 such halves
    // is missed.
    const float steps = (float)((1 << valueBits) - 3);
    const float v = row[best.feature];
    best.scale = widest > 0.0f ? steps / widest : 0.0f;
    const int part = (int)((v - best.low) * (best.scale * (64.0f / steps)));
    int most = 0;
#pragma unroll
    for (int j = kSample / 16; j < kSample; j += kSample / 8)
      most = max(most, __popcll(__ballot(part == __builtin_amdgcn_readlane(part, j))));
    if (2 * most > kSample || !(widest < INFINITY))
      splitFarValues(v, (int)((long long)(middleOf(lo, hi) * kUnitPoints - begin) * kSample /
                              (end - begin)), valueBits, best);
  }
  if (threadIdx.x == 0)
    splits[blockIdx.x] = best;
}

__global__ void keysKernel(const float *__restrict__ X, int d, const int *__restrict__ order,
                           int count, int level, int units, int valueBits,
                           const Split *__restrict__ splits, unsigned int *__restrict__ keys) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= count)
    return;
  const unsigned int path = pathOfUnit(p / kUnitPoints, level, units);
  const Split s = splits[path];
  const unsigned int top = (1u << valueBits) - 1u;
  unsigned int q = 0;
  if (s.feature >= 0) {
    const float v = X[(size_t)order[p] * d + s.feature];
    if (v > s.high)
      q = top;
    else if (v >= s.low)
      q = 1 + min(top - 2, s.shift < 0 ? (unsigned int)((v - s.low) * s.scale)
                                       : (orderOf(v) - orderOf(s.low)) >> s.shift);
  }
  keys[p] = path << valueBits | q;
}

__global__ void startKernel(const int *__restrict__ list, int count, int *__restrict__ order) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < count)
    order[p] = list ? list[p] : p;
}

__global__ void coreKeysKernel(const float *__restrict__ core, int n,
                               unsigned int *__restrict__ keys, int *__restrict__ positions) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) {
    keys[p] = __float_as_uint(core[p]); // non-negative: bits order like values
    positions[p] = p;
  }
}

__global__ void highFlagsKernel(const float *__restrict__ core, int n,
                                const unsigned int *__restrict__ threshold,
                                int *__restrict__ flags) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p <= n)
    flags[p] = p < n && __float_as_uint(core[p]) > *threshold;
}

// Positions in ascending order, the unflagged ones first.
__global__ void partitionKernel(const int *__restrict__ flags, const int *__restrict__ before,
                                int n, int *__restrict__ list) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n)
    list[flags[p] ? n - before[n] + before[p] : p - before[p]] = p;
}

__global__ void composeKernel(const int *__restrict__ newToOld, const int *__restrict__ orig,
                              int n, int *__restrict__ out) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n)
    out[p] = orig[newToOld[p]];
}

__global__ void scatterFloatsKernel(const float *__restrict__ src, const int *__restrict__ to,
                                    int n, float *__restrict__ dst) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n)
    dst[to[p]] = src[p];
}

inline dim3 gridFor(long long count) { return dim3((unsigned)((count + 255) / 256)); }

} // namespace

int spatialOrder(const float *X, int d, const int *list, int count, int *order) {
  hipLaunchKernelGGL(startKernel, gridFor(count), dim3(256), 0, stream(), list, count, order);
  const int units = (count + kUnitPoints - 1) / kUnitPoints;
  const int tiles = (count + kTilePoints - 1) / kTilePoints;
  int levels = 0;
  while ((1LL << levels) < tiles)
    ++levels;
  for (int u = std::min(units, kTileUnits); u > 1; u = (u + 1) / 2)
    ++levels; // inside the tiles
  // Paths and values share 32 bits (2^24 tiles are 2^31 points).
  const int valueBits = std::min(kMaxValueBits, 32 - levels);
  Status s;
  DevArray<Split> splits;
  DevArray<unsigned int> keys, keysOut;
  DevArray<int> other;
  DevArray<unsigned char> temp;
  s(splits.alloc((size_t)1 << levels));
  s(keys.alloc(count));
  s(keysOut.alloc(count));
  s(other.alloc(count));
  s(temp.alloc(sortTempBytes32(count)));
  int *from = order, *to = other.get();
  for (int level = 0; level < levels && s.ok(); ++level) {
    hipLaunchKernelGGL(splitsKernel, dim3(1u << level), dim3(64), 0, stream(), X, d, from, count,
                       level, units, valueBits, splits.get());
    hipLaunchKernelGGL(keysKernel, gridFor(count), dim3(256), 0, stream(), X, d, from, count,
                       level, units, valueBits, splits.get(), keys.get());
    s((int)hipGetLastError());
    s(radixSortPairs(keys.get(), keysOut.get(), from, to, count, level + valueBits, temp));
    std::swap(from, to);
  }
  if (s.ok() && from != order)
    hipLaunchKernelGGL(startKernel, gridFor(count), dim3(256), 0, stream(), from, count, order);
  s((int)hipGetLastError());
  return s.code;
}

int coreStratifiedOrder(const float *X, int n, int d, const float *core, const int *orig,
                        int *newToOld, int *newOrig, bool *stratified) {
  *stratified = false;
  Status s;
  DevArray<unsigned int> keys, keysOut;
  DevArray<int> positions, list, flags, before;
  DevArray<unsigned char> temp, scanTemp;
  s(keys.alloc(n));
  s(keysOut.alloc(n));
  s(positions.alloc(n));
  s(list.alloc(n));
  s(flags.alloc((size_t)n + 1));
  s(before.alloc((size_t)n + 1));
  s(temp.alloc(sortTempBytes32(n)));
  s(scanTemp.alloc(scanTempBytes(n + 1)));
  if (!s.ok())
    return s.code;
  hipLaunchKernelGGL(coreKeysKernel, gridFor(n), dim3(256), 0, stream(), core, n, keys.get(),
                     positions.get());
  s(radixSortPairs(keys.get(), keysOut.get(), positions.get(), list.get(), n, 32, temp));
  hipLaunchKernelGGL(highFlagsKernel, gridFor(n + 1), dim3(256), 0, stream(), core, n,
                     keysOut.get() + (size_t)(0.9 * n), flags.get());
  s(exclusiveScan(flags, before, n + 1, scanTemp));
  hipLaunchKernelGGL(partitionKernel, gridFor(n), dim3(256), 0, stream(), flags.get(),
                     before.get(), n, list.get());
  s((int)hipGetLastError());
  int high = 0;
  s(download(&high, before.get() + n, sizeof(int)));
  if (!s.ok() || high < kTilePoints || n - high < kTilePoints)
    return s.code;
  s(spatialOrder(X, d, list, n - high, newToOld));
  s(spatialOrder(X, d, list.get() + (n - high), high, newToOld + (n - high)));
  hipLaunchKernelGGL(composeKernel, gridFor(n), dim3(256), 0, stream(), newToOld, orig, n,
                     newOrig);
  s((int)hipGetLastError());
  *stratified = s.ok();
  return s.code;
}

int scatterFloats(const float *src, const int *to, int n, float *dst) {
  hipLaunchKernelGGL(scatterFloatsKernel, gridFor(n), dim3(256), 0, stream(), src, to, n, dst);
  return (int)hipGetLastError();
}

} // namespace cuhc

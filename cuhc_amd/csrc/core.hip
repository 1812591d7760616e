// Core distances: core[i] = the k-th smallest distance from point i to the
// points, the point itself counted as the 1st (distance 0), values clamped at
// 0 (reference src/hdbscan.cuh:35-338).
//
// fused (k <= 64): one workgroup per row tile walks the column tiles nearest
//   first and keeps each row's k smallest distances sorted in LDS. After each
//   tile the 16 lanes of a row mark the distances that beat the row's k-th,
//   and insert them together, one value per step (64-bit ballot over the
//   wave: 4 rows insert in parallel). Optional box pruning for points in
//   spatial order, per wave: one box and one largest k-th distance over 128
//   rows computed 47% of the pairs of 100,000 points of 8 features, by 32 rows
//   26% (10^6 points, k = 25: core pass 159 to 135 ms, 100,000: 11.6 to 7.6).
// radix: distances of a block of rows into a bounded buffer, then per row a
//   4-pass MSB-first byte radix select over the FP32 bit patterns with
//   per-wave LDS histograms.
// Both are exact and bit-identical (the k-th smallest value is unique).
//
// Bound by FP32 VALU work and, where the walks' lengths differ, by the longest:
// the pruned pass over all points takes its row tiles largest box first, as
// sparse rows walk farthest (10^6 points, k = 25: 122 to 104 ms; before, 72 ms
// of it issued VALU instructions). With few row tiles a walk is split over
// gridDim.y workgroups. Each keeps a list of its own columns; rows share a bound
// (kthBits), the smallest k-th distance that any split has found, and first the
// one within the home tile, from a pass of its own: values from the bound on
// are left out. A second kernel takes the k-th of a row's lists and bound
// (100,000 points, k = 25: 7.6 to 5.9 ms; 6.5 without the order of the tiles,
// 7.5 without the first bound, as every split filled its lists with far values).
#include "mst.hpp"
#include "primitives.hpp"
#include "tile.hpp"

#include <algorithm>
#include <type_traits>

namespace cuhc {

namespace {

// Column tile boxes (low/high per tile; numTiles > 0 turns pruning on).
struct CoreBoxes {
  const float *low = nullptr, *high = nullptr;
  int numTiles = 0;
};

// Of a walk in splits, split 0 takes the home tile and split s every splits-th
// pair of tiles beside it (-1: none): each column tile is one split's.
DEV int walkTileCore(int rowTile, int step, int numTiles, int splits = 1, int split = 0) {
  const int pair = (step + 1) >> 1;
  if (pair == 0 && split > 0)
    return -1;
  const int off = pair == 0 ? 0 : (pair - 1) * splits + split + 1;
  const int tile = (step & 1) ? rowTile + off : rowTile - off;
  return (tile >= 0 && tile < numTiles) ? tile : -1;
}

HD float coreBoxSlack(int d) { return 1e-5f + (d + 8) * 5e-7f; }

template <class Metric>
DEV float coreBoxBound(const Metric &metric, const float *lowA, const float *highA,
                       const float *lowB, const float *highB, int d) {
  typename Metric::Acc acc = metric.init();
  for (int k = 0; k < d; ++k) {
    const float gap = fmaxf(0.0f, fmaxf(lowB[k] - highA[k], lowA[k] - highB[k]));
    acc = metric.fold(acc, gap, 0.0f);
  }
  return metric.finish(acc);
}

// Inserts v into the ascending list[0..k), dropping the largest, by the 16
// lanes of a tile row (lane16 = 0..15) together: entry s keeps its value up to
// v, and above v takes the larger of v and its predecessor. One LDS round trip;
// one lane shifting the entries took one per entry (k = 25: 2,003 points
// unpruned 3.3 ms, now 0.96; 24,000 points of 20 features 6.9 ms, now 3.6).
DEV void insertSorted(float *list, int k, int lane16, float v) {
  // From the last 16 entries to the first: an entry's predecessor is read
  // before it is written.
#pragma unroll 1
  for (int s = (k - 1) / 16 * 16 + lane16; s >= 0; s -= 16) {
    if (s < k) {
      const float cur = list[s], prev = s > 0 ? list[s - 1] : -INFINITY;
      list[s] = cur > v ? fmaxf(prev, v) : cur;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// Rows are the points themselves (rowsX null: row tile blockIdx.x of X, or
// tile tileList[blockIdx.x] with a list) or listed points (rowsX: numRows
// gathered rows, rowPos their positions in X, for the exact search of
// selected points).
// Three waves per SIMD for the one-fill tiles (d <= 8) of the squared-sum
// metrics: the pass waits on tile loads, and 160 VGPRs hold it without spills
// (at four, 62 registers spill: 10^6 points, d = 8, 225 ms against 166 before
// the rows were bounded by wave).
template <class T, class Metric> constexpr int coreMinWaves() {
  return T::FILL <= 8 &&
                 (std::is_same<Metric, Euclidean>::value || std::is_same<Metric, SqEuclidean>::value)
             ? 3
             : 1;
}

template <class T, class Metric>
__global__ void __launch_bounds__(256, (coreMinWaves<T, Metric>()))
    kthNearestFusedKernel(const float *__restrict__ X, int n, int d, Metric metric, int k,
                          float *__restrict__ core, CoreBoxes boxes, int stepLimit,
                          const float *__restrict__ rowsX, int numRows,
                          const int *__restrict__ rowPos, const int *__restrict__ tileList,
                          unsigned int *__restrict__ kthBits, float *__restrict__ partial) {
  constexpr int TR = T::TR, kWaves = T::THREADS / 64, kWaveRows = T::WAVE_ROWS;
  // Pruned: bounds by wave, whose rows are consecutive then.
  constexpr bool kPruned = T::ROWS_BY_WAVE;
  constexpr int kBatch = 64; // walk steps whose box bounds are computed at once
  __shared__ __align__(16) TileSmem<T> sm;
  // Per wave: the bounds of the batch's steps, the steps within its largest
  // k-th distance when the batch began, and that distance now.
  __shared__ float lowerBound[kWaves][kBatch];
  __shared__ unsigned long long within[kWaves];
  __shared__ float largestKth[kWaves];
  // Per row, the smallest k-th distance published by any split.
  __shared__ float sharedKth[T::DIM];
  extern __shared__ float lists[]; // [DIM][k], then the waves' row boxes [kWaves][2 d] if pruning

  const int rowTile = tileList ? tileList[blockIdx.x] : (int)blockIdx.x;
  const int row0 = rowTile * T::DIM;
  const float *A = rowsX ? rowsX : X;
  const int nA = rowsX ? numRows : n;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int splits = gridDim.y, split = blockIdx.y;
  for (int i = threadIdx.x; i < T::DIM * k; i += T::THREADS)
    lists[i] = INFINITY;
  for (int i = threadIdx.x; i < T::DIM; i += T::THREADS)
    sharedKth[i] = splits > 1 && row0 + i < nA ? __uint_as_float(kthBits[row0 + i]) : INFINITY;
  const bool prune = kPruned && boxes.numTiles > 0;
  float *rowBox = lists + T::DIM * k + wave * 2 * d;
  if (prune) {
    const int row = row0 + wave * kWaveRows + (lane & (kWaveRows - 1));
    for (int f = 0; f < d; ++f) {
      const float v = row < nA ? A[(size_t)row * d + f] : 0.0f;
      float lo = row < nA ? v : INFINITY, hi = row < nA ? v : -INFINITY;
#pragma unroll
      for (int m = kWaveRows / 2; m > 0; m >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, m, 64));
        hi = fmaxf(hi, __shfl_xor(hi, m, 64));
      }
      if (lane == 0) {
        rowBox[f] = lo;
        rowBox[d + f] = hi;
      }
    }
  }
  // A wave without rows needs no tile; the others' lists start empty.
  if (lane == 0)
    largestKth[wave] = row0 + wave * kWaveRows < nA ? INFINITY : -1.0f;
  // The 8-feature tiles serve d <= 8 only (one fill): the row slice is
  // staged once for every tile.
  constexpr bool kRowsResident = T::FILL == 8;
  if (kRowsResident)
    stageRows<T>(sm, A, nA, d, row0);
  __syncthreads();
  const float slack = 1.0f - coreBoxSlack(d);
  const int numTiles = (n + T::DIM - 1) / T::DIM;
  const unsigned long long groupMask = 0xffffull << (lane & 48);
  // Listed rows have no home tile: the walk starts anywhere and covers all;
  // with pruning (rows listed in point order) it starts at the column tile of
  // the tile's first row, which is near the others.
  const int homeTile =
      rowsX ? (prune ? rowPos[row0] / T::DIM : (int)(blockIdx.x % numTiles)) : rowTile;

  // A wave leaves out a step when the box bound between its rows and the
  // column tile exceeds the largest k-th distance of those rows, and the
  // workgroup skips it when every wave does. Every wave computes its bounds of
  // 64 steps at once; only the steps some wave still had within reach when
  // the batch began are looked at again.
  const int steps = min(2 * ((numTiles + splits - 1) / splits) + 1, stepLimit);
  int computed = 0; // tiles, of the workgroup
  for (int base = 0; base < steps; base += kBatch) {
    unsigned long long todo;
    {
      const int step = base + lane;
      const int colTile = step < steps ? walkTileCore(homeTile, step, numTiles, splits, split) : -1;
      float lb = 0.0f;
      if (prune && colTile >= 0)
        lb = coreBoxBound(metric, rowBox, rowBox + d, boxes.low + (size_t)colTile * d,
                          boxes.high + (size_t)colTile * d, d) * slack;
      todo = __ballot(colTile >= 0 && !(prune && lb > largestKth[wave]));
      if (prune) {
        lowerBound[wave][lane] = lb;
        if (lane == 0)
          within[wave] = todo;
        __syncthreads();
        todo = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w)
          todo |= within[w];
      }
    }
    for (; todo; todo &= todo - 1) {
      const int j = __ffsll((long long)todo) - 1;
      // Uniform: written before the barrier after the last computed tile.
      bool active = true;
      if (prune) {
        bool any = false;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          const bool reach = !(lowerBound[w][j] > largestKth[w]);
          any |= reach;
          if (w == wave)
            active = reach;
        }
        if (!any)
          continue;
      }
      const int col0 = walkTileCore(homeTile, base + j, numTiles, splits, split) * T::DIM;
      // With an accumulator bound the tile holds raw accumulators, and only the
      // pairs within the bound of the row's current k-th distance are finished
      // (most pairs of a tile are not, which skips their sqrt).
      constexpr bool kFilter = Metric::kAccFilter;
      float v[TR][TR];
      computeTile<T, Metric, !kFilter, kRowsResident, kPruned>(sm, A, nA, X, n, d, metric, row0,
                                                               col0, v, NoExtraStage{}, active);
      if (active) {
        unsigned long long changed = 0;
#pragma unroll
        for (int r = 0; r < TR; ++r) {
          int rit = T::rowInTile(r);
          asm volatile("" : "+v"(rit)); // computed here, not kept for every row
          const int row = row0 + rit;
          float *list = lists + rit * k;
          unsigned int pending = 0;
          if (row < nA) {
            const float kth = fminf(list[k - 1], sharedKth[rit]);
            const int self = rowsX ? rowPos[row] : row;
            if constexpr (kFilter) {
              const float limit = metric.accBound(kth);
#pragma unroll
              for (int c = 0; c < TR; ++c) {
                const int col = col0 + T::colInTile(c);
                const float acc = v[r][c];
                if (col < n && !(acc > limit)) {
                  const float value = col == self ? 0.0f : fmaxf(metric.finish(acc), 0.0f);
                  v[r][c] = value;
                  if (value < kth)
                    pending |= 1u << c;
                }
              }
            } else {
#pragma unroll
              for (int c = 0; c < TR; ++c) {
                const int col = col0 + T::colInTile(c);
                // The point itself is distance 0 (drops float noise such as cosine's 1e-7).
                v[r][c] = col == self ? 0.0f : fmaxf(v[r][c], 0.0f);
                if (col < n && v[r][c] < kth)
                  pending |= 1u << c;
              }
            }
          }
          // One insertion per row per step until no lane of the wave has work;
          // all lanes stay converged for the ballot. The row's lowest lane with
          // work gives its value, the row's 16 lanes insert it, and every lane
          // drops the values that no longer beat the k-th.
          while (true) {
            const unsigned long long work = __ballot(pending != 0);
            if (work == 0)
              break;
            changed |= work;
            const unsigned long long mine = work & groupMask;
            const int source = mine ? __ffsll((long long)mine) - 1 : lane;
            float value = 0.0f;
            const int first = __ffs(pending) - 1;
#pragma unroll
            for (int cc = 0; cc < TR; ++cc)
              if (cc == first)
                value = v[r][cc];
            value = __shfl(value, source, 64);
            if (lane == source)
              pending &= pending - 1;
            if (mine)
              insertSorted(list, k, lane & 15, value);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (pending) {
              const float kth = list[k - 1];
#pragma unroll
              for (int c = 0; c < TR; ++c)
                if (!(v[r][c] < kth))
                  pending &= ~(1u << c);
            }
          }
        }
        // The wave's rows are its own: it refreshes their largest k-th itself.
        const bool share = splits > 1 && (computed & 3) == 0;
        if (prune && (changed || share)) {
          const int i = wave * kWaveRows + (lane & (kWaveRows - 1));
          float largest = -1.0f;
          if (row0 + i < nA) {
            largest = fminf(lists[i * k + k - 1], sharedKth[i]);
            if (share && lane < kWaveRows) {
              const unsigned int bits = __hip_atomic_load(&kthBits[row0 + i], __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT);
              if (__float_as_uint(largest) < bits)
                atomicMin(&kthBits[row0 + i], __float_as_uint(largest));
              else
                largest = __uint_as_float(bits);
              sharedKth[i] = largest;
            }
          }
#pragma unroll
          for (int m = kWaveRows / 2; m > 0; m >>= 1)
            largest = fmaxf(largest, __shfl_xor(largest, m, 64));
          if (lane == 0)
            largestKth[wave] = largest;
        }
      }
      ++computed;
      __syncthreads(); // the tile is consumed, the largest k-th distances are current
    }
    if (prune)
      __syncthreads(); // lowerBound is rewritten by the next batch
  }
  __syncthreads();
  if (splits > 1) {
    const size_t first = ((size_t)split * n + row0) * k;
    for (int e = threadIdx.x; e < T::DIM * k; e += T::THREADS)
      if (row0 + e / k < nA)
        partial[first + e] = lists[e];
    return;
  }
  for (int i = threadIdx.x; i < T::DIM; i += T::THREADS)
    if (row0 + i < nA)
      core[rowsX ? rowPos[row0 + i] : row0 + i] = lists[i * k + k - 1];
}

constexpr int kMostCoreSplits = 8;

// The k-th smallest value of a row's ascending lists (one per split, +inf
// padded), by a thread per row, or the row's last bound: the lists hold every
// value below it that can be among the k smallest, but not those equal to it.
__global__ void __launch_bounds__(256)
    kthOfListsKernel(const float *__restrict__ partial, int splits, int n, int k,
                     const unsigned int *__restrict__ kthBits, float *__restrict__ core) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n)
    return;
  const size_t stride = (size_t)n * k;
  const float *list = partial + (size_t)p * k;
  float head[kMostCoreSplits];
  int at[kMostCoreSplits];
#pragma unroll
  for (int s = 0; s < kMostCoreSplits; ++s) {
    at[s] = 0;
    head[s] = s < splits ? list[s * stride] : INFINITY;
  }
  float kth = INFINITY;
  for (int q = 0; q < k; ++q) {
    kth = head[0];
#pragma unroll
    for (int s = 1; s < kMostCoreSplits; ++s)
      kth = fminf(kth, head[s]);
    bool taken = false;
#pragma unroll
    for (int s = 0; s < kMostCoreSplits; ++s)
      if (!taken && s < splits && head[s] == kth) {
        taken = true;
        ++at[s];
        head[s] = at[s] < k ? list[s * stride + at[s]] : INFINITY;
      }
  }
  core[p] = fminf(kth, __uint_as_float(kthBits[p]));
}

__global__ void coreBoxesKernel(const float *__restrict__ X, int n, int d, int tileDim,
                                float *low, float *high) {
  const int tile = blockIdx.x;
  const int first = tile * tileDim, last = min(n, first + tileDim);
  for (int f = threadIdx.x; f < d; f += blockDim.x) {
    float lo = INFINITY, hi = -INFINITY;
    for (int p = first; p < last; ++p) {
      const float v = X[(size_t)p * d + f];
      lo = fminf(lo, v);
      hi = fmaxf(hi, v);
    }
    low[(size_t)tile * d + f] = lo;
    high[(size_t)tile * d + f] = hi;
  }
}

// One workgroup (256 threads) per row of the distance block. The block's row r
// is point rowList[firstRow + r] (or firstRow + r without a list); its core
// distance goes to core[that point].
__global__ void __launch_bounds__(256)
    kthSmallestRowKernel(const float *__restrict__ dist, int numCols, int firstRow, int k,
                         const int *__restrict__ rowList, float *__restrict__ core) {
  __shared__ unsigned int hist[4][256];
  __shared__ unsigned int prefix, prefixMask, remaining;
  const int row = blockIdx.x;
  const int self = rowList ? rowList[firstRow + row] : firstRow + row;
  const float *rd = dist + (size_t)row * numCols;
  const int wave = threadIdx.x >> 6;
  if (threadIdx.x == 0) {
    prefix = 0;
    prefixMask = 0;
    remaining = (unsigned)k;
  }
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int i = threadIdx.x; i < 4 * 256; i += 256)
      (&hist[0][0])[i] = 0;
    __syncthreads();
    const unsigned int pre = prefix, mask = prefixMask;
    for (int col = threadIdx.x; col < numCols; col += 256) {
      const float value = col == self ? 0.0f : fmaxf(rd[col], 0.0f);
      const unsigned int bits = __float_as_uint(value);
      if ((bits & mask) == pre)
        atomicAdd(&hist[wave][(bits >> shift) & 0xffu], 1u);
    }
    __syncthreads();
    // The first bin that reaches `remaining`: one wave, four bins per lane (one
    // thread stepping through the bins took 14 us per digit).
    if (wave == 0) {
      const int lane = threadIdx.x;
      unsigned int count[4], sum = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int bin = 4 * lane + q;
        count[q] = hist[0][bin] + hist[1][bin] + hist[2][bin] + hist[3][bin];
        sum += count[q];
      }
      unsigned int upTo = sum;
#pragma unroll
      for (int m = 1; m < 64; m <<= 1) {
        const unsigned int up = __shfl_up(upTo, m, 64);
        if (lane >= m)
          upTo += up;
      }
      const unsigned long long reached = __ballot(upTo >= remaining);
      // Every value is finite: some bin reaches it.
      const int first = reached ? __ffsll((long long)reached) - 1 : 63;
      if (lane == first) {
        unsigned int below = upTo - sum;
        int q = 0;
#pragma unroll
        for (int b = 0; b < 3; ++b)
          if (q == b && below + count[b] < remaining) {
            below += count[b];
            ++q;
          }
        remaining -= below;
        prefix |= (unsigned int)(4 * lane + q) << shift;
        prefixMask |= 0xffu << shift;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0)
    core[self] = __uint_as_float(prefix);
}

template <class F> int withMetricCore(MetricSpec m, F &&f) {
  switch (m.id) {
  case kEuclidean: return f(Euclidean{});
  case kSqEuclidean: return f(SqEuclidean{});
  case kManhattan: return f(Manhattan{});
  case kChebyshev: return f(Chebyshev{});
  case kMinkowski: return f(Minkowski{m.p});
  case kCosine: return f(Cosine{});
  default: return kErrInvalidMetric;
  }
}

// run(fill, pruned) for the features staged per fill, and for tiles with rows by
// wave where the pass prunes. Without, every tile is computed, and rows by wave
// and barriers left to the caller take longer (30,000 points, k = 8, 300 features
// 59.1 ms, now 55.0; 784 129 and 120).
template <class Metric, class F> int withTile(int d, bool prune, F &&run) {
  using Eight = std::integral_constant<int, 8>;
  using Fill = std::integral_constant<int, 32>;
  if constexpr (Metric::kBoxBound)
    if (prune)
      return d <= 8 ? run(Eight{}, std::true_type{}) : run(Fill{}, std::true_type{});
  return d <= 8 ? run(Eight{}, std::false_type{}) : run(Fill{}, std::false_type{});
}

// The tiles by the size of their boxes (squared diagonal, to 7 bits of
// mantissa), largest first.
__global__ void boxSizeKeysKernel(CoreBoxes boxes, int d, unsigned int *__restrict__ keys,
                                  int *__restrict__ tiles) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= boxes.numTiles)
    return;
  float sq = 0.0f;
  for (int f = 0; f < d; ++f) {
    const float side = boxes.high[(size_t)t * d + f] - boxes.low[(size_t)t * d + f];
    sq = fmaf(side, side, sq);
  }
  keys[t] = 0x7fffu - (__float_as_uint(sq) >> 16);
  tiles[t] = t;
}

int sparseFirst(const CoreBoxes &boxes, int tiles, int d, DevArray<int> &order) {
  DevArray<unsigned int> keys, sorted;
  DevArray<int> from;
  DevArray<unsigned char> temp;
  Status s;
  s(keys.alloc(tiles));
  s(sorted.alloc(tiles));
  s(from.alloc(tiles));
  s(order.alloc(tiles));
  s(temp.alloc(sortTempBytes32(tiles)));
  if (!s.ok())
    return s.code;
  hipLaunchKernelGGL(boxSizeKeysKernel, dim3((tiles + 255) / 256), dim3(256), 0, stream(), boxes, d,
                     keys.get(), from.get());
  s((int)hipGetLastError());
  s(radixSortPairs(keys, sorted, from, order, tiles, 15, temp));
  return s.code;
}

// tileList (device, numListed entries): only those row tiles.
int coreFused(const float *X, int n, int d, MetricSpec m, int k, float *core, bool prune,
              int stepLimit = 0x7fffffff, const int *tileList = nullptr, int numListed = 0) {
  return withMetricCore(m, [&](auto metric) {
    using Metric = decltype(metric);
    auto run = [&](auto fill, auto pruned) {
      using T = typename TileFor<Metric, decltype(fill)::value, decltype(pruned)::value>::type;
      const int tiles = (n + T::DIM - 1) / T::DIM;
      size_t smem = (size_t)T::DIM * k * sizeof(float);
      CoreBoxes boxes;
      DevArray<float> low, high;
      Status s;
      if (decltype(pruned)::value) {
        s(low.alloc((size_t)tiles * d));
        s(high.alloc((size_t)tiles * d));
        if (!s.ok())
          return s.code;
        hipLaunchKernelGGL(coreBoxesKernel, dim3(tiles), dim3(64), 0, stream(), X, n, d, T::DIM,
                           low.get(), high.get());
        boxes = CoreBoxes{low, high, tiles};
        smem += (T::THREADS / 64) * 2 * d * sizeof(float);
      }
      // Splits: enough workgroups to even out walks of very different lengths
      // (a resident chip's worth several times over), each with eight column
      // tiles at least. Without the memory for their lists (at most 130 MiB),
      // one.
      int splits = 1;
      DevArray<unsigned int> kthBits;
      DevArray<float> partial;
      DevArray<int> order;
      const bool whole = boxes.numTiles > 0 && !tileList && stepLimit >= 2 * tiles;
      if (whole) {
        splits = std::max(1, std::min({16 * numCUs() / tiles, tiles / 8, kMostCoreSplits}));
        if (splits > 1 && (kthBits.alloc(n) || partial.alloc((size_t)splits * n * k))) {
          (void)hipGetLastError();
          splits = 1;
        }
        s(sparseFirst(boxes, tiles, d, order));
        tileList = order;
      }
      if (!s.ok())
        return s.code;
      PhaseTimer timer(kPhaseCore);
      if (splits > 1)
        hipLaunchKernelGGL((kthNearestFusedKernel<T, Metric>), dim3(tiles), dim3(256), smem,
                           stream(), X, n, d, metric, k, reinterpret_cast<float *>(kthBits.get()),
                           CoreBoxes{}, 1, nullptr, 0, nullptr, nullptr, nullptr, nullptr);
      hipLaunchKernelGGL((kthNearestFusedKernel<T, Metric>),
                         dim3(numListed ? numListed : tiles, splits), dim3(256), smem, stream(), X,
                         n, d, metric, k, core, boxes, stepLimit, nullptr, 0, nullptr, tileList,
                         kthBits.get(), partial.get());
      if (splits > 1)
        hipLaunchKernelGGL(kthOfListsKernel, dim3((n + 255) / 256), dim3(256), 0, stream(),
                           partial.get(), splits, n, k, kthBits.get(), core);
      s((int)hipGetLastError());
      s(sync());
      return s.code;
    };
    return withTile<Metric>(d, prune, run);
  });
}

// Distance rows per radix-select launch: a quarter of the free device memory
// (at most 64 GiB; at n = 10^6 that is 16,384 rows of 4 MB, so one launch
// fills the chip many times over), at least one row, a multiple of the tile
// rows when possible, never more than wanted.
int radixChunkRows(int n, int wanted, int tileRows) {
  if ((size_t)n * wanted <= ((size_t)64 << 20))
    return wanted; // 256 MiB at most: not worth asking
  size_t freeBytes = 0, totalBytes = 0;
  if (hipMemGetInfo(&freeBytes, &totalBytes) != hipSuccess) {
    (void)hipGetLastError();
    freeBytes = (size_t)4 << 30;
  }
  const size_t budget = std::min(freeBytes / 4, (size_t)64 << 30);
  const size_t rowBytes = (size_t)n * sizeof(float);
  size_t rows = std::max<size_t>(1, budget / rowBytes);
  if (rows >= (size_t)tileRows)
    rows = rows / tileRows * tileRows;
  return (int)std::min<size_t>(rows, (size_t)wanted);
}

int coreRadix(const float *X, int n, int d, MetricSpec m, int k, float *core) {
  const int rows = radixChunkRows(n, n, tilePoints(m.id));
  DevArray<float> chunk;
  Status s;
  s(chunk.alloc((size_t)rows * n));
  PhaseTimer timer(kPhaseCore);
  for (int first = 0; s.ok() && first < n; first += rows) {
    const int count = std::min(rows, n - first);
    s(pairwiseMatrix(X + (size_t)first * d, count, X, n, d, m, chunk));
    hipLaunchKernelGGL(kthSmallestRowKernel, dim3(count), dim3(256), 0, stream(), chunk.get(), n,
                       first, k, nullptr, core);
    s((int)hipGetLastError());
  }
  s(sync());
  return s.code;
}

} // namespace

int coreLocal(const float *X, int n, int d, MetricSpec m, int k, int stepLimit, float *out) {
  return coreFused(X, n, d, m, std::min(k, kMaxFusedK), out, false, stepLimit);
}

namespace {

// Exact core distances of listed rows with the fused top-k lists (k <= 64):
// the rows are gathered. Without pruning every column tile is visited; with
// it (points in k-d order, rows listed in ascending position, a box metric)
// each tile of 128 gathered rows gets its own box and skips the column tiles
// whose bound exceeds its largest k-th distance, as the tiles of the points
// themselves do.
int coreForRowsFused(const float *X, int n, int d, MetricSpec m, int k, const int *rows,
                     int numRows, float *core, bool prune) {
  DevArray<float> rowData;
  Status s;
  s(rowData.alloc((size_t)numRows * d));
  if (s.ok())
    s(gatherRows(X, rows, numRows, d, rowData));
  if (!s.ok())
    return s.code;
  return withMetricCore(m, [&](auto metric) {
    using Metric = decltype(metric);
    auto run = [&](auto fill, auto pruned) {
      using T = typename TileFor<Metric, decltype(fill)::value, decltype(pruned)::value>::type;
      const int rowTiles = (numRows + T::DIM - 1) / T::DIM;
      size_t smem = (size_t)T::DIM * k * sizeof(float);
      CoreBoxes boxes;
      DevArray<float> low, high;
      Status st;
      if (decltype(pruned)::value) {
        const int tiles = (n + T::DIM - 1) / T::DIM;
        st(low.alloc((size_t)tiles * d));
        st(high.alloc((size_t)tiles * d));
        if (!st.ok())
          return st.code;
        hipLaunchKernelGGL(coreBoxesKernel, dim3(tiles), dim3(64), 0, stream(), X, n, d, T::DIM,
                           low.get(), high.get());
        boxes = CoreBoxes{low, high, tiles};
        smem += (T::THREADS / 64) * 2 * d * sizeof(float);
      }
      PhaseTimer timer(kPhaseCore);
      hipLaunchKernelGGL((kthNearestFusedKernel<T, Metric>), dim3(rowTiles), dim3(256), smem,
                         stream(), X, n, d, metric, k, core, boxes, 0x7fffffff,
                         rowData.get(), numRows, rows, nullptr, nullptr, nullptr);
      st((int)hipGetLastError());
      st(sync());
      return st.code;
    };
    return withTile<Metric>(d, prune, run);
  });
}

} // namespace

int coreForRows(const float *X, int n, int d, MetricSpec m, int k, const int *rows, int numRows,
                float *core, bool prune) {
  if (numRows <= 0)
    return 0;
  if (k <= kMaxFusedK)
    return coreForRowsFused(X, n, d, m, k, rows, numRows, core, prune);
  const int chunkRows = radixChunkRows(n, numRows, 1);
  DevArray<float> chunk, rowData;
  Status s;
  s(chunk.alloc((size_t)chunkRows * n));
  s(rowData.alloc((size_t)chunkRows * d));
  for (int first = 0; s.ok() && first < numRows; first += chunkRows) {
    const int count = std::min(chunkRows, numRows - first);
    s(gatherRows(X, rows + first, count, d, rowData));
    s(pairwiseMatrix(rowData, count, X, n, d, m, chunk));
    hipLaunchKernelGGL(kthSmallestRowKernel, dim3(count), dim3(256), 0, stream(), chunk.get(), n,
                       first, k, rows, core);
    s((int)hipGetLastError());
  }
  s(sync());
  return s.code;
}

int coreForTiles(const float *X, int n, int d, MetricSpec m, int k, const int *hostTiles,
                 int numTiles, float *core) {
  constexpr int kDim = 128; // the fused kernel's row tile for box metrics
  if (numTiles <= 0)
    return 0;
  Status s;
  if (k <= kMaxFusedK && metricHasBoxBound(m.id)) {
    DevArray<int> list;
    s(list.alloc(numTiles));
    s(upload(list, hostTiles, numTiles * sizeof(int)));
    if (s.ok())
      s(coreFused(X, n, d, m, k, core, true, 0x7fffffff, list, numTiles));
    return s.code;
  }
  std::vector<int> rows;
  for (int t = 0; t < numTiles; ++t)
    for (int p = hostTiles[t] * kDim; p < std::min(n, (hostTiles[t] + 1) * kDim); ++p)
      rows.push_back(p);
  DevArray<int> dRows;
  s(dRows.alloc(rows.size()));
  s(upload(dRows, rows.data(), rows.size() * sizeof(int)));
  if (s.ok())
    s(coreForRows(X, n, d, m, k, dRows, (int)rows.size(), core));
  return s.code;
}

int coreDistances(const float *X, int n, int d, MetricSpec m, int k, float *core, int method,
                  bool prune) {
  if (k < 1 || k > n)
    return kErrInvalidShape;
  if (method == kCoreFused && k > kMaxFusedK)
    return kErrInvalidAlgorithm;
  if (method == kCoreLearned)
    return coreLearned(X, n, d, m, k, core, prune);
  if (method == kCoreFused || (method == kCoreAuto && k <= kMaxFusedK))
    return coreFused(X, n, d, m, k, core, prune);
  const int status = coreRadix(X, n, d, m, k, core);
  if (method == kCoreRadixElseFused && status == (int)hipErrorOutOfMemory) {
    (void)hipGetLastError();
    return coreFused(X, n, d, m, k, core, prune);
  }
  return status;
}

} // namespace cuhc

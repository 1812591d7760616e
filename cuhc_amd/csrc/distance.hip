// All-pairs FP32 kernels: distance matrices (full and condensed), the
// symmetric nearest-other-component pass, and the spatially pruned walk pass.
//
// Reference counterparts: pairwiseDistanceKernel and
// nearestOtherComponentSymmetricKernel (src/distance_matrix.cuh:179-200,
// 287-390), buildTileBoxesKernel / nearestOtherComponentWalkKernel /
// estimatePrunedShare (src/spatial.cuh:136-343, 424-469). The tile fold is
// tile.hpp; argmins carry (weight, index) as one u64 key.
#include "passes.hpp"
#include "primitives.hpp"
#include "tile.hpp"

#include <algorithm>
#include <type_traits>

namespace cuhc {

bool validMetric(int id) { return id >= kEuclidean && id <= kCosine; }
bool metricHasBoxBound(int id) { return validMetric(id) && id != kCosine; }
int tilePoints(int metricId) { return metricId == kCosine ? 64 : 128; }

namespace {

template <class F> int withMetric(MetricSpec m, F &&f) {
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

// LDS staging width: 8 features for d <= 8, else 32 (a fill stages only the
// features present, rounded up to 8).
template <class F> int withFill(int d, F &&f) {
  if (d <= 8)
    return f(std::integral_constant<int, 8>{});
  return f(std::integral_constant<int, 32>{});
}

int persistentBlocks(long long work, int perCU) {
  const long long cap = (long long)numCUs() * perCU;
  return (int)std::max<long long>(1, std::min<long long>(work, cap));
}

// ---------------------------------------------------------------------------
// Distance matrices

template <class T, class Metric>
__global__ void __launch_bounds__(256)
    pairwiseMatrixKernel(const float *__restrict__ A, int nA, const float *__restrict__ B, int nB,
                         int d, Metric metric, float *__restrict__ out, int tilesB) {
  __shared__ __align__(16) TileSmem<T> sm;
  const int tileI = blockIdx.x / tilesB, tileJ = blockIdx.x - tileI * tilesB;
  const int row0 = tileI * T::DIM, col0 = tileJ * T::DIM;
  float v[T::TR][T::TR];
  computeTile<T>(sm, A, nA, B, nB, d, metric, row0, col0, v);
#pragma unroll
  for (int r = 0; r < T::TR; ++r) {
    const int row = row0 + T::rowInTile(r);
    if (row >= nA)
      continue;
#pragma unroll
    for (int c = 0; c < T::TR; ++c) {
      const int col = col0 + T::colInTile(c);
      if (col < nB)
        out[(size_t)row * nB + col] = v[r][c];
    }
  }
}

template <class T, class Metric>
__global__ void __launch_bounds__(256)
    condensedMatrixKernel(const float *__restrict__ X, int n, int d, Metric metric,
                          float *__restrict__ out, long long numPairs) {
  __shared__ __align__(16) TileSmem<T> sm;
  for (long long t = blockIdx.x; t < numPairs; t += gridDim.x) {
    int I, J;
    decodeTrianglePair(t, I, J);
    const int row0 = I * T::DIM, col0 = J * T::DIM;
    float v[T::TR][T::TR];
    computeTile<T>(sm, X, n, X, n, d, metric, row0, col0, v);
#pragma unroll
    for (int r = 0; r < T::TR; ++r) {
      const long long i = row0 + T::rowInTile(r);
      if (i >= n)
        continue;
      const long long base = i * n - i * (i + 1) / 2 - i - 1;
#pragma unroll
      for (int c = 0; c < T::TR; ++c) {
        const long long j = col0 + T::colInTile(c);
        if (j > i && j < n)
          out[base + j] = v[r][c];
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Symmetric nearest-other-component pass

// Reduces a key over the 16 lanes of a tile row (xor 8, 4, 2, 1).
DEV unsigned long long rowGroupMin(unsigned long long k) {
#pragma unroll
  for (int m = 8; m > 0; m >>= 1)
    k = minKey(k, shflXorKey(k, m));
  return k;
}

// Pair filter of the symmetric pass. A point's limit comes from the weight of
// its current nearest (+inf while it has none; the key's high word, read
// alone: nearest only decreases, so a stale read is a looser limit). With a
// metric that has an accumulator bound, a pair passes when its raw accumulator
// is within the larger of its two points' limits, accBound(distBound(w)); every
// pair whose weight is within a point's nearest weight passes.
template <class Metric, class Weight> struct PairFilter {
  static constexpr bool kOn = Metric::kAccFilter && Weight::kDistBound;
  DEV static float limit(const Metric &metric, const Weight &weight,
                         const unsigned long long *nearest, int p) {
    return limitOf(metric, weight,
                   reinterpret_cast<const unsigned int *>(nearest)[2 * (size_t)p + 1]);
  }
  DEV static float limitOf(const Metric &metric, const Weight &weight, unsigned int bits) {
    if (bits == 0xffffffffu)
      return INFINITY;
    const float w = floatOf(bits);
    return metric.accBound(weight.distBound(w));
  }
};

// Row and column data of a symmetric tile staged in LDS with the tile's first
// fill: threads [0, DIM) load column col0 + t, threads [DIM, 2 DIM) row
// row0 + t - DIM (component, weight value, original index and, when
// filtering, the weight bits of the current nearest, turned into a limit).
// Points past n get component -1 (columns) or -2 (rows) and limit -inf.
template <class Metric, class Weight, bool kFilter> struct PairStage {
  using WV = typename Weight::Value;
  struct Value {
    int comp;
    WV val;
    unsigned int id, bits;
  };
  const int *comp;
  const int *orig;
  const unsigned long long *nearest;
  Metric metric;
  Weight weight;
  int row0, col0, n, dim;
  int *sComp;      // [2 dim]: columns, then rows
  WV *sVal;        // [2 dim]
  unsigned *sId;   // [2 dim]
  float *sLimit;   // [2 dim]
  DEV int point() const {
    const int t = (int)threadIdx.x;
    return t < dim ? col0 + t : row0 + (t - dim);
  }
  DEV Value load() const {
    Value v{};
    if ((int)threadIdx.x < 2 * dim) {
      const int pl = min(point(), n - 1);
      v.comp = comp[pl];
      v.val = weight.value(pl);
      v.id = orig ? (unsigned)orig[pl] : (unsigned)pl;
      if (kFilter)
        v.bits = reinterpret_cast<const unsigned int *>(nearest)[2 * (size_t)pl + 1];
    }
    return v;
  }
  DEV void store(const Value &v) const {
    const int t = (int)threadIdx.x;
    if (t < 2 * dim) {
      const int p = point();
      const bool ok = p < n;
      sComp[t] = ok ? v.comp : (t < dim ? -1 : -2);
      sVal[t] = v.val;
      sId[t] = ok ? v.id : (unsigned)p;
      if (kFilter)
        sLimit[t] = ok ? PairFilter<Metric, Weight>::limitOf(metric, weight, v.bits) : -INFINITY;
    }
  }
};

template <class T, class Metric, class Weight>
__global__ void __launch_bounds__(256, 3) // three waves per SIMD (at most 168 VGPRs)
    nearestOtherSymmetricKernel(const float *__restrict__ X, int n, int d, Metric metric,
                                Weight weight, const int *__restrict__ comp,
                                const int *__restrict__ orig,
                                unsigned long long *__restrict__ nearest, long long numPairs,
                                const int *__restrict__ numComp) {
  if (numComp && *numComp <= 1)
    return; // queued ahead of the host: one component is left
  constexpr int TR = T::TR;
  // With an accumulator bound, a pair is finished (sqrt, weight, keys) only
  // when its raw accumulator is within the limit of its row point or of its
  // column point (from their current nearest) and it crosses components.
  // Every point's nearest pair is within its own limit, so every point's
  // result stays exact.
  using Filter = PairFilter<Metric, Weight>;
  constexpr bool kFilter = Filter::kOn;
  __shared__ __align__(16) TileSmem<T> sm;
  __shared__ unsigned long long colBest[T::DIM];
  // Point data of the tile: columns [0, DIM), rows [DIM, 2 DIM).
  __shared__ int sComp[2 * T::DIM];
  __shared__ typename Weight::Value sVal[2 * T::DIM];
  __shared__ unsigned int sId[2 * T::DIM];
  __shared__ float sLimit[2 * T::DIM];
  static_assert(2 * T::DIM <= T::THREADS, "one point per thread");

  for (long long t = blockIdx.x; t < numPairs; t += gridDim.x) {
    int I, J;
    decodeTrianglePair(t, I, J);
    const int row0 = I * T::DIM, col0 = J * T::DIM;
    for (int i = threadIdx.x; i < T::DIM; i += T::THREADS)
      colBest[i] = kEmptyKey; // visible after computeTile's barriers

    float w[TR][TR]; // raw accumulators when filtering
    // The point data arrives with the tile's first fill (read after
    // computeTile's barriers; rewritten only after this tile's last barrier).
    const PairStage<Metric, Weight, kFilter> stage{comp, orig, nearest, metric, weight, row0,
                                                   col0, n, T::DIM, sComp, sVal, sId, sLimit};
    computeTile<T, Metric, !kFilter>(sm, X, n, X, n, d, metric, row0, col0, w, stage);

    int colComp[TR];
    unsigned int colId[TR];
    typename Weight::Value colVal[TR];
#pragma unroll
    for (int c = 0; c < TR; ++c) {
      const int i = T::colInTile(c);
      colComp[c] = sComp[i];
      colVal[c] = sVal[i];
      colId[c] = sId[i];
    }
    // A pair counts if both points exist, lie in different components and
    // have a finite weight (+inf never counts, as in the reference's
    // symmetric pass; NaN counts and packs as 0).
    unsigned long long rowKey[TR];
    unsigned long long countMask = 0;
    float colLimit[TR];
    if constexpr (kFilter) {
#pragma unroll
      for (int c = 0; c < TR; ++c)
        colLimit[c] = sLimit[T::colInTile(c)];
    }
#pragma unroll
    for (int r = 0; r < TR; ++r) {
      const int ri = T::DIM + T::rowInTile(r);
      const int rc = sComp[ri];
      const typename Weight::Value rv = sVal[ri];
      unsigned long long best = kEmptyKey;
      if constexpr (kFilter) {
        const float rowLimit = sLimit[ri];
#pragma unroll
        for (int c = 0; c < TR; ++c) {
          const float acc = w[r][c];
          if (!(acc > fmaxf(rowLimit, colLimit[c])) &&
              colComp[c] != rc) {
            const float ww = weight(metric.finish(acc), rv, colVal[c]);
            w[r][c] = ww;
            if (colComp[c] >= 0 && rc >= 0 && ww != INFINITY) {
              countMask |= 1ull << (r * TR + c);
              best = minKey(best, packKey(ww, colId[c]));
            }
          }
        }
      } else {
#pragma unroll
        for (int c = 0; c < TR; ++c) {
          const float ww = weight(w[r][c], rv, colVal[c]);
          const bool counts = colComp[c] >= 0 && rc >= 0 && colComp[c] != rc && ww != INFINITY;
          w[r][c] = ww;
          if (counts) {
            countMask |= 1ull << (r * TR + c);
            best = minKey(best, packKey(ww, colId[c]));
          }
        }
      }
      // Wave-uniform: skip the reduction when no lane has a candidate.
      rowKey[r] = __ballot(best != kEmptyKey) != 0 ? rowGroupMin(best) : kEmptyKey;
    }
    if (T::tc() == 0) {
#pragma unroll
      for (int r = 0; r < TR; ++r) {
        const int row = row0 + T::rowInTile(r);
        if (row < n && rowKey[r] != kEmptyKey)
          atomicMin(&nearest[row], rowKey[r]);
      }
    }
    if (I != J) {
      // Columns: this thread's rows, then lanes tc+16, +32, +48 of the wave,
      // then the 4 waves through LDS (skipped by a wave with no counted pair).
      if (__ballot(countMask != 0) != 0) {
        unsigned int rowId[TR];
#pragma unroll
        for (int r = 0; r < TR; ++r)
          rowId[r] = sId[T::DIM + T::rowInTile(r)];
#pragma unroll
        for (int c = 0; c < TR; ++c) {
          unsigned long long best = kEmptyKey;
#pragma unroll
          for (int r = 0; r < TR; ++r)
            if (countMask & (1ull << (r * TR + c)))
              best = minKey(best, packKey(w[r][c], rowId[r]));
          best = minKey(best, shflXorKey(best, 16));
          best = minKey(best, shflXorKey(best, 32));
          if ((threadIdx.x & 63) < 16 && best != kEmptyKey)
            atomicMin(&colBest[T::colInTile(c)], best);
        }
      }
      __syncthreads();
      for (int i = threadIdx.x; i < T::DIM; i += T::THREADS) {
        const int col = col0 + i;
        if (col < n && colBest[i] != kEmptyKey)
          atomicMin(&nearest[col], colBest[i]);
      }
    }
    __syncthreads(); // colBest reused by the next tile
  }
}

// ---------------------------------------------------------------------------
// Spatial pruning: boxes and the walk pass

struct Boxes {
  float *low = nullptr, *high = nullptr; // tiles x d
  float *minValue = nullptr;             // smallest per-point weight value in the tile
  int *minComp = nullptr, *maxComp = nullptr;
  int numTiles = 0;
};

// Boxes of the tiles of X (n points of d features, tileDim per tile).
template <class Weight>
__global__ void buildBoxesKernel(const float *__restrict__ X, int n, int d, int tileDim,
                                 Weight weight, const int *__restrict__ comp, Boxes boxes) {
  const int tile = blockIdx.x;
  const int first = tile * tileDim, last = min(n, first + tileDim);
  for (int f = threadIdx.x; f < d; f += blockDim.x) {
    float lo = INFINITY, hi = -INFINITY;
    for (int p = first; p < last; ++p) {
      const float v = X[(size_t)p * d + f];
      lo = fminf(lo, v);
      hi = fmaxf(hi, v);
    }
    boxes.low[(size_t)tile * d + f] = lo;
    boxes.high[(size_t)tile * d + f] = hi;
  }
  // Per-point values and component range: a wave-wide min/max.
  if (threadIdx.x < 64) {
    float mv = INFINITY;
    int cmin = 0x7fffffff, cmax = -1;
    for (int p = first + (int)threadIdx.x; p < last; p += 64) {
      mv = fminf(mv, (float)weight.value(p));
      const int c = comp ? comp[p] : 0;
      cmin = min(cmin, c);
      cmax = max(cmax, c);
    }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) {
      mv = fminf(mv, __shfl_xor(mv, m, 64));
      cmin = min(cmin, __shfl_xor(cmin, m, 64));
      cmax = max(cmax, __shfl_xor(cmax, m, 64));
    }
    if (threadIdx.x == 0) {
      boxes.minValue[tile] = Weight::kHasValue ? mv : 0.0f;
      boxes.minComp[tile] = cmin;
      boxes.maxComp[tile] = cmax;
    }
  }
}

// Relative slack of the box bound (reference src/spatial.cuh:183-185): far
// larger than the rounding of a pair's distance or of the bound, far too
// small to cost pruning.
HD float boxSlack(int d) { return 1e-5f + (d + 8) * 5e-7f; }

template <class Metric>
DEV float boxLowerBound(const Metric &metric, const float *lowA, const float *highA,
                        const float *lowB, const float *highB, int d) {
  typename Metric::Acc acc = metric.init();
  for (int k = 0; k < d; ++k) {
    const float gap = fmaxf(0.0f, fmaxf(lowB[k] - highA[k], lowA[k] - highB[k]));
    acc = metric.fold(acc, gap, 0.0f);
  }
  return metric.finish(acc);
}

// Column tile visited at `step` from row tile I: I, I+1, I-1, I+2, ... (-1 if
// outside). Of a walk in splits, split s takes I itself and every splits-th
// pair after it.
DEV int walkTile(int rowTile, int step, int numTiles, int splits = 1, int split = 0) {
  const int pair = (step + 1) >> 1;
  const int off = pair == 0 ? 0 : (pair - 1) * splits + split + 1;
  const int tile = (step & 1) ? rowTile + off : rowTile - off;
  return (tile >= 0 && tile < numTiles) ? tile : -1;
}

// Column data of a walk tile staged in LDS with the tile's first fill:
// thread t < DIM loads column col0 + t's component, weight value and
// original index (from a clamped index; -1 marks columns past n).
template <class Weight> struct ColumnStage {
  using WV = typename Weight::Value;
  struct Value {
    int comp;
    WV val;
    unsigned int idx;
  };
  const int *comp;
  const int *orig;
  Weight weight;
  int col0, n, dim;
  int *sComp;
  WV *sVal;
  unsigned int *sIdx;
  DEV Value load() const {
    Value v{};
    if ((int)threadIdx.x < dim) {
      const int col = col0 + (int)threadIdx.x;
      const int cl = min(col, n - 1);
      v.comp = comp[cl];
      v.val = weight.value(cl);
      v.idx = orig ? (unsigned)orig[cl] : (unsigned)cl; // null: keys carry positions
    }
    return v;
  }
  DEV void store(const Value &v) const {
    if ((int)threadIdx.x < dim) {
      const bool ok = col0 + (int)threadIdx.x < n;
      sComp[threadIdx.x] = ok ? v.comp : -1;
      sVal[threadIdx.x] = v.val;
      sIdx[threadIdx.x] = v.idx;
    }
  }
};

// One workgroup per row tile walks the column tiles outward from its own
// (walkTile order). Each wave owns 32 consecutive rows and computes the lower
// bounds of the weight between their box and the column tiles' boxes 64 steps
// at a time, one step per lane; it leaves out a step whose bound exceeds every
// one of its rows' need, and the workgroup skips the step when all waves do. A
// row needs candidates below min(its current best, its component's best known
// edge): Boruvka only uses each component's smallest outgoing edge, so once any
// point of the component has found an edge of weight b, no row of that
// component needs a candidate above b (compBest, shared by all workgroups
// through atomicMin on the weight bits; null disables it). The row that holds
// the component's smallest edge always finds it exactly; other rows may stop
// early, and their results are then only upper bounds, which the contraction
// never prefers. The same need filters single pairs: every row's is published
// in LDS, and for metrics with an accumulator bound a pair is finished (sqrt,
// weight, key) only when its raw accumulator is within the row's need and it
// crosses components; the pairs filtered out weigh more than the need.
// A row belongs to one wave, so its best, need and list change without a
// barrier; the tile needs two (its data staged; consumed, with the waves' bounds
// current, on which all waves decide the next step alike).
// Bound by FP32 VALU work at large n, by the longest row tile's walk where all
// row tiles are resident at once. One box and one bound per 128-row tile
// computed nearly twice the pairs (47% of all pairs of 100,000 points of 8
// features against 26% by 32 rows). HDBSCAN's passes over 10^6 points of 8
// features took 290 ms; by wave 235, and with the sparse tiles first 202.
// With few row tiles a walk is split over gridDim.y workgroups, which share a
// row's best through nearest[] (kept lists are merged afterwards, one per
// split): the four passes over 100,000 points took 18.1 ms, and take 5.9.

// The rows of a compact walk: n rows gathered into X (d features each) from
// positions pos[0 .. n) of the full order (ascending); center[t] is the
// full-order tile around which row tile t walks.
struct RowSet {
  const float *X = nullptr;
  int n = 0;
  const int *pos = nullptr;
  const int *center = nullptr;
};

// KEEP: every row keeps its kKeptKeys smallest keys over all other
// components, written to kept[position][0 ..] (ascending, kEmptyKey padded),
// and its need is the last of them, so that later rounds can settle the row
// from the list (compBest must be null: a component's best would cut the
// search at the row's first key).
constexpr int kKeptKeys = 4;

// The keeping walk runs the first round only; three waves per SIMD hide its
// waits better than two (C3's four Borůvka walks: 298 ms with two waves, 265 ms
// with three).
template <class T, class Metric, class Weight, bool COMPACT = false, bool KEEP = false>
__global__ void __launch_bounds__(256, (!KEEP ? 1 : T::FILL == 8 ? 3 : 2))
    nearestOtherWalkKernel(const float *__restrict__ X, int n, int d, Metric metric,
                           Weight weight, const int *__restrict__ comp,
                           const int *__restrict__ orig, Boxes boxes,
                           unsigned int *__restrict__ compBest,
                           unsigned long long *__restrict__ nearest,
                           unsigned long long *wavesComputed, int rowTileStride,
                           int computeSteps, const int *__restrict__ skipComp,
                           const unsigned char *__restrict__ closedRows, RowSet rows,
                           unsigned long long *__restrict__ kept) {
  constexpr int TR = T::TR, kWaves = T::THREADS / 64, kWaveRows = T::WAVE_ROWS;
  constexpr int kBatch = 64;
  static_assert(TR == 8 && kWaveRows == 32 && T::ROWS_BY_WAVE, "a wave's rows are its lower 32 lanes");
  __shared__ unsigned long long rowTop[KEEP ? T::DIM * kKeptKeys : 1];
  // Rows: the full order's tiles, or (COMPACT) the gathered rows, whose
  // position in the full order indexes comp, the weight values, closedRows
  // and nearest.
  const float *__restrict__ rowX = COMPACT ? rows.X : X;
  const int nRows = COMPACT ? rows.n : n;
  auto posOf = [&](int row) { return COMPACT ? rows.pos[row] : row; };
  __shared__ __align__(16) TileSmem<T> sm;
  __shared__ unsigned long long rowBest[T::DIM];
  __shared__ float rowNeed[T::DIM]; // -1: no row
  // Per wave: the batch's bounds, the steps within its reach when the batch
  // began, and its largest need now (-1: no open row).
  __shared__ float lowerBound[kWaves][kBatch];
  __shared__ unsigned long long within[kWaves];
  __shared__ float bound[kWaves];
  __shared__ int sColComp[T::DIM];
  __shared__ typename Weight::Value sColVal[T::DIM];
  __shared__ unsigned int sColIdx[T::DIM];
  extern __shared__ float rowBoxes[]; // per wave low[d], high[d]
  constexpr bool kFilter = Metric::kAccFilter && Weight::kDistBound;

  // Last tiles first: in the order by core distance they hold the sparse points,
  // whose walks are the longest.
  const int rowTile = (int)(gridDim.x - 1 - blockIdx.x) * rowTileStride;
  const int numTiles = boxes.numTiles;
  const int row0 = rowTile * T::DIM;
  const int center = COMPACT ? rows.center[rowTile] : rowTile;
  const int splits = gridDim.y, split = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // A row is open unless it lies past the end, in the skipped component, or
  // is closed (its exact answer is already in nearest[]).
  const int skip = skipComp ? *skipComp : -1;
  auto isOpen = [&](int row) {
    if (row >= nRows)
      return false;
    const int p = posOf(row);
    return comp[p] != skip && !(closedRows && closedRows[p]);
  };
  // Lanes 0..31 own the wave's rows: whether open, component, and the
  // component's best known edge (refreshed once per batch).
  const int own = wave * kWaveRows + (lane & (kWaveRows - 1)), ownRow = row0 + own;
  const bool open = lane < kWaveRows && isOpen(ownRow);
  const int ownComp = open ? comp[posOf(ownRow)] : 0;
  float cap = INFINITY;
  if (!__syncthreads_or(open))
    return; // uniform: every row of the tile is settled
  if (KEEP)
    for (int i = threadIdx.x; i < T::DIM * kKeptKeys; i += T::THREADS)
      rowTop[i] = kEmptyKey;
  if (lane < kWaveRows) {
    rowBest[own] = kEmptyKey;
    rowNeed[own] = open ? INFINITY : -1.0f;
  }
  if (lane == 0)
    bound[wave] = INFINITY;
  // The box, smallest weight value and components of the wave's open rows.
  float *rowBox = rowBoxes + wave * 2 * d;
  for (int f = 0; f < d; ++f) {
    const float v = open ? rowX[(size_t)ownRow * d + f] : 0.0f;
    float lo = open ? v : INFINITY, hi = open ? v : -INFINITY;
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
  float rowMinValue = open && Weight::kHasValue ? (float)weight.value(posOf(ownRow)) : INFINITY;
  int compLow = open ? ownComp : 0x7fffffff, compHigh = open ? ownComp : -1;
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) {
    rowMinValue = fminf(rowMinValue, __shfl_xor(rowMinValue, m, 64));
    compLow = min(compLow, __shfl_xor(compLow, m, 64));
    compHigh = max(compHigh, __shfl_xor(compHigh, m, 64));
  }
  if (!Weight::kHasValue)
    rowMinValue = 0.0f;
  auto capOf = [&](unsigned int bits) { return bits == 0xffffffffu ? INFINITY : floatOf(bits); };
  const float slack = 1.0f - boxSlack(d);

  int rowComp[TR];
  typename Weight::Value rowVal[TR];
#pragma unroll
  for (int r = 0; r < TR; ++r) {
    const int row = row0 + T::rowInTile(r);
    rowComp[r] = isOpen(row) ? comp[posOf(row)] : -2;
    rowVal[r] = weight.value(row < nRows ? posOf(row) : 0);
  }
  unsigned long long computed = 0;
  // The 8-feature tiles serve d <= 8 only (one fill): the row slice is
  // staged once for every tile.
  constexpr bool kRowsResident = T::FILL == 8;
  if (kRowsResident)
    stageRows<T>(sm, rowX, nRows, d, row0);
  __syncthreads();

  // The wave's bound: the largest need over its open rows (inf while a row of
  // a component without a known edge has no candidate yet, -1 without open
  // rows). Publishes each row's need.
  auto newBound = [&]() {
    float need = -1.0f;
    if (open) {
      const unsigned long long k =
          KEEP ? rowTop[own * kKeptKeys + kKeptKeys - 1] : rowBest[own];
      const float w = k == kEmptyKey ? INFINITY : keyWeight(k);
      if (compBest && w < cap) {
        atomicMin(&compBest[ownComp], bitsOf(w));
        cap = w;
      }
      need = fminf(w, cap);
      rowNeed[own] = need;
    }
#pragma unroll
    for (int m = kWaveRows / 2; m > 0; m >>= 1)
      need = fmaxf(need, __shfl_xor(need, m, 64));
    if (lane == 0)
      bound[wave] = need;
    return __shfl(need, 0, 64);
  };

  const int steps = 2 * ((numTiles + splits - 1) / splits) + 1;
  for (int base = 0; base < steps; base += kBatch) {
    // Other workgroups may have found better edges for these components, and
    // other splits for these rows.
    if (compBest && open)
      cap = fminf(cap, capOf(compBest[ownComp]));
    if (!KEEP && splits > 1 && open) {
      unsigned long long *shared = &nearest[posOf(ownRow)];
      const unsigned long long mine = rowBest[own];
      const unsigned long long theirs =
          __hip_atomic_load(shared, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (mine < theirs)
        atomicMin(shared, mine);
      else
        rowBest[own] = theirs;
    }
    const float reach = newBound();
    {
      // -1: never computed (outside the grid, or both sides wholly one component).
      const int step = base + lane;
      const int colTile = step < steps ? walkTile(center, step, numTiles, splits, split) : -1;
      float lb = -1.0f;
      if (colTile >= 0 && !(compLow == compHigh && boxes.minComp[colTile] == compLow &&
                            boxes.maxComp[colTile] == compLow)) {
        const float db = boxLowerBound(metric, rowBox, rowBox + d, boxes.low + (size_t)colTile * d,
                                       boxes.high + (size_t)colTile * d, d);
        lb = weight(db, rowMinValue, boxes.minValue[colTile]) * slack;
      }
      lowerBound[wave][lane] = lb;
      const unsigned long long mask = __ballot(lb >= 0.0f && !(lb > reach));
      if (lane == 0)
        within[wave] = mask;
    }
    __syncthreads();
    unsigned long long todo = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
      todo |= within[w];
    for (; todo; todo &= todo - 1) {
      const int j = __ffsll((long long)todo) - 1;
      // Uniform: written before the barrier after the last computed tile.
      bool active = false;
      int activeWaves = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float lb = lowerBound[w][j];
        const bool in = lb >= 0.0f && !(lb > bound[w]);
        activeWaves += in;
        if (w == wave)
          active = in;
      }
      if (activeWaves == 0)
        continue;
      const int colTile = walkTile(center, base + j, numTiles, splits, split);
      computed += activeWaves;
      if (base + j >= computeSteps)
        continue; // estimate: counted against the bound reached so far, not computed
      const int col0 = colTile * T::DIM;
      float w[TR][TR]; // raw accumulators when filtering
      // The column data arrives with the tile's first fill (LDS, read after
      // computeTile's barriers; rewritten only after this tile's last barrier).
      const ColumnStage<Weight> stage{comp, orig, weight, col0, n, T::DIM,
                                      sColComp, sColVal, sColIdx};
      computeTile<T, Metric, !kFilter, kRowsResident, true>(sm, rowX, nRows, X, n, d, metric,
                                                            row0, col0, w, stage, active);
      if (active) {
        bool improved = false; // a row's best (or list) of this wave
        int colComp[TR];
        typename Weight::Value colVal[TR];
        unsigned int colIdx[TR];
#pragma unroll
        for (int c = 0; c < TR; ++c) {
          const int i = T::colInTile(c);
          colComp[c] = sColComp[i];
          colVal[c] = sColVal[i];
          colIdx[c] = sColIdx[i];
        }
        if constexpr (KEEP) {
          const unsigned long long groupMask = 0xffffull << (lane & 48);
#pragma unroll
          for (int r = 0; r < TR; ++r) {
            int i = T::rowInTile(r);
            asm volatile("" : "+v"(i)); // computed here, not kept for every row
            unsigned long long *top = rowTop + i * kKeptKeys;
            // Pairs that can enter the row's list.
            const float need = rowNeed[i];
            const float limit = need < 0.0f ? -INFINITY
                                : kFilter   ? metric.accBound(weight.distBound(need))
                                            : INFINITY;
            const unsigned long long last = top[kKeptKeys - 1];
            unsigned int pending = 0;
#pragma unroll
            for (int c = 0; c < TR; ++c) {
              const float acc = w[r][c];
              if (!(acc > limit) && colComp[c] != rowComp[r] && rowComp[r] >= 0 &&
                  colComp[c] >= 0) {
                const float ww = weight(kFilter ? metric.finish(acc) : acc, rowVal[r], colVal[c]);
                w[r][c] = ww;
                if (ww != INFINITY && packKey(ww, colIdx[c]) < last)
                  pending |= 1u << c;
              }
            }
            // One insertion per row group at a time; the lanes stay converged.
            // The row's lowest lane with work gives its key, and its 16 lanes
            // insert it: entry q takes the larger of the key and its
            // predecessor where it is above the key.
            while (true) {
              const unsigned long long work = __ballot(pending != 0);
              if (work == 0)
                break;
              improved = true;
              const unsigned long long mine = work & groupMask;
              const int source = mine ? __ffsll((long long)mine) - 1 : lane;
              const int c = __ffs(pending) - 1;
              float wv = 0.0f;
              unsigned int idx = 0;
#pragma unroll
              for (int cc = 0; cc < TR; ++cc)
                if (cc == c) {
                  wv = w[r][cc];
                  idx = colIdx[cc];
                }
              if (lane == source)
                pending &= pending - 1;
              const unsigned long long key =
                  packKey(__shfl(wv, source, 64), (unsigned int)__shfl((int)idx, source, 64));
              const int q = lane & 15;
              if (mine && q < kKeptKeys) {
                const unsigned long long cur = top[q], prev = q > 0 ? top[q - 1] : 0;
                if (cur > key)
                  top[q] = prev > key ? prev : key;
              }
              __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
              __builtin_amdgcn_wave_barrier();
              __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
              if (pending) {
                const unsigned long long now = top[kKeptKeys - 1];
#pragma unroll
                for (int cc = 0; cc < TR; ++cc)
                  if (!(packKey(w[r][cc], colIdx[cc]) < now))
                    pending &= ~(1u << cc);
              }
            }
          }
        } else {
#pragma unroll
          for (int r = 0; r < TR; ++r) {
            unsigned long long best = kEmptyKey;
            if constexpr (kFilter) {
              const float need = rowNeed[T::rowInTile(r)];
              const float limit = need < 0.0f ? -INFINITY : metric.accBound(weight.distBound(need));
#pragma unroll
              for (int c = 0; c < TR; ++c) {
                const float acc = w[r][c];
                if (!(acc > limit) && colComp[c] != rowComp[r]) {
                  const float ww = weight(metric.finish(acc), rowVal[r], colVal[c]);
                  if (rowComp[r] >= 0 && colComp[c] >= 0 && ww != INFINITY)
                    best = minKey(best, packKey(ww, colIdx[c]));
                }
              }
            } else {
#pragma unroll
              for (int c = 0; c < TR; ++c) {
                const float ww = weight(w[r][c], rowVal[r], colVal[c]);
                const bool counts = rowComp[r] >= 0 && colComp[c] >= 0 &&
                                    colComp[c] != rowComp[r] && ww != INFINITY;
                if (counts)
                  best = minKey(best, packKey(ww, colIdx[c]));
              }
            }
            // Wave-uniform: most rows of most tiles have no candidate.
            if (__ballot(best != kEmptyKey) != 0) {
              best = rowGroupMin(best);
              if (T::tc() == 0 && best != kEmptyKey) {
                const int i = T::rowInTile(r);
                if (best < rowBest[i]) {
                  rowBest[i] = best;
                  improved = true;
                }
              }
            }
          }
        }
        // The needs and the bound change only with a row's best.
        if (__ballot(improved) != 0) {
          __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
          (void)newBound();
        }
      }
      __syncthreads(); // the tile is consumed, the waves' bounds are current
    }
    __syncthreads(); // lowerBound is rewritten by the next batch
  }
  if (KEEP) {
    for (int e = threadIdx.x; e < T::DIM * kKeptKeys; e += T::THREADS) {
      const int i = e / kKeptKeys;
      if (row0 + i < nRows)
        kept[((size_t)split * n + posOf(row0 + i)) * kKeptKeys + e % kKeptKeys] = rowTop[e];
    }
    for (int i = threadIdx.x; i < T::DIM; i += T::THREADS)
      rowBest[i] = rowTop[i * kKeptKeys];
  }
  for (int i = threadIdx.x; i < T::DIM; i += T::THREADS)
    if (row0 + i < nRows && rowBest[i] != kEmptyKey)
      atomicMin(&nearest[posOf(row0 + i)], rowBest[i]);
  if (wavesComputed && threadIdx.x == 0)
    atomicAdd(wavesComputed, computed);
}

// Seeds each component's best known edge weight for the next pass from the
// previous pass's results: a point whose previous candidate lies in another
// component still has that edge. With few components the workgroup first
// combines its points in LDS (one global atomic per component per workgroup).
constexpr int kSeedLds = 4096;

__global__ void __launch_bounds__(256)
    seedComponentBestKernel(const unsigned long long *__restrict__ nearest,
                            const int *__restrict__ comp, const int *__restrict__ posOf, int n,
                            int numComp, unsigned int *compBest) {
  __shared__ unsigned int local[kSeedLds];
  const bool useLds = numComp <= kSeedLds;
  if (useLds) {
    for (int c = threadIdx.x; c < numComp; c += blockDim.x)
      local[c] = 0xffffffffu;
    __syncthreads();
  }
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    const unsigned long long key = nearest[p];
    if (key == kEmptyKey)
      continue;
    const int q = (int)keyIndex(key);
    const int c = comp[p];
    if (comp[posOf ? posOf[q] : q] == c)
      continue; // the partner joined this component
    const unsigned int bits = (unsigned int)(key >> 32);
    if (useLds)
      atomicMin(&local[c], bits);
    else
      atomicMin(&compBest[c], bits);
  }
  if (useLds) {
    __syncthreads();
    for (int c = threadIdx.x; c < numComp; c += blockDim.x)
      if (local[c] != 0xffffffffu)
        atomicMin(&compBest[c], local[c]);
  }
}

__global__ void inverseOrderKernel(const int *__restrict__ orig, int n, int *__restrict__ posOf) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n)
    posOf[orig[p]] = p;
}

__global__ void gatherRowsKernel(const float *__restrict__ src, const int *__restrict__ order,
                                 int n, int d, float *__restrict__ dst) {
  const size_t total = (size_t)n * d;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total;
       e += (size_t)gridDim.x * blockDim.x) {
    const size_t row = e / d, f = e - row * d;
    dst[e] = src[(size_t)order[row] * d + f];
  }
}

__global__ void iotaKernel(int *out, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    out[i] = i;
}

template <class Metric, class F> int withWeightFor(const Metric &, WeightSpec w, F &&f) {
  switch (w.kind) {
  case kWeightPlain: return f(PlainWeight{});
  case kWeightMReach:
    return w.alpha == 1.0f ? f(MReachWeightT<false>{w.core, 1.0f})
                           : f(MReachWeightT<true>{w.core, w.alpha});
  default: return kErrInvalidAlgorithm;
  }
}

} // namespace

// ---------------------------------------------------------------------------
// Host entry points

int pairwiseMatrix(const float *A, int nA, const float *B, int nB, int d, MetricSpec m,
                   float *out) {
  return withMetric(m, [&](auto metric) {
    using Metric = decltype(metric);
    return withFill(d, [&](auto fill) {
      using T = typename TileFor<Metric, decltype(fill)::value>::type;
      const int tilesA = (nA + T::DIM - 1) / T::DIM, tilesB = (nB + T::DIM - 1) / T::DIM;
      const long long blocks = (long long)tilesA * tilesB;
      if (blocks > 0x7fffffffLL)
        return (int)hipErrorInvalidConfiguration;
      hipLaunchKernelGGL((pairwiseMatrixKernel<T, Metric>), dim3((unsigned)blocks), dim3(256), 0,
                         stream(), A, nA, B, nB, d, metric, out, tilesB);
      return (int)hipGetLastError();
    });
  });
}

int condensedMatrix(const float *X, int n, int d, MetricSpec m, float *out) {
  return withMetric(m, [&](auto metric) {
    using Metric = decltype(metric);
    return withFill(d, [&](auto fill) {
      using T = typename TileFor<Metric, decltype(fill)::value>::type;
      const long long tiles = (n + T::DIM - 1) / T::DIM;
      const long long pairs = tiles * (tiles + 1) / 2;
      hipLaunchKernelGGL((condensedMatrixKernel<T, Metric>), dim3(persistentBlocks(pairs, 8)),
                         dim3(256), 0, stream(), X, n, d, metric, out, pairs);
      return (int)hipGetLastError();
    });
  });
}

int nearestOtherSymmetric(const float *X, int n, int d, MetricSpec m, WeightSpec w,
                          const int *comp, const int *orig, unsigned long long *nearest,
                          const int *numComp) {
  return withMetric(m, [&](auto metric) {
    using Metric = decltype(metric);
    return withWeightFor(metric, w, [&](auto weight) {
      using Weight = decltype(weight);
      return withFill(d, [&](auto fill) {
        using T = typename TileFor<Metric, decltype(fill)::value>::type;
        const long long tiles = (n + T::DIM - 1) / T::DIM, pairs = tiles * (tiles + 1) / 2;
        PhaseTimer timer(kPhaseDistanceTiles);
        addUnits(kPhaseDistanceTiles, (long long)n * (n + 1) / 2);
        hipLaunchKernelGGL((nearestOtherSymmetricKernel<T, Metric, Weight>),
                           dim3(persistentBlocks(pairs, 8)), dim3(256), 0, stream(), X, n, d,
                           metric, weight, comp, orig, nearest, pairs, numComp);
        return (int)hipGetLastError();
      });
    });
  });
}

bool shouldPrune(int mode, int metricId, int n, int d) {
  const int tiles = (n + 127) / 128;
  if (!metricHasBoxBound(metricId) || mode == kPruneNever || tiles < 2 ||
      d > kPruneHardMaxFeatures)
    return false;
  return mode == kPruneAlways || (n >= kPruneMinPoints && d <= kPruneMaxFeatures);
}

int gatherRows(const float *src, const int *order, int n, int d, float *dst) {
  hipLaunchKernelGGL(gatherRowsKernel, dim3(std::max(1, std::min(4096, (n * d + 255) / 256))),
                     dim3(256), 0, stream(), src, order, n, d, dst);
  return (int)hipGetLastError();
}

namespace {

struct DeviceBoxes {
  DevArray<float> low, high, minValue;
  DevArray<int> minComp, maxComp;
  Boxes view;
  int alloc(int tiles, int d) {
    Status s;
    s(low.alloc((size_t)tiles * d));
    s(high.alloc((size_t)tiles * d));
    s(minValue.alloc(tiles));
    s(minComp.alloc(tiles));
    s(maxComp.alloc(tiles));
    view = Boxes{low, high, minValue, minComp, maxComp, tiles};
    return s.code;
  }
};

// Walk steps computed per row tile by the sampled estimate (stride > 1); later
// steps are only counted against the bound the computed ones reached (an
// overestimate of the pruned share: the bound would keep shrinking).
constexpr int kEstimateSteps = 64;

// Splits of a walk over rowTiles row tiles: enough workgroups to even out the
// row tiles' very different lengths (a resident chip's worth several times
// over), each with eight column tiles at least. However many row tiles
// there are, a split walks about longest column tiles at most: a later round
// leaves a few sparse rows that walk all the way alone (rounds 3 and 4 over 10^6
// points of 8 features, 7,813 tiles: 30 ms each, 6 of them VALU work; by 1,024
// tiles 13 ms).
int walkSplits(int rowTiles, int tiles, int most, int longest) {
  const int wanted = std::max(16 * numCUs() / std::max(1, rowTiles), tiles / longest);
  return std::max(1, std::min({wanted, tiles / 8, most}));
}
constexpr int kMostSplits = 64;
constexpr int kLongestWalk = 1024;
constexpr int kKeptSplits = 4; // each split keeps a list of its own to merge

// The lowest keys of a row's lists (ascending, distinct columns but for the
// row's own tile, which every split walks) into the first list.
__global__ void mergeKeptKernel(const unsigned long long *__restrict__ lists, int splits, int n,
                                unsigned long long *__restrict__ kept) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n)
    return;
  unsigned long long key[kKeptKeys];
#pragma unroll
  for (int q = 0; q < kKeptKeys; ++q)
    key[q] = lists[(size_t)p * kKeptKeys + q];
  for (int s = 1; s < splits; ++s)
#pragma unroll
    for (int e = 0; e < kKeptKeys; ++e) {
      unsigned long long k = lists[((size_t)s * n + p) * kKeptKeys + e];
      bool known = false;
#pragma unroll
      for (int q = 0; q < kKeptKeys; ++q)
        known |= key[q] == k;
      if (known)
        continue;
#pragma unroll
      for (int q = 0; q < kKeptKeys; ++q) {
        const unsigned long long cur = key[q];
        key[q] = minKey(cur, k);
        k = k < cur ? cur : k;
      }
    }
#pragma unroll
  for (int q = 0; q < kKeptKeys; ++q)
    kept[(size_t)p * kKeptKeys + q] = key[q];
}

// Dynamic LDS of the walk: a row box per wave.
template <class T> size_t walkBoxBytes(int d) {
  return (size_t)(T::THREADS / 64) * 2 * d * sizeof(float);
}

template <class T, class Metric, class Weight>
int runWalk(const float *X, int n, int d, const Metric &metric, const Weight &weight,
            const int *comp, const int *orig, unsigned int *compBest,
            unsigned long long *nearest, double *share, PassStats *stats, int stride,
            const int *skipComp, const unsigned char *closedRows,
            unsigned long long *kept = nullptr) {
  const int tiles = (n + T::DIM - 1) / T::DIM;
  DeviceBoxes boxes;
  DevArray<unsigned long long> counter;
  Status s;
  s(boxes.alloc(tiles, d));
  s(counter.alloc(1));
  if (!s.ok())
    return s.code;
  s(fill(counter, 0, sizeof(unsigned long long)));
  hipLaunchKernelGGL((buildBoxesKernel<Weight>), dim3(tiles), dim3(64), 0, stream(), X, n, d,
                     T::DIM, weight, comp, boxes.view);
  s((int)hipGetLastError());
  const int sampled = (tiles + stride - 1) / stride;
  {
    PhaseTimer timer(kPhaseDistanceTiles);
    bool launched = false;
    if constexpr (Weight::kDistBound) { // not Ward's, which keeps its own lists
      if (kept) {
        // Without the memory for the splits' lists, one split.
        int splits = walkSplits(sampled, tiles, kKeptSplits, 0x7fffffff);
        DevArray<unsigned long long> lists;
        if (splits > 1 && lists.alloc((size_t)splits * n * kKeptKeys)) {
          (void)hipGetLastError();
          splits = 1;
        }
        hipLaunchKernelGGL((nearestOtherWalkKernel<T, Metric, Weight, false, true>),
                           dim3(sampled, splits), dim3(256), walkBoxBytes<T>(d), stream(), X, n, d,
                           metric, weight, comp, orig, boxes.view, nullptr, nearest,
                           counter.get(), stride, stride > 1 ? kEstimateSteps : 0x7fffffff,
                           skipComp, closedRows, RowSet{}, splits > 1 ? lists.get() : kept);
        if (splits > 1)
          hipLaunchKernelGGL(mergeKeptKernel, dim3((n + 255) / 256), dim3(256), 0, stream(),
                             lists.get(), splits, n, kept);
        launched = true;
      }
    }
    if (!launched)
      hipLaunchKernelGGL((nearestOtherWalkKernel<T, Metric, Weight>),
                         dim3(sampled, stride > 1 ? 1 : walkSplits(sampled, tiles, kMostSplits,
                                                                   kLongestWalk)),
                         dim3(256), walkBoxBytes<T>(d), stream(), X, n, d, metric, weight, comp, orig,
                         boxes.view, compBest, nearest, counter.get(), stride,
                         stride > 1 ? kEstimateSteps : 0x7fffffff, skipComp, closedRows,
                         RowSet{}, nullptr);
    s((int)hipGetLastError());
  }
  unsigned long long computed = 0;
  s(download(&computed, counter, sizeof(computed)));
  // The kernel counts quarter tiles (a wave's rows).
  constexpr int kWaves = T::THREADS / 64;
  const unsigned long long total = (unsigned long long)sampled * tiles;
  *share = total ? (double)computed / (double)(total * kWaves) : 1.0;
  addUnits(kPhaseDistanceTiles, (long long)computed * T::WAVE_ROWS * T::DIM);
  if (stats && s.ok()) {
    stats->tilesComputed += (computed + kWaves - 1) / kWaves;
    stats->tilesTotal += total;
  }
  return s.code;
}

// Open rows of a walk: not closed and not in the skipped component.
__global__ void openRowFlagsKernel(const int *__restrict__ comp, const int *__restrict__ skipComp,
                                   const unsigned char *__restrict__ closedRows, int n,
                                   int *flags) {
  const int skip = skipComp ? *skipComp : -1;
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p <= n; p += gridDim.x * blockDim.x)
    flags[p] = p < n && comp[p] != skip && !closedRows[p];
}

__global__ void openRowListKernel(const int *__restrict__ flags, const int *__restrict__ index,
                                  int n, int *rowPos) {
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x)
    if (flags[p])
      rowPos[index[p]] = p;
}

// The full-order tile of each compact row tile's middle row.
__global__ void rowTileCentersKernel(const int *__restrict__ rowPos, int nOpen, int tileDim,
                                     int rowTiles, int *center) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < rowTiles)
    center[t] = rowPos[min(t * tileDim + tileDim / 2, nOpen - 1)] / tileDim;
}

// The walk over the open rows only, when closed rows are given: those rows
// (in the full order, so spatially coherent) are gathered into compact row
// tiles with their own boxes, each walking the column tiles around the full
// order's tile of its middle row. With most rows closed, a tile of the full
// order usually keeps a few open rows and walks as far as they need; the
// compact tiles walk for open rows only. The share reported is of the full
// grid's tile pairs.
template <class T, class Metric, class Weight>
int runWalkOpen(const float *X, int n, int d, const Metric &metric, const Weight &weight,
                const int *comp, const int *orig, unsigned int *compBest,
                unsigned long long *nearest, double *share, PassStats *stats,
                const int *skipComp, const unsigned char *closedRows, double keptShare) {
  const int tiles = (n + T::DIM - 1) / T::DIM;
  Status s;
  DevArray<int> flags, index, rowPos;
  DevArray<unsigned char> temp;
  s(flags.alloc((size_t)n + 1));
  s(index.alloc((size_t)n + 1));
  s(rowPos.alloc(n));
  s(temp.alloc(scanTempBytes(n + 1)));
  if (!s.ok())
    return s.code;
  const int blocks = std::max(1, std::min(4 * numCUs(), (n + 256) / 256));
  hipLaunchKernelGGL(openRowFlagsKernel, dim3(blocks), dim3(256), 0, stream(), comp, skipComp,
                     closedRows, n, flags.get());
  s(exclusiveScan(flags, index, n + 1, temp));
  int nOpen = 0;
  s(download(&nOpen, index.get() + n, sizeof(int)));
  if (!s.ok())
    return s.code;
  // A walk of every row that leaves out few pairs takes 2.3 symmetric passes
  // (92,000 points of 60 features in blobs, manhattan: 33 and 13.3 ms; whole
  // calls 92.8 ms with the walks alone, 73.5 with this rule).
  if (keptShare * nOpen > 0.5 * n) {
    *share = -1.0;
    return 0;
  }
  if (4LL * nOpen > 3LL * n) // most rows open: the full order's tiles
    return runWalk<T>(X, n, d, metric, weight, comp, orig, compBest, nearest, share, stats, 1,
                      skipComp, closedRows);
  *share = 0.0;
  if (nOpen == 0)
    return 0;
  hipLaunchKernelGGL(openRowListKernel, dim3(blocks), dim3(256), 0, stream(), flags.get(),
                     index.get(), n, rowPos.get());
  const int rowTiles = (nOpen + T::DIM - 1) / T::DIM;
  DeviceBoxes colBoxes;
  DevArray<float> rowX;
  DevArray<int> center;
  DevArray<unsigned long long> counter;
  s(colBoxes.alloc(tiles, d));
  s(rowX.alloc((size_t)nOpen * d));
  s(center.alloc(rowTiles));
  s(counter.alloc(1));
  if (!s.ok())
    return s.code;
  s(fill(counter, 0, sizeof(unsigned long long)));
  s(gatherRows(X, rowPos, nOpen, d, rowX));
  hipLaunchKernelGGL((buildBoxesKernel<Weight>), dim3(tiles), dim3(64), 0, stream(), X, n, d,
                     T::DIM, weight, comp, colBoxes.view);
  hipLaunchKernelGGL(rowTileCentersKernel, dim3((rowTiles + 255) / 256), dim3(256), 0, stream(),
                     rowPos.get(), nOpen, T::DIM, rowTiles, center.get());
  s((int)hipGetLastError());
  RowSet rows;
  rows.X = rowX;
  rows.n = nOpen;
  rows.pos = rowPos;
  rows.center = center;
  {
    PhaseTimer timer(kPhaseDistanceTiles);
    hipLaunchKernelGGL((nearestOtherWalkKernel<T, Metric, Weight, true>),
                       dim3(rowTiles, walkSplits(rowTiles, tiles, kMostSplits, kLongestWalk)),
                       dim3(256), walkBoxBytes<T>(d), stream(), X, n, d, metric, weight, comp,
                       orig, colBoxes.view, compBest, nearest, counter.get(), 1, 0x7fffffff,
                       skipComp, closedRows, rows, nullptr);
    s((int)hipGetLastError());
  }
  unsigned long long computed = 0;
  s(download(&computed, counter, sizeof(computed)));
  const unsigned long long total = (unsigned long long)tiles * tiles;
  constexpr int kWaves = T::THREADS / 64; // the kernel counts quarter tiles
  *share = (double)computed / (double)(total * kWaves);
  addUnits(kPhaseDistanceTiles, (long long)computed * T::WAVE_ROWS * T::DIM);
  if (stats && s.ok()) {
    stats->tilesComputed += (computed + kWaves - 1) / kWaves;
    stats->tilesTotal += total;
  }
  return s.code;
}

} // namespace

int nearestOtherWalk(const float *X, int n, int d, MetricSpec m, WeightSpec w, const int *comp,
                     const int *orig, unsigned int *compBest, unsigned long long *nearest,
                     double *share, PassStats *stats, int stride, const int *skipComp,
                     const unsigned char *closedRows, unsigned long long *kept,
                     double keptShare) {
  if (!metricHasBoxBound(m.id))
    return kErrInvalidMetric;
  if (kept && (w.kind == kWeightWard || closedRows || stride != 1))
    return kErrInvalidAlgorithm;
  if (w.kind == kWeightWard) {
    if (m.id != kSqEuclidean)
      return kErrInvalidMetric;
    return withFill(d, [&](auto fill) {
      using T = Tile<8, decltype(fill)::value, true>;
      return runWalk<T>(X, n, d, SqEuclidean{}, WardWeight{w.size}, comp, orig, compBest,
                        nearest, share, stats, stride, skipComp, closedRows);
    });
  }
  return withMetric(m, [&](auto metric) {
    using Metric = decltype(metric);
    if constexpr (!Metric::kBoxBound) {
      return kErrInvalidMetric;
    } else {
      return withWeightFor(metric, w, [&](auto weight) {
        return withFill(d, [&](auto fill) {
          using T = Tile<8, decltype(fill)::value, true>;
          // Closed rows (their answers settled from lists): walk the open rows
          // only.
          if (closedRows && stride == 1)
            return runWalkOpen<T>(X, n, d, metric, weight, comp, orig, compBest, nearest, share,
                                  stats, skipComp, closedRows, keptShare);
          return runWalk<T>(X, n, d, metric, weight, comp, orig, compBest, nearest, share,
                            stats, stride, skipComp, closedRows, kept);
        });
      });
    }
  });
}

namespace {

__global__ void settleFromKeptKernel(const unsigned long long *__restrict__ kept, int n,
                                     const int *__restrict__ comp, const int *__restrict__ posOf,
                                     const int *__restrict__ skipComp,
                                     unsigned long long *__restrict__ nearest,
                                     unsigned int *__restrict__ compBest,
                                     unsigned char *__restrict__ closed) {
  const int skip = skipComp ? *skipComp : -1;
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    const int c = comp[p];
    bool settled = false;
    if (c != skip) {
#pragma unroll
      for (int q = 0; q < kKeptKeys && !settled; ++q) {
        const unsigned long long key = kept[(size_t)p * kKeptKeys + q];
        if (key == kEmptyKey)
          break;
        const int j = posOf ? posOf[keyIndex(key)] : (int)keyIndex(key);
        if (comp[j] != c) {
          nearest[p] = key;
          if (compBest)
            atomicMin(&compBest[c], (unsigned int)(key >> 32));
          settled = true;
        }
      }
    }
    closed[p] = settled ? 1 : 0;
  }
}

} // namespace

namespace {

// Rows left open whose list ends above the best edge known for their component:
// every point the list misses weighs at least its last key, so the row cannot
// hold the component's smallest edge, and closes without an answer.
__global__ void closeHopelessKernel(const unsigned long long *__restrict__ kept, int n,
                                    const int *__restrict__ comp,
                                    const unsigned int *__restrict__ compBest,
                                    unsigned char *__restrict__ closed) {
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x)
    if (!closed[p]) {
      const unsigned long long last = kept[(size_t)p * kKeptKeys + kKeptKeys - 1];
      if (last == kEmptyKey || (unsigned int)(last >> 32) > compBest[comp[p]])
        closed[p] = 1;
    }
}

} // namespace

int settleFromKept(const unsigned long long *kept, int n, const int *comp, const int *posOf,
                   const int *skipComp, unsigned long long *nearest, unsigned int *compBest,
                   unsigned char *closed) {
  const int blocks = std::max(1, std::min(4 * numCUs(), (n + 255) / 256));
  hipLaunchKernelGGL(settleFromKeptKernel, dim3(blocks), dim3(256), 0, stream(), kept, n, comp,
                     posOf, skipComp, nearest, compBest, closed);
  if (compBest)
    hipLaunchKernelGGL(closeHopelessKernel, dim3(blocks), dim3(256), 0, stream(), kept, n, comp,
                       compBest, closed);
  return (int)hipGetLastError();
}

int seedComponentBest(const unsigned long long *nearest, const int *comp, const int *posOf,
                      int n, int numComp, bool fromNearest, unsigned int *compBest) {
  Status st;
  st(fill(compBest, 0xff, (size_t)numComp * sizeof(unsigned int)));
  if (fromNearest) {
    const int blocks = std::max(1, std::min(4 * numCUs(), (n + 255) / 256));
    hipLaunchKernelGGL(seedComponentBestKernel, dim3(blocks), dim3(256), 0, stream(), nearest,
                       comp, posOf, n, numComp, compBest);
    st((int)hipGetLastError());
  }
  return st.code;
}

int inverseOrder(const int *orig, int n, int *posOf) {
  hipLaunchKernelGGL(inverseOrderKernel, dim3((n + 255) / 256), dim3(256), 0, stream(), orig, n,
                     posOf);
  return (int)hipGetLastError();
}

namespace {

// Component sizes; with few components each workgroup counts in LDS first
// (same-address atomics from every point would serialise).
constexpr int kSizeLds = 4096;

__global__ void __launch_bounds__(256)
    componentSizesKernel(const int *__restrict__ comp, int n, int numComp, int *sizes) {
  __shared__ int local[kSizeLds];
  const bool useLds = numComp <= kSizeLds;
  if (useLds) {
    for (int c = threadIdx.x; c < numComp; c += blockDim.x)
      local[c] = 0;
    __syncthreads();
  }
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    if (useLds)
      atomicAdd(&local[comp[p]], 1);
    else
      atomicAdd(&sizes[comp[p]], 1);
  }
  if (useLds) {
    __syncthreads();
    for (int c = threadIdx.x; c < numComp; c += blockDim.x)
      if (local[c])
        atomicAdd(&sizes[c], local[c]);
  }
}

// At most one component holds more than half of the points.
__global__ void majorityKernel(const int *__restrict__ sizes, int numComp, int n,
                               int *majority) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < numComp && 2 * (long long)sizes[c] > (long long)n)
    *majority = c;
}

} // namespace

int majorityComponent(const int *comp, int n, int numComp, int *sizes, int *majority) {
  Status s;
  s(fill(majority, 0xff, sizeof(int))); // -1
  if (2 * (long long)numComp > (long long)n + 1) // every component has at most n - numComp + 1 points
    return s.code;
  s(fill(sizes, 0, (size_t)numComp * sizeof(int)));
  const int blocks = std::max(1, std::min(1024, (n + 255) / 256));
  hipLaunchKernelGGL(componentSizesKernel, dim3(blocks), dim3(256), 0, stream(), comp, n, numComp,
                     sizes);
  hipLaunchKernelGGL(majorityKernel, dim3((numComp + 255) / 256), dim3(256), 0, stream(), sizes,
                     numComp, n, majority);
  s((int)hipGetLastError());
  return s.code;
}

int estimatePrunedShare(const float *X, int n, int d, MetricSpec m, double *share) {
  constexpr int kSampleTiles = 32;
  const int tiles = (n + 127) / 128;
  const int stride = std::max(1, tiles / kSampleTiles);
  DevArray<int> comp, orig;
  DevArray<unsigned long long> nearest;
  Status s;
  s(comp.alloc(n));
  s(orig.alloc(n));
  s(nearest.alloc(n));
  if (!s.ok())
    return s.code;
  hipLaunchKernelGGL(iotaKernel, dim3(std::min(1024, (n + 255) / 256)), dim3(256), 0, stream(),
                     comp.get(), n);
  hipLaunchKernelGGL(iotaKernel, dim3(std::min(1024, (n + 255) / 256)), dim3(256), 0, stream(),
                     orig.get(), n);
  s(fill(nearest, 0xff, nearest.bytes()));
  s(nearestOtherWalk(X, n, d, m, WeightSpec{}, comp, orig, nullptr, nearest, share, nullptr,
                     stride));
  return s.code;
}

} // namespace cuhc

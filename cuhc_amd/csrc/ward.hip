// Exact Ward linkage without the n x n matrix: rounds of reciprocal nearest
// neighbours (reference src/rnn_ward.cuh) and the nearest-neighbour chain
// (src/nn_chain.cuh).
//
// Precision: cluster centroids live in FP64 on the GPU and every merge updates
// them in FP64 (c_a + (c_b - c_a) * n_b / (n_a + n_b), exact for duplicate
// centroids); merge heights are accumulated in FP64,
// sqrt(2 n_a n_b / (n_a + n_b) * sum (c_a - c_b)^2). The RNN rounds choose
// nearest neighbours by FP32 searches of an FP32 copy of the centroids and
// Ward's FP32 weight (symmetric bit for bit, so the closest pair always sees
// each other and every round makes progress).
#include "linkage.hpp"
#include "mst.hpp"
#include "primitives.hpp"
#include "tile.hpp"

#include <hip/hip_cooperative_groups.h>

#include <algorithm>
#include <numeric>
#include <type_traits>

namespace cuhc {

namespace {

namespace cg = cooperative_groups;

struct Clusters {
  double *c64;
  float *c32;
  int *size;
  int *rep;
};

struct DevMerge {
  int u, v;
  double h;
};

// ---------------------------------------------------------------------------
// Rounds of reciprocal nearest neighbours.
//
// Every cluster keeps a list of its kList nearest clusters, exactly the lowest
// keys (FP32 Ward weight, slot), and a bound below every key that is not in the
// list; its nearest is the list's first. A round merges the reciprocal pairs
// and compacts the slots in order. The weights between clusters that did not
// merge do not change, so a list without its merged entries still holds the
// lowest keys, and only the merged clusters and those whose list ran out search
// again (a few tenths of the rows against all columns; the lower triangle of
// all pairs before). A search row that is a new cluster offers its weight to
// every column whose bound lies above it (pushed[]); the lowest offer enters
// the column's list, which ends there: what else was offered weighs more. Slots
// keep their order through a compaction, so keys keep theirs and every
// nearest, ties included, is the one a pass over all pairs would find.
//
// Bound by FP32 VALU work at large m, by launches and dependent waits at small:
// the cluster count stays on the device, so that rounds are queued several at a
// time without a host read, each of 4 launches (up to 8,192 clusters; 8 above,
// three of them the scan that numbers the survivors).
// A pass over all pairs per round and its read took 4.3 ms for 3,001 points of
// 13 features (55 rounds) and 99 ms for 100,000 of 32 (95 rounds); now 2.6 and
// 61 ms.
constexpr int kList = 4;       // 8 searches a quarter fewer pairs and takes as long
constexpr int kRoundsAhead = 8;    // rounds queued per host read
// Workgroups per CU, and the work items a search is split into: two for each
// of them on 256 CUs (with 1,024 items a third of the chip waited for the
// second ones).
constexpr int kSearchGroups = 3;
constexpr int kSearchItems = 1536;
constexpr int kSmallSearch = 16384; // clusters up to which tiles are 64 a side

struct RoundState {
  int m;        // clusters
  int merges;   // recorded so far
  int searches; // rows of the current search
  int stop;     // a round fell below the wanted progress: queued rounds do nothing
  int rounds;   // rounds done
  unsigned long long pairs; // weights computed by the searches
};

struct Lists {
  unsigned long long *keys;  // [m][kList], ascending, kEmptyKey padded
  unsigned long long *bound; // [m]
};

// Column splits of a search and its work items (row tile, split).
DEV int searchSplits(int rows, int m, int dim) {
  const int rowTiles = (rows + dim - 1) / dim, colTiles = (m + dim - 1) / dim;
  return max(1, min(colTiles, kSearchItems / max(1, rowTiles)));
}

DEV bool roundOver(const RoundState *st) { return st->stop != 0 || st->m <= 1; }

DEV int reciprocalPartner(const unsigned long long *keys, int i) {
  const unsigned long long k = keys[(size_t)i * kList];
  if (k == kEmptyKey)
    return -1;
  const int j = keyIndex(k);
  const unsigned long long back = keys[(size_t)j * kList];
  return back != kEmptyKey && keyIndex(back) == i ? j : -1;
}

// The end of a round: its place in the merges, the new count, and whether it
// made enough progress.
DEV void endRound(RoundState *st, int now, float minProgress, int *roundEnd) {
  if (roundOver(st))
    return;
  const int before = st->m;
  roundEnd[st->rounds++] = st->merges;
  st->m = now;
  if (now > 1 && (now == before || (float)(before - now) < minProgress * (float)before))
    st->stop = 1;
}

__global__ void roundEndKernel(RoundState *st, const int *__restrict__ mNow, float minProgress,
                               int *roundEnd) {
  endRound(st, *mNow, minProgress, roundEnd);
}

// partner[i] (-1: none) and survives[i] for i <= mMost (mMost: the most
// clusters there can be); the scan of survives numbers the next round's slots.
__global__ void survivorsKernel(Lists lists, RoundState *st, int mMost, int *partner,
                                int *survives) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i > mMost)
    return;
  const int m = roundOver(st) ? 0 : st->m;
  int keep = 0;
  if (i < m) {
    const int j = reciprocalPartner(lists.keys, i);
    partner[i] = j;
    keep = !(j >= 0 && j < i);
  }
  survives[i] = keep;
  if (i == 0)
    st->searches = 0;
}

// The same and its scan by one workgroup, after the end of the round before
// (first: there is none). newIndex[mMost] receives the survivors.
constexpr int kSmallThreads = 1024;
constexpr int kSmallPer = 8;
constexpr int kSmallClusters = kSmallThreads * kSmallPer;

__global__ void __launch_bounds__(kSmallThreads)
    smallRoundKernel(Lists lists, RoundState *st, int mMost, bool first, float minProgress,
                     int *roundEnd, int *partner, int *newIndex) {
  __shared__ int waveTotal[kSmallThreads / 64];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  if (t == 0 && !first)
    endRound(st, newIndex[mMost], minProgress, roundEnd);
  __syncthreads();
  if (roundOver(st))
    return;
  const int m = st->m;
  const int per = (m + kSmallThreads - 1) / kSmallThreads, i0 = t * per;
  int keep = 0; // bit q: slot i0 + q survives
#pragma unroll
  for (int q = 0; q < kSmallPer; ++q) {
    const int i = i0 + q;
    if (q < per && i < m) {
      const int j = reciprocalPartner(lists.keys, i);
      partner[i] = j;
      keep |= !(j >= 0 && j < i) ? 1 << q : 0;
    }
  }
  int upTo = __popc(keep);
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(upTo, d, 64);
    if (lane >= d)
      upTo += up;
  }
  if (lane == 63)
    waveTotal[wave] = upTo;
  __syncthreads();
  int at = upTo - __popc(keep), total = 0;
  for (int w = 0; w < kSmallThreads / 64; ++w) {
    at += w < wave ? waveTotal[w] : 0;
    total += waveTotal[w];
  }
#pragma unroll
  for (int q = 0; q < kSmallPer; ++q)
    if (q < per && i0 + q < m) {
      newIndex[i0 + q] = at;
      at += keep >> q & 1;
    }
  __syncthreads();
  if (t == 0) {
    newIndex[mMost] = total; // past every slot
    st->searches = 0;
  }
}

// Surviving slot i goes to newIndex[i]; if it pairs with a higher slot j, the
// merged centroid goes there and the merge is recorded (heights in FP64). The
// first slotBlocks workgroups take a slot per thread (sizes, merges, and the
// slot's list: carried over, or put on the search list as slot with the top bit
// for a new cluster, searchOf[slot] its place or -1), the others a centroid
// coordinate per thread.
__global__ void __launch_bounds__(256)
    rnnMergeKernel(Clusters cur, Clusters next, Lists from, Lists to,
                   const int *__restrict__ partner, const int *__restrict__ newIndex, int d,
                   RoundState *st, DevMerge *merges, unsigned int *searchRows, int *searchOf,
                   unsigned long long *pushed, int slotBlocks) {
  if (roundOver(st))
    return;
  const int m = st->m;
  if ((int)blockIdx.x >= slotBlocks) {
    const size_t total = (size_t)m * d;
    for (size_t e = ((size_t)blockIdx.x - slotBlocks) * blockDim.x + threadIdx.x; e < total;
         e += (size_t)(gridDim.x - slotBlocks) * blockDim.x) {
      const int i = (int)(e / d), k = (int)(e - (size_t)i * d);
      const int j = partner[i];
      if (j >= 0 && j < i)
        continue;
      const double ci = cur.c64[e];
      double c = ci;
      if (j >= 0) {
        const double si = cur.size[i], sj = cur.size[j];
        c = fma(cur.c64[(size_t)j * d + k] - ci, sj / (si + sj), ci);
      }
      const size_t at = (size_t)newIndex[i] * d + k;
      next.c64[at] = c;
      next.c32[at] = (float)c;
    }
    return;
  }
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m)
    return;
  const int j = partner[i];
  if (j >= 0 && j < i)
    return;
  const int at = newIndex[i];
  next.size[at] = cur.size[i] + (j >= 0 ? cur.size[j] : 0);
  next.rep[at] = cur.rep[i];
  pushed[at] = kEmptyKey;
  int left = 0;
  if (j < 0) {
    for (int q = 0; q < kList; ++q) {
      const unsigned long long key = from.keys[(size_t)i * kList + q];
      if (key == kEmptyKey)
        break;
      const int s = keyIndex(key);
      if (partner[s] < 0)
        to.keys[(size_t)at * kList + left++] =
            (key & 0xffffffff00000000ull) | (unsigned int)newIndex[s];
    }
    for (int q = left; q < kList; ++q)
      to.keys[(size_t)at * kList + q] = kEmptyKey;
    const unsigned long long bound = from.bound[i];
    to.bound[at] = bound == kEmptyKey ? kEmptyKey
                                      : (bound & 0xffffffff00000000ull) |
                                            (unsigned int)newIndex[keyIndex(bound)];
  }
  if (left == 0) {
    const int place = atomicAdd(&st->searches, 1);
    searchRows[place] = (unsigned int)at | (j >= 0 ? 0x80000000u : 0u);
    searchOf[at] = place;
  } else {
    searchOf[at] = -1;
  }
  if (j >= 0) {
    const double *a = cur.c64 + (size_t)i * d, *b = cur.c64 + (size_t)j * d;
    double sq = 0.0;
    for (int f = 0; f < d; ++f) {
      const double diff = a[f] - b[f];
      sq = fma(diff, diff, sq);
    }
    const double si = cur.size[i], sj = cur.size[j];
    const int u = cur.rep[i], v = cur.rep[j];
    merges[atomicAdd(&st->merges, 1)] =
        DevMerge{min(u, v), max(u, v), sqrt(2.0 * (si * sj) / (si + sj) * sq)};
  }
}

// The first round's search: every slot, none of them new.
__global__ void searchAllKernel(int n, unsigned int *searchRows, int *searchOf,
                                unsigned long long *pushed, RoundState *st) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    searchRows[i] = (unsigned int)i;
    searchOf[i] = i;
    pushed[i] = kEmptyKey;
  }
  if (i == 0)
    st->searches = n;
}

// Lists from an exact pass that kept `per` lowest keys of every point: each
// list's bound is the last of them that it takes.
__global__ void listsFromKeysKernel(const unsigned long long *__restrict__ keys, int per, int n,
                                    Lists lists) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n)
    return;
  for (int q = 0; q < kList; ++q)
    lists.keys[(size_t)i * kList + q] = q < per ? keys[(size_t)i * per + q] : kEmptyKey;
  lists.bound[i] = keys[(size_t)i * per + min(per, kList) - 1];
}

// Minimum over the 16 lanes of a tile row, in all of them (DPP row rotations).
template <int CTRL> DEV unsigned long long rotateMin(unsigned long long v) {
  const unsigned int lo =
      (unsigned int)__builtin_amdgcn_update_dpp(-1, (int)(unsigned int)v, CTRL, 0xf, 0xf, false);
  const unsigned int hi = (unsigned int)__builtin_amdgcn_update_dpp(
      -1, (int)(unsigned int)(v >> 32), CTRL, 0xf, 0xf, false);
  return minKey(v, ((unsigned long long)hi << 32) | lo);
}
DEV unsigned long long rowMin16(unsigned long long v) {
  v = rotateMin<0x128>(v); // row_ror:8, 4, 2, 1
  v = rotateMin<0x124>(v);
  v = rotateMin<0x122>(v);
  return rotateMin<0x121>(v);
}

// The filter of PairFilter (distance.hip) for Ward: 2 si sj / (si + sj) >=
// min(si, sj), so a pair whose sq min(si, sj) is above the limit of a key's
// weight weighs more than the key.
DEV float wardLimit(unsigned long long key) {
  return key == kEmptyKey ? INFINITY : keyWeight(key) * (1.0f + 0x1p-20f) + FLT_MIN;
}

// Search rows against all m columns, in work items of a tile of rows and every
// splits-th column tile (128 points a side; 64 for few clusters: one tile's
// lists take longer than its distances, and more, smaller items share them). A row's kList lowest keys over an item's columns
// go to partial[place][split][kList]; a new cluster's weight goes to
// pushed[column] where it is below the column's bound.
template <int TR_, int FILL>
__global__ void __launch_bounds__(256, 3)
    wardSearchKernel(const float *__restrict__ C, int d, const int *__restrict__ size,
                     const unsigned int *__restrict__ searchRows, const int *__restrict__ searchOf,
                     const unsigned long long *__restrict__ bound, const RoundState *st,
                     const int *__restrict__ mNow, unsigned long long *__restrict__ partial,
                     unsigned long long *__restrict__ pushed) {
  using T = Tile<TR_, FILL, true>;
  constexpr int TR = T::TR, DIM = T::DIM;
  __shared__ __align__(16) TileSmem<T> sm;
  __shared__ unsigned long long top[DIM][kList];
  __shared__ int rowSlot[DIM];   // -1: no row
  __shared__ float rowSize[DIM];
  __shared__ unsigned char rowNew[DIM];
  __shared__ float colSize[DIM], colLimit[DIM]; // limit -inf: takes no offers
  __shared__ unsigned int colBits[DIM];
  if (roundOver(st))
    return;
  const int m = *mNow, rows = st->searches;
  const int rowTiles = (rows + DIM - 1) / DIM, colTiles = (m + DIM - 1) / DIM;
  const int splits = searchSplits(rows, m, DIM);
  const SqEuclidean metric;
  const int tid = threadIdx.x, lane = tid & 63;
  const unsigned long long groupMask = 0xffffull << (lane & 48);
  const int row4 = T::rowInTile(0), tc4 = 4 * T::tc();
  for (int item = blockIdx.x; item < rowTiles * splits; item += gridDim.x) {
    const int rowTile = item / splits, split = item - rowTile * splits;
    __syncthreads(); // the last item's LDS is consumed
    if (tid < DIM) {
      const int at = rowTile * DIM + tid;
      const unsigned int entry = at < rows ? searchRows[at] : 0u;
      const int slot = at < rows ? (int)(entry & 0x7fffffffu) : -1;
      rowSlot[tid] = slot;
      rowSize[tid] = slot >= 0 ? (float)size[slot] : 1.0f;
      rowNew[tid] = entry >> 31;
    }
    for (int i = tid; i < DIM * kList; i += T::THREADS)
      (&top[0][0])[i] = kEmptyKey;
    __syncthreads();
    bool first = true;
    // From the column tile nearest the first row's own, and around: where slots
    // are in spatial order the lists are tight from there on.
    const int count = (colTiles - split + splits - 1) / splits;
    const int start = min(count - 1, max(0, rowSlot[0] / DIM - split) / splits);
    for (int i = 0; i < count; ++i) {
      const int at = start + i < count ? start + i : start + i - count;
      const int col0 = (split + at * splits) * DIM;
      float acc[TR][TR];
#pragma unroll
      for (int r = 0; r < TR; ++r)
#pragma unroll
        for (int c = 0; c < TR; ++c)
          acc[r][c] = 0.0f;
      for (int f0 = 0; f0 < d; f0 += FILL) {
        const int nf8 = (min(FILL, d - f0) + 7) & ~7;
        // Rows of one fill stay in LDS for all of the item's tiles.
        if (first || d > FILL)
          for (int idx = tid; idx < DIM * nf8; idx += T::THREADS) {
            const int p = idx / nf8, k = idx - p * nf8, slot = rowSlot[p];
            sm.a[k][p] = slot >= 0 && f0 + k < d ? C[(size_t)slot * d + f0 + k] : 0.0f;
          }
        stageSlice<T>(sm.b, C, m, d, col0, f0, nf8);
        if (f0 == 0 && tid < DIM) {
          const int col = col0 + tid;
          const bool in = col < m;
          const unsigned long long b = in && searchOf[col] < 0 ? bound[col] : 0ull;
          colSize[tid] = in ? (float)size[col] : -1.0f;
          colLimit[tid] = in && searchOf[col] < 0 ? wardLimit(b) : -INFINITY;
          colBits[tid] = (unsigned int)(b >> 32);
        }
        __syncthreads();
        for (int k0 = 0; k0 < nf8; k0 += 8) {
#pragma unroll
          for (int kk = 0; kk < 8; ++kk) {
            const int k = k0 + kk;
            float av[TR], bv[TR];
#pragma unroll
            for (int h = 0; h < TR / 4; ++h) {
              const float4 a4 = *reinterpret_cast<const float4 *>(&sm.a[k][row4 + h * 16]);
              const float4 b4 = *reinterpret_cast<const float4 *>(&sm.b[k][h * 64 + tc4]);
              av[4 * h + 0] = a4.x; av[4 * h + 1] = a4.y; av[4 * h + 2] = a4.z; av[4 * h + 3] = a4.w;
              bv[4 * h + 0] = b4.x; bv[4 * h + 1] = b4.y; bv[4 * h + 2] = b4.z; bv[4 * h + 3] = b4.w;
            }
#pragma unroll
            for (int r = 0; r < TR; ++r)
#pragma unroll
              for (int c = 0; c < TR; ++c)
                acc[r][c] = metric.fold(acc[r][c], av[r], bv[c]);
          }
        }
        if (f0 + FILL < d)
          __syncthreads(); // the fill is consumed
      }
      float cs[TR], cl[TR];
#pragma unroll
      for (int c = 0; c < TR; ++c) {
        cs[c] = colSize[T::colInTile(c)];
        cl[c] = colLimit[T::colInTile(c)];
      }
#pragma unroll
      for (int r = 0; r < TR; ++r) {
        int i = T::rowInTile(r);
        asm volatile("" : "+v"(i)); // computed here, not kept for every row
        const int slot = rowSlot[i];
        const float rs = rowSize[i];
        unsigned long long *list = top[i];
        const unsigned long long last = list[kList - 1];
        const float limit = slot < 0 ? -INFINITY : wardLimit(last);
        const bool offers = rowNew[i];
        unsigned int pending = 0;
#pragma unroll
        for (int c = 0; c < TR; ++c) {
          const int col = col0 + T::colInTile(c);
          const float least = acc[r][c] * fminf(rs, cs[c]);
          if (!(least > fmaxf(limit, cl[c])) && cs[c] >= 0.0f && slot >= 0 && col != slot) {
            const bool forRow = !(least > limit), forCol = offers && !(least > cl[c]);
            const float w = (2.0f * (rs * cs[c])) / (rs + cs[c]) * acc[r][c];
            acc[r][c] = w;
            if (w != INFINITY) {
              if (forRow && packKey(w, (unsigned)col) < last)
                pending |= 1u << c;
              if (forCol && bitsOf(w) <= colBits[T::colInTile(c)])
                atomicMin(&pushed[col], packKey(w, (unsigned)slot));
            }
          }
        }
        if (first) {
          // Empty lists: the row's kList lowest, one after the other, from the
          // lowest of every lane.
#pragma unroll 1
          for (int q = 0; q < kList && __ballot(pending != 0) != 0; ++q) {
            unsigned long long mineLow = kEmptyKey;
#pragma unroll
            for (int c = 0; c < TR; ++c)
              if (pending >> c & 1)
                mineLow = minKey(mineLow, packKey(acc[r][c], (unsigned)(col0 + T::colInTile(c))));
            const unsigned long long low = rowMin16(mineLow);
            if (low == mineLow && low != kEmptyKey) {
#pragma unroll
              for (int c = 0; c < TR; ++c)
                if (col0 + T::colInTile(c) == keyIndex(low))
                  pending &= ~(1u << c);
            }
            if (T::tc() == 0)
              list[q] = low;
          }
        } else {
          // One insertion per row at a time, by its 16 lanes together.
          while (true) {
            const unsigned long long work = __ballot(pending != 0);
            if (work == 0)
              break;
            const unsigned long long mine = work & groupMask;
            const int source = mine ? __ffsll((long long)mine) - 1 : lane;
            const int c = __ffs(pending) - 1;
            float wv = 0.0f;
#pragma unroll
            for (int cc = 0; cc < TR; ++cc)
              if (cc == c)
                wv = acc[r][cc];
            const int colOf = c < 0 ? 0 : col0 + (c >> 2) * 64 + tc4 + (c & 3);
            if (lane == source)
              pending &= pending - 1;
            const unsigned long long key =
                packKey(__shfl(wv, source, 64), (unsigned int)__shfl(colOf, source, 64));
            const int q = lane & 15;
            if (mine && q < kList) {
              const unsigned long long cur = list[q], prev = q > 0 ? list[q - 1] : 0;
              if (cur > key)
                list[q] = prev > key ? prev : key;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (pending) {
              const unsigned long long now = list[kList - 1];
#pragma unroll
              for (int cc = 0; cc < TR; ++cc)
                if (!(packKey(acc[r][cc], (unsigned)(col0 + T::colInTile(cc))) < now))
                  pending &= ~(1u << cc);
            }
          }
        }
      }
      first = false;
      __syncthreads(); // the tile is consumed
    }
    for (int i = tid; i < DIM * kList; i += T::THREADS) {
      const int r = i / kList, at = rowTile * DIM + r;
      if (at < rows)
        partial[((size_t)at * splits + split) * kList + i % kList] = top[r][i % kList];
    }
  }
}

// The round's lists, 16 lanes per slot: a search row's from its parts (a lane
// merges every 16th part, then the lanes' lowest leave in order), another's
// with the lowest offer to it.
__global__ void __launch_bounds__(256)
    wardFinishKernel(Lists lists, const int *__restrict__ searchOf,
                     const unsigned long long *__restrict__ partial,
                     const unsigned long long *__restrict__ pushed,
                     const int *__restrict__ mNow, RoundState *st, int dim) {
  if (roundOver(st))
    return;
  const int m = *mNow, i = (int)((blockIdx.x * blockDim.x + threadIdx.x) / 16);
  if (i >= m)
    return;
  const int sub = threadIdx.x & 15;
  if (i == 0 && sub == 0)
    st->pairs += (unsigned long long)st->searches * (unsigned long long)m;
  unsigned long long *list = lists.keys + (size_t)i * kList;
  const int place = searchOf[i];
  unsigned long long key[kList];
  if (place >= 0) {
    const int splits = searchSplits(st->searches, m, dim);
    const unsigned long long *part = partial + (size_t)place * splits * kList;
#pragma unroll
    for (int q = 0; q < kList; ++q)
      key[q] = sub < splits ? part[sub * kList + q] : kEmptyKey;
    for (int s = sub + 16; s < splits; s += 16)
      for (int q = 0; q < kList; ++q) {
        unsigned long long k = part[s * kList + q];
        if (!(k < key[kList - 1]))
          break; // the part's keys ascend
#pragma unroll
        for (int p = 0; p < kList; ++p) {
          const unsigned long long cur = key[p];
          key[p] = minKey(cur, k);
          k = k < cur ? cur : k;
        }
      }
    unsigned long long low = kEmptyKey;
#pragma unroll
    for (int q = 0; q < kList; ++q) {
      low = rowMin16(key[0]);
      if (key[0] == low) {
#pragma unroll
        for (int p = 0; p + 1 < kList; ++p)
          key[p] = key[p + 1];
        key[kList - 1] = kEmptyKey;
      }
      if (sub == 0)
        list[q] = low;
    }
    if (sub == 0)
      lists.bound[i] = low; // every other key is above the last
  } else if (sub == 0) {
    const unsigned long long offer = pushed[i];
    if (!(offer < lists.bound[i]))
      return;
    int kept = 0;
#pragma unroll
    for (int q = 0; q < kList; ++q) {
      key[q] = list[q];
      kept += key[q] < offer;
    }
#pragma unroll
    for (int q = 0; q < kList; ++q)
      if (q >= kept)
        list[q] = q == kept ? offer : kEmptyKey;
    lists.bound[i] = offer; // what else was offered, or is beyond the list, is above it
  }
}

__global__ void roundStartKernel(RoundState *st, int n) {
  *st = RoundState{n, 0, 0, 0, 0, 0};
}

// Every point its own cluster; rep = its original index (orig, null: the
// position), comp = its slot.
__global__ void initClustersKernel(const float *X, int n, int d, Clusters c, int *comp,
                                   const int *orig) {
  const size_t total = (size_t)n * d;
  for (size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x; e < total;
       e += (size_t)gridDim.x * blockDim.x) {
    c.c64[e] = (double)X[e];
    c.c32[e] = X[e];
  }
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    c.size[i] = 1;
    c.rep[i] = orig ? orig[i] : i;
    comp[i] = i;
  }
}

// Condensed Ward distances between cluster centroids, in FP64 from the FP64
// centroids, stored as FP32.
__global__ void wardCondensedKernel(const double *c, const int *size, int m, int d, float *D) {
  const long long total = (long long)m * (m - 1) / 2;
  for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < total;
       t += (long long)gridDim.x * blockDim.x) {
    // row i from t: largest i with i*m - i*(i+1)/2 <= t
    const double mm = m;
    long long i = (long long)((2.0 * mm - 1.0 - sqrt((2.0 * mm - 1.0) * (2.0 * mm - 1.0) -
                                                     8.0 * (double)t)) * 0.5);
    if (i < 0)
      i = 0;
    while (i > 0 && i * m - i * (i + 1) / 2 > t)
      --i;
    while ((i + 1) * m - (i + 1) * (i + 2) / 2 <= t)
      ++i;
    const long long j = t - (i * m - i * (i + 1) / 2) + i + 1;
    double sq = 0.0;
    for (int f = 0; f < d; ++f) {
      const double diff = c[i * d + f] - c[j * d + f];
      sq = fma(diff, diff, sq);
    }
    const double si = size[i], sj = size[j];
    D[t] = (float)sqrt(2.0 * (si * sj) / (si + sj) * sq);
  }
}

bool wardMatrixFits(int m) {
  size_t freeBytes = 0, totalBytes = 0;
  if (hipMemGetInfo(&freeBytes, &totalBytes) != hipSuccess)
    return false;
  freeBytes += cachedDeviceBytes();
  return 4.0 * ((double)m * (m - 1) / 2) <= 0.9 * (double)freeBytes;
}

int denseTail(const Clusters &c, int m, int d, int n, std::vector<Edge> &merges) {
  DevArray<float> D;
  Status s;
  s(D.alloc((size_t)m * (m - 1) / 2));
  if (!s.ok())
    return s.code;
  hipLaunchKernelGGL(wardCondensedKernel, dim3(2048), dim3(256), 0, stream(), c.c64, c.size, m,
                     d, D.get());
  s((int)hipGetLastError());
  std::vector<double> tree((size_t)(m - 1) * 4);
  if (s.ok())
    s(denseLinkageOnCondensed(D, m, kWard, c.size, c.rep, n, tree.data()));
  if (!s.ok())
    return s.code;
  // Tree ids -> representative points: a new cluster is represented by the
  // representative of its first child.
  std::vector<int> repOfStep(m - 1);
  auto repOf = [&](double id, int step) {
    const int cl = (id >= 0 && id < n + step) ? (int)id : -1;
    return cl < n ? cl : repOfStep[cl - n];
  };
  for (int step = 0; step < m - 1; ++step) {
    const double *row = &tree[(size_t)step * 4];
    const int u = repOf(row[0], step), v = repOf(row[1], step);
    merges.push_back(Edge{std::min(u, v), std::max(u, v), row[2]});
    repOfStep[step] = u;
  }
  return 0;
}

int chainTail(const Clusters &c, int m, int d, std::vector<Edge> &merges) {
  std::vector<Edge> tail;
  int status = nnChainMerges(c.c64, c.size, m, d, tail);
  std::vector<int> rep(m);
  if (status == 0)
    status = download(rep.data(), c.rep, m * sizeof(int));
  if (status == 0)
    for (const Edge &e : tail) {
      const int u = rep[e.u], v = rep[e.v];
      merges.push_back(Edge{std::min(u, v), std::max(u, v), e.w});
    }
  return status;
}

// ---------------------------------------------------------------------------
// Nearest-neighbour chain (cooperative kernel)

struct ChainState {
  double *c; // m x d, slot s = centroid of the cluster in slot s
  int *size; // 0 = retired
  int *chain;
  int *ctl;  // [0] chain length, [1] current slot (-1 = done), [2] next start, [3] merges
  double *blockDist;
  int *blockIdx_;
  DevMerge *merges;
  int m, d;
  long long maxSteps;
};

struct DistIdx {
  double dist;
  int idx;
};

DEV bool lessDI(double d1, int i1, double d2, int i2) {
  return d1 < d2 || (d1 == d2 && i1 < i2);
}

template <int BS> DEV DistIdx blockMinDI(DistIdx v, DistIdx *red) {
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) {
    const double od = __shfl_xor(v.dist, m, 64);
    const int oi = __shfl_xor(v.idx, m, 64);
    if (lessDI(od, oi, v.dist, v.idx)) {
      v.dist = od;
      v.idx = oi;
    }
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0)
    red[threadIdx.x >> 6] = v;
  __syncthreads();
  DistIdx r = red[0];
  for (int w = 1; w < BS / 64; ++w)
    if (lessDI(red[w].dist, red[w].idx, r.dist, r.idx))
      r = red[w];
  __syncthreads();
  return r;
}

constexpr int kChainBlock = 256;

__global__ void __launch_bounds__(kChainBlock) nnChainKernel(ChainState st) {
  cg::grid_group grid = cg::this_grid();
  extern __shared__ double ca[]; // d doubles: the current slot's centroid
  __shared__ DistIdx red[kChainBlock / 64];
  __shared__ int shA, shPrev, shMerge;
  const int m = st.m, d = st.d;
  const int per = (m + gridDim.x - 1) / gridDim.x;
  const int first = blockIdx.x * per, last = min(m, first + per);

  for (long long step = 0; step < st.maxSteps; ++step) {
    if (threadIdx.x == 0) {
      shA = st.ctl[1];
      const int len = st.ctl[0];
      shPrev = len >= 2 ? st.chain[len - 2] : -1;
    }
    __syncthreads();
    const int a = shA, prev = shPrev;
    if (a < 0)
      return; // uniform: every workgroup read the same value after the barrier
    for (int k = threadIdx.x; k < d; k += kChainBlock)
      ca[k] = st.c[(size_t)a * d + k];
    __syncthreads();
    const double sa = st.size[a];
    DistIdx best{INFINITY, 0x7fffffff};
    for (int s = first + (int)threadIdx.x; s < last; s += kChainBlock) {
      const int ss = st.size[s];
      if (ss == 0 || s == a)
        continue;
      const double *cs = st.c + (size_t)s * d;
      double sq = 0.0;
      for (int f = 0; f < d; ++f) {
        const double diff = ca[f] - cs[f];
        sq = fma(diff, diff, sq);
      }
      const double w = 2.0 * (sa * ss) / (sa + ss) * sq;
      const int idx = s == prev ? -1 : s; // the previous chain element wins ties
      if (lessDI(w, idx, best.dist, best.idx)) {
        best.dist = w;
        best.idx = idx;
      }
    }
    best = blockMinDI<kChainBlock>(best, red);
    if (threadIdx.x == 0) {
      st.blockDist[blockIdx.x] = best.dist;
      st.blockIdx_[blockIdx.x] = best.idx;
    }
    grid.sync();
    if (blockIdx.x == 0) {
      DistIdx all{INFINITY, 0x7fffffff};
      for (int b = threadIdx.x; b < (int)gridDim.x; b += kChainBlock)
        if (lessDI(st.blockDist[b], st.blockIdx_[b], all.dist, all.idx)) {
          all.dist = st.blockDist[b];
          all.idx = st.blockIdx_[b];
        }
      all = blockMinDI<kChainBlock>(all, red);
      if (threadIdx.x == 0) {
        const int nearest = all.idx == -1 ? prev : all.idx;
        if (nearest == prev || nearest == 0x7fffffff) {
          shMerge = nearest == 0x7fffffff ? -2 : prev;
        } else {
          shMerge = -1;
          st.chain[st.ctl[0]++] = nearest;
          st.ctl[1] = nearest;
        }
      }
      __syncthreads();
      if (shMerge == -2) {
        if (threadIdx.x == 0)
          st.ctl[1] = -1; // no candidate (non-finite data): stop; the host reports it
      } else if (shMerge >= 0) {
        const int b = shMerge;
        const int keep = min(a, b), retire = max(a, b);
        const double sb = st.size[b];
        const double wb = sb / (sa + sb);
        for (int k = threadIdx.x; k < d; k += kChainBlock)
          st.c[(size_t)keep * d + k] = fma(st.c[(size_t)b * d + k] - ca[k], wb, ca[k]);
        if (threadIdx.x == 0) {
          st.merges[st.ctl[3]++] = DevMerge{keep, retire, sqrt(all.dist)};
          st.size[keep] = st.size[a] + st.size[b];
          st.size[retire] = 0;
          st.ctl[0] -= 2;
          if (st.ctl[3] == m - 1) {
            st.ctl[1] = -1;
          } else if (st.ctl[0] > 0) {
            st.ctl[1] = st.chain[st.ctl[0] - 1];
          } else {
            int start = st.ctl[2];
            while (start < m && st.size[start] == 0)
              ++start;
            st.ctl[2] = start;
            st.chain[0] = start;
            st.ctl[0] = 1;
            st.ctl[1] = start < m ? start : -1;
          }
        }
      }
    }
    grid.sync();
  }
}

} // namespace

int nnChainMerges(const double *centroids, const int *sizes, int m, int d,
                  std::vector<Edge> &merges) {
  merges.clear();
  if (m < 2)
    return 0;
  int coop = 0;
  (void)hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, 0);
  if (!coop)
    return (int)hipErrorNotSupported;
  const size_t smem = (size_t)d * sizeof(double);
  int perCU = 0;
  Status s;
  s((int)hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, nnChainKernel, kChainBlock, smem));
  if (!s.ok())
    return s.code;
  const int blocks = std::max(1, std::min(perCU * numCUs(), (m + kChainBlock - 1) / kChainBlock));
  ChainState st{};
  DevArray<double> c, blockDist;
  DevArray<int> size, chain, ctl, blockIdx;
  DevArray<DevMerge> dm;
  s(c.alloc((size_t)m * d));
  s(size.alloc(m));
  s(chain.alloc(m + 1));
  s(ctl.alloc(4));
  s(blockDist.alloc(blocks));
  s(blockIdx.alloc(blocks));
  s(dm.alloc(m - 1));
  if (!s.ok())
    return s.code;
  s((int)hipMemcpyAsync(c, centroids, (size_t)m * d * sizeof(double), hipMemcpyDeviceToDevice,
                        stream()));
  if (sizes) {
    s((int)hipMemcpyAsync(size, sizes, m * sizeof(int), hipMemcpyDeviceToDevice, stream()));
  } else {
    std::vector<int> ones(m, 1);
    s(upload(size, ones.data(), m * sizeof(int)));
  }
  const int ctl0[4] = {1, 0, 0, 0};
  const int zero = 0;
  s(upload(ctl, ctl0, sizeof(ctl0)));
  s(upload(chain, &zero, sizeof(int)));
  st.c = c;
  st.size = size;
  st.chain = chain;
  st.ctl = ctl;
  st.blockDist = blockDist;
  st.blockIdx_ = blockIdx;
  st.merges = dm;
  st.m = m;
  st.d = d;
  st.maxSteps = 3LL * m + 16; // each step pushes or merges; a chain never exceeds m
  if (s.ok()) {
    void *args[] = {&st};
    s((int)hipLaunchCooperativeKernel((const void *)nnChainKernel, dim3(blocks),
                                      dim3(kChainBlock), args, smem, stream()));
  }
  s(sync());
  int ctlOut[4] = {0, 0, 0, 0};
  s(download(ctlOut, ctl, sizeof(ctlOut)));
  std::vector<DevMerge> out(m - 1);
  s(download(out.data(), dm, (m - 1) * sizeof(DevMerge)));
  if (!s.ok())
    return s.code;
  const int count = std::min(ctlOut[3], m - 1);
  for (int i = 0; i < count; ++i)
    merges.push_back(Edge{out[i].u, out[i].v, out[i].h});
  return 0;
}

int nnChainWard(const float *X, int n, int d, double *tree) {
  if (n < 2)
    return 0;
  DevArray<double> c;
  Status s;
  s(c.alloc((size_t)n * d));
  if (!s.ok())
    return s.code;
  DevArray<float> c32;
  DevArray<int> size, rep, comp;
  s(c32.alloc((size_t)n * d));
  s(size.alloc(n));
  s(rep.alloc(n));
  s(comp.alloc(n));
  Clusters cl{c, c32, size, rep};
  hipLaunchKernelGGL(initClustersKernel, dim3(1024), dim3(256), 0, stream(), X, n, d, cl,
                     comp.get(), nullptr);
  std::vector<Edge> merges;
  if (s.ok())
    s(nnChainMerges(c, nullptr, n, d, merges));
  if (s.ok() && !mergesToTreeOrder(merges, n))
    s(kErrNonFinite);
  if (s.ok())
    treeFromOrderedMerges(merges, n, tree);
  return s.code;
}

int rnnWard(const float *X, int n, int d, const RnnOptions &opt, double *tree) {
  if (n < 2)
    return 0;
  DevArray<double> c64a, c64b;
  DevArray<float> c32a, c32b;
  DevArray<int> sizeA, sizeB, repA, repB, comp, partner, survives, newIndex, searchOf, roundEnds;
  DevArray<unsigned int> searchRows;
  DevArray<unsigned long long> keysA, keysB, boundA, boundB, partial, pushed;
  DevArray<unsigned char> scanTemp;
  DevArray<RoundState> state;
  DevArray<DevMerge> merges;
  Status s;
  const size_t nd = (size_t)n * d;
  s(c64a.alloc(nd));
  s(c64b.alloc(nd));
  s(c32a.alloc(nd));
  s(c32b.alloc(nd));
  s(sizeA.alloc(n));
  s(sizeB.alloc(n));
  s(repA.alloc(n));
  s(repB.alloc(n));
  s(comp.alloc(n));
  s(partner.alloc(n));
  s(survives.alloc((size_t)n + 1));
  s(newIndex.alloc((size_t)n + 1));
  s(searchOf.alloc(n));
  s(searchRows.alloc(n));
  s(keysA.alloc((size_t)n * kList));
  s(keysB.alloc((size_t)n * kList));
  s(boundA.alloc(n));
  s(boundB.alloc(n));
  s(pushed.alloc(n));
  // A search has at most kSearchItems items or one split: rows x splits <=
  // 128 kSearchItems, or the rows.
  s(partial.alloc(((size_t)128 * kSearchItems + n) * kList));
  s(scanTemp.alloc(scanTempBytes(n + 1)));
  s(state.alloc(1));
  s(roundEnds.alloc(n));
  s(merges.alloc(n - 1));
  if (!s.ok())
    return s.code;
  Clusters cur{c64a, c32a, sizeA, repA}, next{c64b, c32b, sizeB, repB};
  Lists lists{keysA, boundA}, listsNext{keysB, boundB};
  hipLaunchKernelGGL(initClustersKernel, dim3(1024), dim3(256), 0, stream(), X, n, d, cur,
                     comp.get(), opt.orig);
  hipLaunchKernelGGL(roundStartKernel, dim3(1), dim3(1), 0, stream(), state.get(), n);
  // Searches and their lists; count: the clusters, on the device, at most most.
  auto search = [&](const int *count, int most) {
    const int dim = most <= kSmallSearch ? 64 : 128;
    {
      PhaseTimer timer(kPhaseDistanceTiles);
      auto launch = [&](auto side, auto fill) {
        hipLaunchKernelGGL((wardSearchKernel<decltype(side)::value, decltype(fill)::value>),
                           dim3(kSearchGroups * numCUs()), dim3(256), 0, stream(), cur.c32, d,
                           cur.size, searchRows.get(), searchOf.get(), lists.bound, state.get(),
                           count, partial.get(), pushed.get());
      };
      using Four = std::integral_constant<int, 4>;
      using Eight = std::integral_constant<int, 8>;
      using Fill = std::integral_constant<int, 32>;
      if (dim == 64)
        d <= 8 ? launch(Four{}, Eight{}) : launch(Four{}, Fill{});
      else
        d <= 8 ? launch(Eight{}, Eight{}) : launch(Eight{}, Fill{});
    }
    PhaseTimer timer(kPhaseRnn);
    hipLaunchKernelGGL(wardFinishKernel, dim3((most + 15) / 16), dim3(256), 0, stream(), lists,
                       searchOf.get(), partial.get(), pushed.get(), count, state.get(), dim);
    return (int)hipGetLastError();
  };
  auto gridOf = [](long long count) { return dim3((unsigned)((count + 255) / 256)); };

  // A pruned pass (points in k-d order: merged clusters take the lower slot's
  // place in the compacted order, so slots stay spatially coherent and the
  // cluster tiles keep tight boxes) finds every cluster's nearest again: lists
  // of one key. It stops for good once a pass computes more than
  // kWardGiveUpShare of the tile pairs, and the searches go on from its lists.
  bool pruneThisPass = opt.prune;
  DevArray<unsigned long long> nearest;
  auto prunedPass = [&](int m) {
    Status st;
    if (!nearest.get())
      st(nearest.alloc(n));
    if (st.ok())
      st(fill(nearest, 0xff, m * sizeof(unsigned long long)));
    WeightSpec w;
    w.kind = kWeightWard;
    w.size = cur.size;
    double share = 1.0;
    if (st.ok())
      st(nearestOtherWalk(cur.c32, m, d, MetricSpec{kSqEuclidean, 2.0f}, w, comp, nullptr, nullptr,
                          nearest, &share, opt.stats));
    pruneThisPass = share <= kWardGiveUpShare;
    if (st.ok())
      hipLaunchKernelGGL(listsFromKeysKernel, gridOf(m), dim3(256), 0, stream(), nearest.get(), 1,
                         m, lists);
    st((int)hipGetLastError());
    return st.code;
  };

  // The first lists: from the mixed pass (every cluster is one point, size 1,
  // component = slot: the Ward weight 2 * 1 * 1 / (1 + 1) * sq is sq exactly,
  // and the pass keeps every point's lowest exact (FP32 squared distance, slot)
  // keys), from a pruned pass, or from a search of all rows.
  if (opt.mixedFirstPass) {
    int created = 0;
    s(nearest.alloc(n));
    MixedPass *mp = s.ok() ? mixedPassCreate(cur.c32, n, d, &created) : nullptr;
    s(created);
    if (mp) {
      s(fill(nearest, 0xff, n * sizeof(unsigned long long)));
      s(mixedPassRun(mp, comp, n, true, true, nearest));
      int per = 0;
      const unsigned long long *keys = mixedPassLists(mp, &per);
      if (s.ok())
        hipLaunchKernelGGL(listsFromKeysKernel, gridOf(n), dim3(256), 0, stream(), keys, per, n,
                           lists);
      s(sync()); // the pass's buffers are read
      mixedPassDestroy(mp);
    }
  } else if (opt.prune) {
    s(prunedPass(n));
  } else {
    hipLaunchKernelGGL(searchAllKernel, gridOf(n), dim3(256), 0, stream(), n, searchRows.get(),
                       searchOf.get(), pushed.get(), state.get());
    s(search(&state.get()->m, n));
  }
  s((int)hipGetLastError());

  RoundState host{n, 0, 0, 0, 0, 0};
  int queued = 0; // rounds queued so far
  enum { kNone, kDense, kChain } tail = kNone;
  while (s.ok() && host.m > 1) {
    if (opt.allowDense && host.m <= opt.denseBelow && wardMatrixFits(host.m)) {
      tail = kDense;
      break;
    }
    // Up to kRoundsAhead rounds, launched for the clusters that the last read
    // found; one at a time where a hand-over size is to be met, and while a
    // round's work outweighs its read by far and shrinks the next launches.
    const int ahead = opt.denseBelow > 0 || pruneThisPass ? 1
                      : host.m > 32768                    ? 2
                                                          : kRoundsAhead;
    const int most = host.m;
    for (int r = 0; r < ahead && s.ok(); ++r, ++queued) {
      const int *count = newIndex.get() + most; // survivors: the next count
      const bool small = most <= kSmallClusters;
      {
        PhaseTimer timer(kPhaseRnn);
        if (small) {
          hipLaunchKernelGGL(smallRoundKernel, dim3(1), dim3(kSmallThreads), 0, stream(), lists,
                             state.get(), most, r == 0, opt.minProgress, roundEnds.get(),
                             partner.get(), newIndex.get());
        } else {
          hipLaunchKernelGGL(survivorsKernel, gridOf(most + 1), dim3(256), 0, stream(), lists,
                             state.get(), most, partner.get(), survives.get());
          s(exclusiveScan(survives.get(), newIndex.get(), most + 1, scanTemp.get()));
        }
        const int slotBlocks = (most + 255) / 256;
        const int blocks = (int)std::min<long long>(2048, ((long long)most * d + 255) / 256);
        hipLaunchKernelGGL(rnnMergeKernel, dim3(slotBlocks + blocks), dim3(256), 0, stream(), cur,
                           next, lists, listsNext, partner.get(), newIndex.get(), d, state.get(),
                           merges.get(), searchRows.get(), searchOf.get(), pushed.get(),
                           slotBlocks);
      }
      std::swap(cur, next);
      std::swap(lists, listsNext);
      int now = 0;
      if (pruneThisPass)
        s(download(&now, count, sizeof(now)));
      s(pruneThisPass && now > 1 ? prunedPass(now) : search(count, most));
      if (!small || r + 1 == ahead) {
        PhaseTimer timer(kPhaseRnn);
        hipLaunchKernelGGL(roundEndKernel, dim3(1), dim3(1), 0, stream(), state.get(), count,
                           opt.minProgress, roundEnds.get());
      }
      s((int)hipGetLastError());
    }
    s(download(&host, state, sizeof(host)));
    if (s.ok() && host.stop && host.m > 1) {
      tail = opt.allowDense && wardMatrixFits(host.m) ? kDense : kChain;
      break;
    }
  }
  if (s.ok() && timingEnabled()) {
    RoundState end{};
    s(download(&end, state, sizeof(end)));
    addUnits(kPhaseDistanceTiles, (long long)end.pairs);
  }
  // Queued rounds after the last swapped the buffers for nothing.
  if ((queued - host.rounds) & 1)
    std::swap(cur, next);
  const int m = host.m, merged = host.merges;
  std::vector<int> roundEnd(host.rounds);
  std::vector<DevMerge> dm(merged);
  s(download(roundEnd.data(), roundEnds, roundEnd.size() * sizeof(int)));
  s(download(dm.data(), merges, merged * sizeof(DevMerge)));
  if (!s.ok())
    return s.code;
  std::vector<Edge> all(merged);
  for (int i = 0; i < merged; ++i)
    all[i] = Edge{dm[i].u, dm[i].v, dm[i].h};
  // Within a round merges arrive in atomic order; sort each round so the
  // result does not depend on scheduling. Rounds stay in order (children first).
  for (size_t r = 0; r < roundEnd.size(); ++r)
    std::sort(all.begin() + (r == 0 ? 0 : roundEnd[r - 1]), all.begin() + roundEnd[r], edgeLess);
  if (tail == kDense)
    s(denseTail(cur, m, d, n, all));
  else if (tail == kChain)
    s(chainTail(cur, m, d, all));
  if (s.ok() && !mergesToTreeOrder(all, n))
    s(kErrNonFinite);
  if (s.ok())
    treeFromOrderedMerges(all, n, tree);
  return s.code;
}

} // namespace cuhc

// Dense agglomerative clustering with Lance-Williams updates over a condensed
// distance matrix in HBM (reference src/linkage.cuh: the same linkages, FP64
// updates stored as FP32, lowest-slot ties; a different layout and loop).
//
// Layout: D(i, j), i < j, at i*n - i*(i+1)/2 + (j - i - 1): scipy's pdist order,
// n (n - 1) / 2 floats (20 GB at n = 100k). Slot s holds one active cluster;
// merging slots a < b puts the merged cluster in a and retires b. (A square
// matrix, whose merged rows are read in order, takes twice the memory and
// gives nothing: the update's reads fell from 312 to 97 ms at n = 100k, and
// writing the merged slots' columns rose from 29 to 190 ms.)
//
// Forward nearest cache: fn(i) = argmin over active j > i of (D(i, j), j). The
// closest pair (lowest distance, then lowest i, then lowest j) is
// (i*, fn(i*)) with i* the argmin over slots of (D(i, fn(i)), i). A merge
// changes D(a, k) for every k and retires b, so only rows k < b can need a new
// fn: rows with fn in {a, b} are rescanned unless the merged distance is still
// the row's minimum; row a's new fn is the minimum of its new distances.
//
// The merge loop is a cooperative persistent kernel (one workgroup per CU)
// that makes up to kMaxBatch merges per two grid barriers, or, where few merges
// of a batch stand, another that makes one per barrier (denseChainKernel).
// Workgroup g owns a contiguous range of slots (rows): their fn, size, bound
// and pending flag live in its LDS, it alone writes D(k, a) / D(a, k) for its
// rows k, and every workgroup keeps the active flags of all slots as a bitmask
// in LDS. A batch has two halves, each ended by a grid barrier:
//   A select:  every workgroup reads all records and takes the same batch: the
//              lowest pairs in (distance, row) order, up to the first that
//              touches a slot of an earlier one, that is not below every
//              pending row's lower bound, or that lies beyond the rows a
//              workgroup published. Rows left pending by the previous batch
//              are rescanned meanwhile, in column chunks shared by all waves.
//     update:  D(a_t, k) of every merge t of the batch for its own rows k,
//              each rounded as the one-at-a-time loop rounds it, kept in LDS;
//              it publishes, per merge, the smallest new distance and the two
//              lowest keys of its part of row a_t.
//   B commit:  from those, every workgroup finds the same valid prefix of the
//              batch: merge t stands if its distance is below every new
//              distance of the merges before it (then the one-at-a-time loop
//              picks it next; the first always stands). The workgroup writes
//              the prefix's distances of its rows and updates their fn and the
//              lower bound of their other keys. A row whose fn was a or b, and
//              whose new distance is not below that bound, is pending: the
//              bound now covers all its keys.
//     record:  its kTop lowest (distance, row) keys and fn columns, its lowest
//              pending bound and its pending rows.
// The merges, their order, ties and every rounding are those of merging the
// lowest (distance, i, j) pair one at a time. Neighbouring merges rarely touch
// each other: 12 of 16 stand per batch at n = 5,000, 14 at 12,000.
// Bound by latency (barriers and dependent memory round trips), so the batch
// divides it: see denseMergeKernel for the measured times.
// Per-workgroup records replace same-address atomics, which serialize across
// workgroups. The tree row is written on the device; there is no host round
// trip between merges.

#include "linkage.hpp"

#include <algorithm>

namespace cuhc {

namespace {

constexpr int kThreads = 512;
constexpr int kChunk = 8192;                     // columns per initial-scan work item
constexpr int kWaves = kThreads / 64;
constexpr int kRescanCols = 1024;                // columns per rescan work item (one wave)
constexpr int kRescanPer = kRescanCols / 64;
constexpr int kScanPer = 16;                     // columns per thread and step of a lone row's scan
constexpr int kMaxOwned = 2048;                  // rows per workgroup (LDS row state)
constexpr int kUpdatePer = 4;                    // owned rows per lane per load batch
constexpr int kMaxBatch = 16;                    // merges per batch
constexpr int kMinGroups = 8;                    // workgroups of the merge kernel at least
constexpr int kTop = 4;                          // lowest rows carried in a record
constexpr int kInlineRows = 6;                   // pending rows carried in a record
constexpr int kRecordWords = 12;                 // u64 words per workgroup record (96 bytes)
constexpr int kStepWords = 6;                    // the same of a single merge (48 bytes)
// A running average of the merges that stand per batch (the last 16 or so): the
// batch loop is left for single merges below kFewStand. Batches take 25 to 30 us
// and single merges 7 to 14 (n = 2,000 to 30,000). Runs of single merges start at
// kFirstRun and double while the batches between them make fewer merges than
// that; the average starts low after a run, so that the try is short.
constexpr float kFewStand = 2.0f, kFirstAverage = 4.0f, kNextAverage = 2.5f;
constexpr int kFirstRun = 256, kLongestRun = 4096;
constexpr int kGroup = 16;                       // workgroups per first-level barrier counter
constexpr int kLineWords = 32;                   // one 128-byte line in 32-bit words
constexpr unsigned int kSpinLimit = 1u << 22;    // barrier polls (seconds) before aborting

// Order-preserving map of a float to 32 bits (all non-NaN values), so that
// (distance, index) fits one u64 key without clamping negative distances.
HD unsigned int orderedBits(float f) {
  const unsigned int b = bitsOf(f);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
HD float fromOrderedBits(unsigned int o) {
  return floatOf((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
}
HD unsigned long long denseKey(float f, unsigned int idx) {
  return ((unsigned long long)orderedBits(f) << 32) | idx;
}

HD size_t condensedIndex(long long i, long long j, long long n) {
  // i < j
  return (size_t)(i * n - i * (i + 1) / 2 + (j - i - 1));
}

template <int LINKAGE>
DEV float lanceWilliams(float dakF, float dbkF, float dabF, int naI, int nbI, int nkI) {
  const double dak = dakF, dbk = dbkF, dab = dabF, na = naI, nb = nbI, nk = nkI;
  if constexpr (LINKAGE == kSingle) {
    return (float)fmin(dak, dbk);
  } else if constexpr (LINKAGE == kComplete) {
    return (float)fmax(dak, dbk);
  } else if constexpr (LINKAGE == kAverage) {
    return (float)((na * dak + nb * dbk) / (na + nb));
  } else {
    const double total = na + nb + nk;
    const double sq = ((na + nk) * dak * dak + (nb + nk) * dbk * dbk - nk * dab * dab) / total;
    return (float)sqrt(fmax(sq, 0.0));
  }
}

// Grid barrier for cooperatively launched (co-resident) workgroups: a
// two-level counter tree, kGroup workgroups per first-level counter and one
// root counter, each on its own line, and a generation word that the last
// arrival advances. No counter sees more than max(kGroup, groups) contending
// atomics. Counters only grow; the last arrival at a level is the one whose
// increment completes a multiple of that level's membership.
// Each wave waits for its own stores; one thread per workgroup then releases
// at agent scope (L2 write-back), arrives, polls the generation with relaxed
// loads (an acquire per poll would invalidate caches on every poll) and
// acquires once. A wait longer than kSpinLimit polls, or an abort word set by
// another workgroup, sets the abort word and returns false, so every
// workgroup leaves the loop.
struct Barrier {
  unsigned int *words; // [kLineWords * (3 + groups)]: generation, abort, groups, root
  int groups;
};

DEV unsigned int fetchAdd(unsigned int *p) {
  return __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

DEV bool gridBarrier(const Barrier &bar, unsigned int &generation, int *ok) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    ++generation;
    unsigned int *gen = bar.words;
    unsigned int *abortWord = bar.words + kLineWords;
    const int group = (int)blockIdx.x / kGroup;
    const unsigned int members = (unsigned int)min(kGroup, (int)gridDim.x - group * kGroup);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    const unsigned int old = fetchAdd(bar.words + kLineWords * (2 + group));
    if ((old + 1) % members == 0) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "agent");
      const unsigned int r = fetchAdd(bar.words + kLineWords * (2 + bar.groups));
      if ((r + 1) % (unsigned int)bar.groups == 0) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "agent");
        __hip_atomic_store(gen, generation, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    int result = 1;
    for (unsigned int polls = 0;; ++polls) {
      if (__hip_atomic_load(gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == generation)
        break;
      if ((polls & 63) == 63 &&
          (polls >= kSpinLimit ||
           __hip_atomic_load(abortWord, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
        __hip_atomic_store(abortWord, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        result = 0;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    *ok = result;
  }
  __syncthreads();
  return *ok != 0;
}

// At a kernel's start, before its first barrier: the generation that the last
// kernel left, and whether one of its waits gave up.
DEV unsigned int barrierGeneration(const Barrier &bar) {
  return __hip_atomic_load(bar.words, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
DEV bool barrierAborted(const Barrier &bar) {
  return __hip_atomic_load(bar.words + kLineWords, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
}

struct DenseState {
  float *D;
  int n;
  int firstNewId;
  int per;   // rows per workgroup
  int batch; // merges per batch (at most kMaxBatch)
  float average; // merges per batch that the batch loop starts from
  int *size; // cluster size and scipy id by slot
  int *id;
  // Per slot, [2][n]: the forward nearest key and the second lowest key of
  // the row, from denseInitKernel and, while a row is pending, from its rescan.
  // Between the kernels of the merge loop every row's, a pending one's nearest
  // empty and its bound in the other's place.
  unsigned long long *scanned;
  // One record per workgroup (kRecordWords words): [0..3] its kTop lowest
  // selection keys, [4..5] their fn columns, [6] the lowest lower-bound key of
  // its pending rows, [7] the number of its pending rows, [8..10] the first
  // kInlineRows of them (two per word); all of them in pendingRows[g per ...]
  // when there are more. Written in the second half of a batch and read in
  // the first half of the next, so a barrier lies between any write and read.
  unsigned long long *records;
  int *pendingRows;
  // Single merges: one record of kStepWords words per workgroup, in two buffers
  // that alternate by merge (a barrier lies between): its lowest selection key,
  // that key's column, the two lowest keys of its part of row a, and the lowest
  // lower-bound key of its pending rows.
  unsigned long long *steps; // [2][G][kStepWords]
  unsigned int *active;      // between the kernels: bit j = slot j active
  int *done;                 // between the kernels: merges made
  // Per merge of the batch and workgroup, [kMaxBatch][G]: the two lowest keys
  // of its part of row a, and the ordered bits of its smallest new distance.
  // Written in the first half, read in the second.
  unsigned long long *partFn, *partNext;
  unsigned int *partMin;
  int2 *items;                // initial fn: (row, first column) work items
  double *tree;               // (n - 1) x 4, device
  unsigned long long *clocks; // null, or [4]: device-clock ticks per part of a batch
  Barrier bar;
};

DEV unsigned long long blockMinKey(unsigned long long v, unsigned long long *red) {
#pragma unroll
  for (int m = 32; m > 0; m >>= 1)
    v = minKey(v, shflXorKey(v, m));
  const int wave = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0)
    red[wave] = v;
  __syncthreads();
  unsigned long long r = red[0];
  for (int w = 1; w < kThreads / 64; ++w)
    r = minKey(r, red[w]);
  return r;
}

// Keeps the two lowest keys of everything offered.
DEV void offer(unsigned long long &lowest, unsigned long long &next, unsigned long long key) {
  next = minKey(next, key < lowest ? lowest : key);
  lowest = minKey(lowest, key);
}

// Adds (lowest, next) of a part of a row to the row's two lowest keys: of the
// minima, every one but the last is displaced into next.
DEV void offerAtomic(unsigned long long *lowest, unsigned long long *next,
                     unsigned long long partLowest, unsigned long long partNext) {
  if (partLowest == kEmptyKey)
    return;
  const unsigned long long old = atomicMin(lowest, partLowest);
  const unsigned long long displaced = minKey(partNext, old < partLowest ? partLowest : old);
  if (displaced != kEmptyKey)
    atomicMin(next, displaced);
}

__global__ void __launch_bounds__(kThreads) denseInitKernel(DenseState s, int numItems) {
  __shared__ unsigned long long red[kThreads / 64];
  // Work item t: row r, chunk c, enumerated row by row (every slot is active).
  for (int t = blockIdx.x; t < numItems; t += gridDim.x) {
    const int2 it = s.items[t];
    const int j1 = min(s.n, it.y + kChunk);
    unsigned long long lowest = kEmptyKey, next = kEmptyKey;
    const size_t base = condensedIndex(it.x, it.x + 1, s.n) - (size_t)(it.x + 1);
    for (int j = it.y + (int)threadIdx.x; j < j1; j += kThreads)
      offer(lowest, next, denseKey(s.D[base + j], (unsigned)j));
    const unsigned long long k = blockMinKey(lowest, red);
    const unsigned long long k2 = blockMinKey(lowest == k ? next : lowest, red);
    if (threadIdx.x == 0)
      offerAtomic(&s.scanned[it.x], &s.scanned[s.n + it.x], k, k2);
  }
}

// Selection key of a row: (distance of its forward nearest, row).
DEV unsigned long long selectionKey(unsigned long long fn, int row) {
  return fn == kEmptyKey ? kEmptyKey : (fn & 0xffffffff00000000ull) | (unsigned int)row;
}

DEV bool isActive(const unsigned int *activeBits, int j) {
  return (activeBits[j >> 5] >> (j & 31)) & 1u;
}

// Wave-wide minima by DPP row shifts and broadcasts (lane 63 ends with the
// minimum; lanes without a source keep all ones): a step costs a few VALU
// instructions instead of an LDS permute's round trip.
template <int CTRL> DEV unsigned int dppMin(unsigned int v) {
  return min(v, (unsigned int)__builtin_amdgcn_update_dpp(-1, (int)v, CTRL, 0xf, 0xf, false));
}
template <int CTRL> DEV unsigned long long dppMin(unsigned long long v) {
  const unsigned int lo =
      (unsigned int)__builtin_amdgcn_update_dpp(-1, (int)(unsigned int)v, CTRL, 0xf, 0xf, false);
  const unsigned int hi = (unsigned int)__builtin_amdgcn_update_dpp(
      -1, (int)(unsigned int)(v >> 32), CTRL, 0xf, 0xf, false);
  return minKey(v, ((unsigned long long)hi << 32) | lo);
}
template <class V> DEV V dppMinAll(V v) {
  v = dppMin<0x111>(v); // row_shr:1, 2, 4, 8: lane 15 of each row
  v = dppMin<0x112>(v);
  v = dppMin<0x114>(v);
  v = dppMin<0x118>(v);
  v = dppMin<0x142>(v); // row_bcast:15, then 31
  return dppMin<0x143>(v);
}
DEV unsigned int waveMinBits(unsigned int v) {
  return (unsigned int)__builtin_amdgcn_readlane((int)dppMinAll(v), 63);
}
DEV unsigned long long waveMinKey(unsigned long long v) {
  v = dppMinAll(v);
  const unsigned int lo = (unsigned int)__builtin_amdgcn_readlane((int)(unsigned int)v, 63);
  const unsigned int hi = (unsigned int)__builtin_amdgcn_readlane((int)(unsigned int)(v >> 32), 63);
  return ((unsigned long long)hi << 32) | lo;
}

// The two lowest keys over the wave.
DEV void waveLowest2(unsigned long long &lowest, unsigned long long &next) {
  const unsigned long long low = waveMinKey(lowest);
  next = waveMinKey(lowest == low ? next : lowest); // keys are distinct, or empty
  lowest = low;
}

// LDS written by some lanes of a wave, then read by others of the same wave.
DEV void waveSync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Bound by latency: two grid barriers (2.7 us each) and a dozen dependent
// memory and LDS round trips per batch at small n; by the column reads
// (64-byte lines around scattered 4-byte entries) at large n. One merge per
// barrier took 14.0 us per merge at n = 5,003 and 15.8 us at n = 100,000;
// batches take 2.2 us (437 batches of 25 us) and 5.8 us.
// Where few merges of a batch stand it hands over to denseChainKernel; a form
// that limited its batches to one merge instead kept both barriers and halves.
// Keeping a bound below a row's other keys beside its fn (instead of its old
// fn as a pending row's bound) took n = 5,003 from 610 batches to 437: fewer
// selections meet a pending row. One instantiation per linkage, short loops
// left rolled: the batch's code should stay in the 64 KB instruction cache.
template <int LINKAGE>
__global__ void __launch_bounds__(kThreads) denseMergeKernel(DenseState s) {
  static_assert(kMaxBatch * kTop == 64, "the batch's candidates fill one wave");
  constexpr int kSorted = 32; // candidates examined in order, retired rows included
  // [0, (n + 31) / 32): bit j = slot j active; then the new distances
  // [batch][per] of the batch's merges to this workgroup's rows.
  extern __shared__ unsigned int dynamicLds[];
  // Per row: its fn, and a lower bound of its other keys (a pending row's fn
  // is not known: the bound covers all of its keys).
  __shared__ unsigned long long ownFn[kMaxOwned], ownNext[kMaxOwned];
  __shared__ int ownSize[kMaxOwned];
  // -1, or the row's part in the batch: t for slot a of merge t, kMaxBatch + t
  // for slot b.
  __shared__ signed char ownSlot[kMaxOwned];
  __shared__ unsigned char ownPending[kMaxOwned];
  __shared__ int pendRow[kMaxOwned]; // this workgroup's pending rows
  __shared__ int pendCount;
  // Every workgroup's pending rows: workgroup w's at [listStart[w], listStart[w + 1]).
  __shared__ int listStart[kThreads + 1];
  __shared__ int listRows[kInlineRows * kThreads];
  __shared__ __align__(16) unsigned long long heads[kThreads]; // lowest key per workgroup
  __shared__ int headRank[kThreads];
  __shared__ __align__(16) unsigned long long cand[64];
  __shared__ unsigned int candCol[64];
  __shared__ unsigned long long sorted[kSorted];
  __shared__ unsigned int sortedCol[kSorted];
  __shared__ int slotA[kMaxBatch], slotB[kMaxBatch], sizeA[kMaxBatch], sizeB[kMaxBatch];
  __shared__ int idA[kMaxBatch], idB[kMaxBatch];
  __shared__ float dist[kMaxBatch];
  __shared__ unsigned long long rowFn[kMaxBatch], rowNext[kMaxBatch];
  __shared__ unsigned int newMin[kMaxBatch];
  __shared__ int batchCount; // merges in the batch, or -1: no pair is left
  __shared__ unsigned long long waveKey[2 * kWaves];
  __shared__ int waveInt[2 * kWaves];
  __shared__ __align__(16) unsigned long long topKey[kWaves * kTop];
  __shared__ int barrierOk;

  const int n = s.n, per = s.per;
  const int G = gridDim.x, g = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int mine0 = min(n, g * per), mine1 = min(n, mine0 + per), rows = mine1 - mine0;
  const int words = (n + 31) >> 5;
  unsigned int *activeBits = dynamicLds;
  float *newDist = reinterpret_cast<float *>(dynamicLds + words);
  const int maxChunks = (n - 1 + kRescanCols - 1) / kRescanCols;
  const int rankers = kThreads / G, rankSpan = (G + rankers - 1) / rankers;
  int done = *s.done;
  if (done >= n - 1 || barrierAborted(s.bar))
    return;
  unsigned int generation = barrierGeneration(s.bar);
  const bool clocked = s.clocks && g == 0 && tid == 0;
  unsigned long long ticks[4] = {0, 0, 0, 0}, t0 = 0;
  auto lap = [&](int part) {
    if (clocked) {
      const unsigned long long t = wall_clock64();
      ticks[part] += t - t0;
      t0 = t;
    }
  };
  auto entry = [&](int i, int j) -> size_t {
    return i < j ? condensedIndex(i, j, n) : condensedIndex(j, i, n);
  };

  // This workgroup's kTop lowest settled rows, wave by wave (thread t looks
  // at rows t, t + kThreads, ...; keys are distinct, so the next lowest is the
  // lowest above the last).
  auto waveTop = [&]() {
    auto keyOf = [&](int r) {
      return r < rows && !ownPending[r] ? selectionKey(ownFn[r], mine0 + r) : kEmptyKey;
    };
    const unsigned long long first = keyOf(tid); // most workgroups own at most kThreads rows
    unsigned long long last = 0;
    for (int q = 0; q < kTop; ++q) {
      unsigned long long best = q == 0 || first > last ? first : kEmptyKey;
      for (int r = tid + kThreads; r < rows; r += kThreads) {
        const unsigned long long key = keyOf(r);
        if (q == 0 || key > last)
          best = minKey(best, key);
      }
      best = waveMinKey(best);
      if (lane == 0)
        topKey[wave * kTop + q] = best;
      last = best;
    }
  };
  // After a barrier behind waveTop: the record, by wave 0.
  auto writeRecord = [&]() {
    if (wave != 0)
      return;
    unsigned long long *rec = s.records + (size_t)g * kRecordWords;
    const unsigned long long key = lane < kWaves * kTop ? topKey[lane] : kEmptyKey;
    // A wave's keys are in order; only the waves that own rows have any.
    const int listed = min(kWaves, (rows + 63) / 64) * kTop;
    int rank = lane;
    if (listed > kTop) {
      rank = 0;
#pragma unroll 4
      for (int j = 0; j < listed; ++j) {
        const unsigned long long other = topKey[j];
        rank += other < key || (other == key && j < lane);
      }
      if (lane >= listed)
        rank = kTop;
    }
    if (rank < kTop) {
      rec[rank] = key;
      reinterpret_cast<unsigned int *>(rec + kTop)[rank] =
          key == kEmptyKey ? 0u : (unsigned int)ownFn[keyIndex(key) - mine0];
    }
    const int count = pendCount;
    unsigned long long bound = kEmptyKey;
    for (int i = lane; i < count; i += 64)
      bound = minKey(bound, selectionKey(ownNext[pendRow[i] - mine0], pendRow[i]));
    bound = waveMinKey(bound);
    if (lane == 0) {
      rec[6] = bound;
      rec[7] = (unsigned long long)count;
    }
    if (lane < kInlineRows / 2) {
      const int r0 = 2 * lane < count ? pendRow[2 * lane] : 0;
      const int r1 = 2 * lane + 1 < count ? pendRow[2 * lane + 1] : 0;
      rec[8 + lane] = (unsigned long long)(unsigned)r0 | ((unsigned long long)(unsigned)r1 << 32);
    }
  };
  // The q-th row of all pending rows (listStart ready).
  auto listRow = [&](int q, bool spilled) {
    if (!spilled)
      return listRows[q];
    int lo = 0, hi = G; // the w with listStart[w] <= q < listStart[w + 1]
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (listStart[mid] <= q)
        lo = mid;
      else
        hi = mid;
    }
    const int i = q - listStart[lo];
    if (listStart[lo + 1] - listStart[lo] > kInlineRows)
      return s.pendingRows[(size_t)lo * per + i];
    const unsigned long long w = s.records[(size_t)lo * kRecordWords + 8 + i / 2];
    return (int)(unsigned)(i & 1 ? w >> 32 : w);
  };

  for (int w = tid; w < words; w += kThreads)
    activeBits[w] = s.active[w];
  if (tid == 0)
    pendCount = 0;
  __syncthreads();
  for (int r = tid; r < rows; r += kThreads) {
    ownFn[r] = s.scanned[mine0 + r];
    ownNext[r] = s.scanned[n + mine0 + r];
    ownSize[r] = s.size[mine0 + r];
    ownSlot[r] = -1;
    const bool pending = ownFn[r] == kEmptyKey && ownNext[r] != kEmptyKey;
    ownPending[r] = pending;
    if (pending) {
      pendRow[atomicAdd(&pendCount, 1)] = mine0 + r;
      s.scanned[n + mine0 + r] = kEmptyKey;
    }
  }
  waveTop();
  __syncthreads();
  writeRecord();
  if (pendCount > kInlineRows)
    for (int i = tid; i < pendCount; i += kThreads)
      s.pendingRows[(size_t)g * per + i] = pendRow[i];
  if (!gridBarrier(s.bar, generation, &barrierOk))
    return;
  if (clocked)
    t0 = wall_clock64();

  float average = s.average; // merges that stand per batch
  bool leave = false;        // no more batches: pending rows settle, then the loop is left
  while (done < n - 1) {
    // ---- First half: select the batch.
    unsigned long long sel[kTop], bound = kEmptyKey;
    unsigned int col[kTop] = {};
    int cnt = 0;
    int inl[kInlineRows] = {};
#pragma unroll
    for (int q = 0; q < kTop; ++q)
      sel[q] = kEmptyKey;
    if (tid < G) {
      const ulonglong2 *r =
          reinterpret_cast<const ulonglong2 *>(s.records + (size_t)tid * kRecordWords);
      unsigned long long w[kRecordWords];
#pragma unroll
      for (int i = 0; i < kRecordWords / 2; ++i) {
        const ulonglong2 v = r[i];
        w[2 * i] = v.x;
        w[2 * i + 1] = v.y;
      }
#pragma unroll
      for (int q = 0; q < kTop; ++q) {
        sel[q] = w[q];
        col[q] = (unsigned)(w[kTop + q / 2] >> (32 * (q & 1)));
      }
      bound = w[6];
      cnt = (int)w[7];
#pragma unroll
      for (int i = 0; i < kInlineRows / 2; ++i) {
        inl[2 * i] = (int)(unsigned)w[8 + i];
        inl[2 * i + 1] = (int)(unsigned)(w[8 + i] >> 32);
      }
    }
    heads[tid] = sel[0];
    headRank[tid] = 0;
    if (tid < 64)
      cand[tid] = kEmptyKey;
    if (tid < kMaxBatch) {
      rowFn[tid] = kEmptyKey;
      rowNext[tid] = kEmptyKey;
      newMin[tid] = 0xffffffffu;
    }
    // A workgroup's rows beyond its kTop lowest are not listed: no key above
    // such a workgroup's last listed one may be taken.
    unsigned long long guard = waveMinKey(sel[kTop - 1]);
    bound = waveMinKey(bound);
    int incl = cnt;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(incl, d, 64);
      if (lane >= d)
        incl += v;
    }
    const bool spill = __ballot(cnt > kInlineRows) != 0;
    if (lane == 0) {
      waveKey[wave] = bound;
      waveKey[kWaves + wave] = guard;
      waveInt[kWaves + wave] = spill;
    }
    if (lane == 63)
      waveInt[wave] = incl;
    __syncthreads();
    int start = incl - cnt, listCount = 0;
    bool spilled = false;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      bound = minKey(bound, waveKey[w]);
      guard = minKey(guard, waveKey[kWaves + w]);
      start += w < wave ? waveInt[w] : 0;
      listCount += waveInt[w];
      spilled |= waveInt[kWaves + w] != 0;
    }
    if (tid < G) {
      listStart[tid] = start;
      if (!spilled)
        for (int i = 0; i < cnt; ++i)
          listRows[start + i] = inl[i];
    }
    if (tid == 0)
      listStart[G] = listCount;
    // The kMaxBatch lowest heads' workgroups hold the kMaxBatch lowest keys:
    // each head's rank, by kThreads / G threads per head.
    if (tid < rankers * G) {
      const int i = tid % G, lo = tid / G * rankSpan, hi = min(G, lo + rankSpan);
      const unsigned long long key = heads[i];
      int below = 0;
#pragma unroll 8
      for (int j = lo; j < hi; ++j)
        below += heads[j] < key;
      if (below)
        atomicAdd(&headRank[i], below);
    }
    auto take = [&](int at, int i, int j, unsigned long long key) {
      slotA[at] = i;
      slotB[at] = j;
      dist[at] = fromOrderedBits((unsigned)(key >> 32));
      if (i >= mine0 && i < mine1)
        ownSlot[i - mine0] = (signed char)at;
      if (j >= mine0 && j < mine1)
        ownSlot[j - mine0] = (signed char)(kMaxBatch + at);
    };
    __syncthreads();
    if (tid < G && sel[0] != kEmptyKey) {
      const int r = headRank[tid];
      if (r < kMaxBatch) {
#pragma unroll
        for (int q = 0; q < kTop; ++q) {
          cand[r * kTop + q] = sel[q];
          candCol[r * kTop + q] = col[q];
        }
      }
    }
    __syncthreads();
    if (wave == 0) {
      const unsigned long long key = cand[lane];
      // Nor any key above the last of the chosen heads: a workgroup that is
      // not among them may have a lower one.
      guard = minKey(guard, cand[(kMaxBatch - 1) * kTop]);
      int rank = 0;
#pragma unroll 8
      for (int j = 0; j < 64; ++j) {
        const unsigned int lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)key, j);
        const unsigned int hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(key >> 32), j);
        rank += (((unsigned long long)hi << 32) | lo) < key;
      }
      const int valid = min(kSorted, __popcll(__ballot(key != kEmptyKey)));
      if (key != kEmptyKey && rank < kSorted) {
        sorted[rank] = key;
        sortedCol[rank] = candCol[lane];
      }
      waveSync();
      // Lane t looks at the t-th lowest row. It ends the batch if its column
      // is a slot of an earlier pair of the batch; if the row itself is an
      // earlier pair's slot b, it retires with that merge and is passed over.
      const bool have = lane < valid;
      const unsigned long long k = have ? sorted[lane] : kEmptyKey;
      const int i = keyIndex(k), j = have ? (int)sortedCol[lane] : -1;
      unsigned long long stop = __ballot(!have || !(k < bound) || k > guard), retired = 0;
      for (int t = 0; !(stop >> t & 1); ++t) { // lane 63 always stops
        if (retired >> t & 1)
          continue;
        const int ti = __builtin_amdgcn_readlane(i, t), tj = __builtin_amdgcn_readlane(j, t);
        const unsigned long long after = ~1ull << t;
        stop |= (__ballot(j == ti) | __ballot(j == tj)) & after;
        retired |= __ballot(i == tj) & after;
      }
      const unsigned long long inMask = ((stop & -stop) - 1) & ~retired;
      const bool in = inMask >> lane & 1;
      const int at = __popcll(inMask & ((1ull << lane) - 1));
      const int limit = leave ? 0 : s.batch;
      if (in && at < limit)
        take(at, i, j, k);
      if (lane == 0)
        batchCount = valid == 0 && bound == kEmptyKey ? -1 : min(limit, __popcll(inMask));
    } else {
      // The pending rows are scanned again (no distance is written in this
      // half), one column chunk per wave and step.
      const unsigned int numItems = (unsigned)listCount * (unsigned)maxChunks;
      for (unsigned int t = (unsigned)((wave - 1) * G + g); t < numItems;
           t += (unsigned)((kWaves - 1) * G)) {
        const unsigned int q = t / (unsigned)maxChunks;
        const int r = listRow((int)q, spilled);
        const int j0 = r + 1 + (int)(t - q * (unsigned)maxChunks) * kRescanCols;
        if (j0 >= n)
          continue;
        const size_t base = condensedIndex(r, r + 1, n) - (size_t)(r + 1);
        float v[kRescanPer];
#pragma unroll
        for (int u = 0; u < kRescanPer; ++u) {
          const int j = j0 + lane + u * 64;
          v[u] = j < n ? s.D[base + j] : 0.0f;
        }
        unsigned long long lowest = kEmptyKey, next = kEmptyKey;
#pragma unroll
        for (int u = 0; u < kRescanPer; ++u) {
          const int j = j0 + lane + u * 64;
          if (j < n && isActive(activeBits, j))
            offer(lowest, next, denseKey(v[u], (unsigned)j));
        }
        waveLowest2(lowest, next);
        if (lane == 0)
          offerAtomic(&s.scanned[r], &s.scanned[n + r], lowest, next);
      }
    }
    __syncthreads();
    const int m = batchCount;
    if (m < 0) {
      // No pair (non-finite distances): the remaining rows report -1. Every
      // workgroup reduced the same records, so all of them stop here.
      if (g == 0)
        for (int r = done + tid; r < n - 1; r += kThreads)
          for (int c = 0; c < 4; ++c)
            s.tree[(size_t)r * 4 + c] = -1.0;
      done = n - 1;
      break;
    }
    const int numInstall = pendCount;
    lap(0);

    // The new distances of this workgroup's rows, a wave per merge.
    for (int t = wave; t < m; t += kWaves) {
      const int a = slotA[t], b = slotB[t];
      // The sizes (and, for the tree, the ids) arrive with the distances.
      const int na = s.size[a], nb = s.size[b];
      int ia = 0, ib = 0;
      if (g == 0) {
        ia = s.id[a];
        ib = s.id[b];
      }
      const float dab = dist[t];
      unsigned long long part = kEmptyKey, partNext = kEmptyKey;
      unsigned int lowest = 0xffffffffu;
      for (int base = lane; base < rows; base += 64 * kUpdatePer) {
        bool live[kUpdatePer];
        float dak[kUpdatePer], dbk[kUpdatePer];
#pragma unroll
        for (int u = 0; u < kUpdatePer; ++u) {
          const int r = base + 64 * u, k = mine0 + r;
          // Slot b of an earlier merge has retired by this one; slot a of an
          // earlier merge follows below.
          const int slot = r < rows ? ownSlot[r] : 0;
          live[u] = r < rows && k != a && k != b && isActive(activeBits, k) &&
                    !(slot >= 0 && (slot & (kMaxBatch - 1)) < t);
          if (live[u]) {
            dak[u] = s.D[entry(a, k)];
            dbk[u] = s.D[entry(b, k)];
          }
        }
#pragma unroll
        for (int u = 0; u < kUpdatePer; ++u) {
          if (!live[u])
            continue;
          const int r = base + 64 * u, k = mine0 + r;
          const float nd = lanceWilliams<LINKAGE>(dak[u], dbk[u], dab, na, nb, ownSize[r]);
          if (ownSlot[r] < 0 && k > a)
            offer(part, partNext, denseKey(nd, (unsigned)k));
          newDist[t * per + r] = nd;
          lowest = min(lowest, orderedBits(nd));
        }
      }
      waveLowest2(part, partNext);
      lowest = waveMinBits(lowest);
      if (lane == 0) {
        sizeA[t] = na;
        sizeB[t] = nb;
        idA[t] = ia;
        idB[t] = ib;
        atomicMin(&newMin[t], lowest);
        offerAtomic(&rowFn[t], &rowNext[t], part, partNext);
      }
    }
    // Pairs of merges u < t with slot a_u among this workgroup's rows: merge
    // u's distances to a_t and b_t first, then merge t's to a_u.
    if (tid < kMaxBatch * kMaxBatch) {
      const int t = tid / kMaxBatch, u = tid % kMaxBatch;
      const int k = u < t && t < m ? slotA[u] : -1;
      if (k >= mine0 && k < mine1) {
        const int a = slotA[t], b = slotB[t], kb = slotB[u];
        const int na = s.size[a], nb = s.size[b], ka = ownSize[k - mine0], kbSize = s.size[kb];
        const float aa = s.D[entry(k, a)], ab = s.D[entry(k, b)];
        const float ba = s.D[entry(kb, a)], bb = s.D[entry(kb, b)];
        const float xa = lanceWilliams<LINKAGE>(aa, ba, dist[u], ka, kbSize, na);
        const float xb = lanceWilliams<LINKAGE>(ab, bb, dist[u], ka, kbSize, nb);
        const float nd = lanceWilliams<LINKAGE>(xa, xb, dist[t], na, nb, ka + kbSize);
        newDist[t * per + k - mine0] = nd;
        atomicMin(&newMin[t], orderedBits(nd));
        offerAtomic(&rowFn[a < k ? t : u], &rowNext[a < k ? t : u],
                    denseKey(nd, (unsigned)max(a, k)), kEmptyKey);
      }
    }
    __syncthreads();
    if (tid < m) {
      s.partFn[tid * G + g] = rowFn[tid];
      s.partNext[tid * G + g] = rowNext[tid];
      s.partMin[tid * G + g] = newMin[tid];
    }
    lap(1);
    if (!gridBarrier(s.bar, generation, &barrierOk))
      return;
    lap(2);

    // ---- Second half: the valid prefix, committed.
    if (tid == 0)
      pendCount = 0;
    // Every load of the half's start is issued before the first is used.
    const int installRow = tid < numInstall ? pendRow[tid] : -1;
    const unsigned long long installFn = installRow >= 0 ? s.scanned[installRow] : kEmptyKey;
    const unsigned long long installNext =
        installRow >= 0 ? s.scanned[n + installRow] : kEmptyKey;
    constexpr int kPerWave = kMaxBatch / kWaves;
    unsigned long long fn[kPerWave], next[kPerWave];
    unsigned int lowest[kPerWave];
#pragma unroll
    for (int p = 0; p < kPerWave; ++p) {
      fn[p] = kEmptyKey;
      next[p] = kEmptyKey;
      lowest[p] = 0xffffffffu;
    }
    for (int w0 = lane; w0 < G; w0 += 256) {
      unsigned long long f[kPerWave][4], x[kPerWave][4];
      unsigned int l[kPerWave][4];
#pragma unroll
      for (int p = 0; p < kPerWave; ++p)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int t = wave + p * kWaves, w = w0 + 64 * u;
          const bool in = t < m && w < G;
          f[p][u] = in ? s.partFn[t * G + w] : kEmptyKey;
          x[p][u] = in ? s.partNext[t * G + w] : kEmptyKey;
          l[p][u] = in ? s.partMin[t * G + w] : 0xffffffffu;
        }
#pragma unroll
      for (int p = 0; p < kPerWave; ++p)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          offer(fn[p], next[p], f[p][u]);
          next[p] = minKey(next[p], x[p][u]);
          lowest[p] = min(lowest[p], l[p][u]);
        }
    }
#pragma unroll
    for (int p = 0; p < kPerWave; ++p) {
      if (wave + p * kWaves >= m)
        break;
      waveLowest2(fn[p], next[p]);
      lowest[p] = waveMinBits(lowest[p]);
      if (lane == 0) {
        rowFn[wave + p * kWaves] = fn[p];
        rowNext[wave + p * kWaves] = next[p];
        newMin[wave + p * kWaves] = lowest[p];
      }
    }
    // Rows rescanned in the first half settle.
    if (installRow >= 0) {
      ownPending[installRow - mine0] = 0;
      ownFn[installRow - mine0] = installFn;
      ownNext[installRow - mine0] = installNext;
    }
    for (int i = kThreads + tid; i < numInstall; i += kThreads) {
      const int r = pendRow[i];
      ownPending[r - mine0] = 0;
      ownFn[r - mine0] = s.scanned[r];
      ownNext[r - mine0] = s.scanned[n + r];
    }
    __syncthreads();
    // Merge t stands if it is below every new distance of the merges before
    // it: lane t compares it with the minimum over lanes < t.
    int valid = m;
    unsigned int least = newMin[0]; // the smallest new distance of the batch
    if (m > 1) {
      unsigned int before = lane < m ? newMin[lane] : 0xffffffffu;
      const unsigned int own = lane < m ? orderedBits(dist[lane]) : 0xffffffffu;
#pragma unroll
      for (int d = 1; d < kMaxBatch; d <<= 1) {
        const unsigned int v = __shfl_up(before, d, 64);
        if (lane >= d)
          before = min(before, v);
      }
      least = (unsigned int)__builtin_amdgcn_readlane((int)before, kMaxBatch - 1);
      before = __shfl_up(before, 1, 64);
      const unsigned long long cut = __ballot(lane >= m || (lane > 0 && !(own < before)));
      valid = __ffsll((long long)cut) - 1; // m <= 16: lane 63 is cut
    }
    if (leave) // every row is settled
      break;
    const bool whole = valid == m;
    if (m > 0) {
      average += ((float)valid - average) * (1.0f / 16);
      leave = average < kFewStand;
    }
    int slotsA[kMaxBatch], slotsB[kMaxBatch]; // uniform
    {
      const int laneA = lane < m ? slotA[lane] : 0, laneB = lane < m ? slotB[lane] : 0;
#pragma unroll
      for (int t = 0; t < kMaxBatch; ++t) {
        slotsA[t] = __builtin_amdgcn_readlane(laneA, t);
        slotsB[t] = __builtin_amdgcn_readlane(laneB, t);
      }
    }
    for (int t = wave; t < valid; t += kWaves) {
      const int a = slotA[t], b = slotB[t];
      for (int r = lane; r < rows; r += 64) {
        const int k = mine0 + r, slot = ownSlot[r];
        if (k == a || k == b || !isActive(activeBits, k))
          continue;
        // Entries of slots that retire in the prefix are dead; entries
        // between two merged slots are written for the later merge.
        if (slot >= kMaxBatch ? slot - kMaxBatch < valid : slot > t && slot < valid)
          continue;
        s.D[entry(a, k)] = newDist[t * per + r];
      }
    }
    for (int r = tid; r < rows; r += kThreads) {
      const int k = mine0 + r, slot = ownSlot[r];
      if (!isActive(activeBits, k))
        continue;
      if (slot >= kMaxBatch && slot - kMaxBatch < valid) {
        ownFn[r] = kEmptyKey; // retired
        ownPending[r] = 0;
        continue;
      }
      unsigned long long f = ownFn[r], other = ownNext[r];
      bool rescan = false;
      if (slot >= 0 && slot < kMaxBatch && slot < valid) {
        const int size = sizeA[slot] + sizeB[slot];
        ownSize[r] = size;
        s.size[k] = size;
        // A cut batch: the parts leave out slots that stay, so the row is
        // scanned again; no new distance of the batch is below the bound.
        f = rowFn[slot];
        other = rowNext[slot];
        if (!whole) {
          rescan = true;
          other = (unsigned long long)least << 32;
        }
      } else {
        // The merges that change this row's two lowest: those that take its
        // nearest, and those whose new distance is below its bound (only the
        // columns a > k and b > k are this row's).
        float nd[kMaxBatch];
#pragma unroll
        for (int t = 0; t < kMaxBatch; ++t)
          nd[t] = t < valid ? newDist[t * per + r] : 0.0f;
        const int fk = f == kEmptyKey ? -1 : keyIndex(f);
        const unsigned int otherBits = (unsigned)(other >> 32);
        unsigned int changes = 0;
#pragma unroll
        for (int t = 0; t < kMaxBatch; ++t) {
          const bool change = slotsA[t] == fk || slotsB[t] == fk ||
                              (k < slotsA[t] && orderedBits(nd[t]) <= otherBits);
          changes |= change && t < valid ? 1u << t : 0u;
        }
        for (; changes; changes &= changes - 1) {
          const int t = __ffs(changes) - 1, a = slotA[t], b = slotB[t];
          const unsigned long long c =
              k < a ? denseKey(newDist[t * per + r], (unsigned)a) : kEmptyKey;
          const int at = f == kEmptyKey ? -1 : keyIndex(f);
          if (rescan) {
            other = minKey(other, c);
          } else if (at == a || at == b) {
            // Its nearest is gone: the new distance replaces it if it is
            // below all others; with no others, none is left.
            if (c < other || other == kEmptyKey)
              f = c;
            else
              rescan = true;
          } else {
            offer(f, other, c);
          }
        }
      }
      if (rescan) {
        const int at = atomicAdd(&pendCount, 1);
        pendRow[at] = k;
        ownPending[r] = 1;
        s.scanned[k] = kEmptyKey;
        s.scanned[n + k] = kEmptyKey;
      }
      ownFn[r] = f;
      ownNext[r] = other;
    }
    waveTop();
    __syncthreads();
    writeRecord();
    if (tid >= 64 && tid < 64 + m) {
      const int t = tid - 64, a = slotA[t], b = slotB[t];
      if (t < valid)
        atomicAnd(&activeBits[b >> 5], ~(1u << (b & 31)));
      if (a >= mine0 && a < mine1)
        ownSlot[a - mine0] = -1;
      if (b >= mine0 && b < mine1)
        ownSlot[b - mine0] = -1;
      if (g == 0 && t < valid) {
        double *row = s.tree + (size_t)(done + t) * 4;
        row[0] = (double)min(idA[t], idB[t]);
        row[1] = (double)max(idA[t], idB[t]);
        row[2] = (double)dist[t];
        row[3] = (double)(sizeA[t] + sizeB[t]);
        s.id[a] = s.firstNewId + done + t;
      }
    }
    if (pendCount > kInlineRows)
      for (int i = tid; i < pendCount; i += kThreads)
        s.pendingRows[(size_t)g * per + i] = pendRow[i];
    done += valid;
    lap(3);
    if (!gridBarrier(s.bar, generation, &barrierOk))
      return;
    lap(2);
  }
  // The state of the loop, for a run of single merges.
  for (int r = tid; r < rows; r += kThreads) {
    s.scanned[mine0 + r] = ownFn[r];
    s.scanned[n + mine0 + r] = ownFn[r] == kEmptyKey ? kEmptyKey : ownNext[r];
  }
  if (g == 0)
    for (int w = tid; w < words; w += kThreads)
      s.active[w] = activeBits[w];
  if (g == 0 && tid == 0)
    *s.done = done;
  if (clocked)
    for (int i = 0; i < 4; ++i)
      s.clocks[i] += ticks[i];
}

// A run of merges made one at a time, one grid barrier each: for chains, where
// every merge takes in the cluster just made or ties with the next (duplicates),
// so that a batch keeps its first merge only. A merge is committed in the phase
// that computes its distances; row a's new nearest is known in the next phase,
// from every workgroup's part of the row. A row that loses its nearest is
// pending, its other keys' bound below all of its keys, and is scanned again,
// by its own workgroup, only when no settled row's key is below that bound: in
// a chain of single linkage such a row is nearer to the grown cluster and joins
// it before. (Scanned at once, chains of 30,000 points took up to 33 us per
// merge, of 100,000 41.)
// Bound by latency, as the batches: one barrier and three dependent round trips
// per merge. Chains of single linkage took 25 us per merge as batches of one (n =
// 30,000; 16 at 2,000), two barriers each, and 14 in a loop of this kind that
// scanned rows over all workgroups in the next phase; now 7 (n = 2,000) to 11.5.
template <int LINKAGE>
__global__ void __launch_bounds__(kThreads) denseChainKernel(DenseState s, int run) {
  extern __shared__ unsigned int activeBits[]; // [(n + 31) / 32]
  // Per row, as in the batch loop; a pending row's fn is empty, its next a bound
  // below all of its keys. Both are empty for a row that has none.
  __shared__ unsigned long long ownFn[kMaxOwned], ownNext[kMaxOwned];
  __shared__ int ownSize[kMaxOwned];
  __shared__ int scanRow[kMaxOwned]; // rows to scan again
  __shared__ int scanCount;
  // Per wave: lowest key, its column, the two lowest of row a's part, bound.
  __shared__ unsigned long long inKey[kWaves], inFn[kWaves], inNext[kWaves], inBound[kWaves];
  __shared__ unsigned int inCol[kWaves];
  __shared__ unsigned long long outKey[kWaves], outFn[kWaves], outNext[kWaves], outBound[kWaves];
  __shared__ unsigned int outCol[kWaves];
  __shared__ int barrierOk;

  const int n = s.n, per = s.per;
  const int G = gridDim.x, g = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int mine0 = min(n, g * per), mine1 = min(n, mine0 + per), rows = mine1 - mine0;
  const int words = (n + 31) >> 5;
  int done = *s.done;
  if (done >= n - 1 || barrierAborted(s.bar))
    return;
  const int until = min(n - 1, done + run);
  unsigned int generation = barrierGeneration(s.bar);
  const bool clocked = s.clocks && g == 0 && tid == 0;
  unsigned long long ticks[4] = {0, 0, 0, 0}, t0 = clocked ? wall_clock64() : 0;
  auto lap = [&](int part) {
    if (clocked) {
      const unsigned long long t = wall_clock64();
      ticks[part] += t - t0;
      t0 = t;
    }
  };
  auto entry = [&](int i, int j) -> size_t {
    return i < j ? condensedIndex(i, j, n) : condensedIndex(j, i, n);
  };
  for (int w = tid; w < words; w += kThreads)
    activeBits[w] = s.active[w];
  // A thread holds rows tid, tid + kThreads, ...: only it touches their state.
  // key, col and bound: over its rows, the lowest settled key, its column, and
  // the lowest bound of a pending row.
  unsigned long long key = kEmptyKey, bound = kEmptyKey;
  unsigned int col = 0;
  auto note = [&](int r) {
    const unsigned long long f = ownFn[r];
    const unsigned long long k = selectionKey(f == kEmptyKey ? ownNext[r] : f, mine0 + r);
    if (f == kEmptyKey) {
      bound = minKey(bound, k);
    } else if (k < key) {
      key = k;
      col = keyIndex(f);
    }
  };
  for (int r = tid; r < rows; r += kThreads) {
    ownFn[r] = s.scanned[mine0 + r];
    ownNext[r] = s.scanned[n + mine0 + r];
    ownSize[r] = s.size[mine0 + r];
    note(r);
  }
  if (tid == 0)
    scanCount = 0;
  // The workgroup's record: the waves' results through LDS, by wave 0.
  auto publish = [&](unsigned long long part, unsigned long long partNext, int buffer) {
    unsigned long long low = waveMinKey(key), least = waveMinKey(bound);
    waveLowest2(part, partNext);
    if (low != kEmptyKey ? key == low : lane == 0) { // keys are distinct
      outKey[wave] = low;
      outCol[wave] = col;
      outFn[wave] = part;
      outNext[wave] = partNext;
      outBound[wave] = least;
    }
    lap(1);
    __syncthreads();
    if (wave != 0)
      return;
    const unsigned long long k = lane < kWaves ? outKey[lane] : kEmptyKey;
    part = lane < kWaves ? outFn[lane] : kEmptyKey;
    partNext = lane < kWaves ? outNext[lane] : kEmptyKey;
    least = waveMinKey(lane < kWaves ? outBound[lane] : kEmptyKey);
    low = waveMinKey(k);
    waveLowest2(part, partNext);
    if (low != kEmptyKey ? k == low : lane == 0) {
      ulonglong2 *r = reinterpret_cast<ulonglong2 *>(s.steps + ((size_t)buffer * G + g) * kStepWords);
      r[0] = make_ulonglong2(low, (unsigned long long)outCol[lane]);
      r[1] = make_ulonglong2(part, partNext);
      r[2] = make_ulonglong2(least, 0);
    }
  };
  publish(kEmptyKey, kEmptyKey, 0);
  if (!gridBarrier(s.bar, generation, &barrierOk))
    return;
  lap(2);

  int prevA = -1, prevSize = 0;
  for (int buffer = 0;; buffer ^= 1) {
    // The lowest pair, and the previous merge's row from its parts.
    unsigned long long fn = kEmptyKey, next = kEmptyKey;
    key = bound = kEmptyKey;
    if (tid < G) {
      const ulonglong2 *r =
          reinterpret_cast<const ulonglong2 *>(s.steps + ((size_t)buffer * G + tid) * kStepWords);
      const ulonglong2 v = r[0], part = r[1];
      bound = r[2].x;
      key = v.x;
      col = (unsigned)v.y;
      fn = part.x;
      next = part.y;
    }
    unsigned long long low = waveMinKey(key), least = waveMinKey(bound);
    waveLowest2(fn, next);
    if (low != kEmptyKey ? key == low : lane == 0) {
      inKey[wave] = low;
      inCol[wave] = col;
      inFn[wave] = fn;
      inNext[wave] = next;
      inBound[wave] = least;
    }
    __syncthreads();
    low = least = fn = next = kEmptyKey;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      if (inKey[w] < low) {
        low = inKey[w];
        col = inCol[w];
      }
      least = minKey(least, inBound[w]);
      offer(fn, next, inFn[w]);
      next = minKey(next, inNext[w]);
    }
    if (prevA >= mine0 && prevA < mine1 && (prevA - mine0) % kThreads == tid) {
      ownFn[prevA - mine0] = fn;
      ownNext[prevA - mine0] = next;
      ownSize[prevA - mine0] = prevSize;
      s.size[prevA] = prevSize;
    }
    if (done == until)
      break;
    if (prevA >= 0 && selectionKey(fn, prevA) < low) {
      low = selectionKey(fn, prevA);
      col = keyIndex(fn);
    }
    if (least != kEmptyKey && !(low < least)) {
      // A pending row may hold the lowest key: those whose bound is not above it
      // are scanned, and the records published again.
      for (int r = tid; r < rows; r += kThreads)
        if (ownFn[r] == kEmptyKey && ownNext[r] != kEmptyKey &&
            selectionKey(ownNext[r], mine0 + r) <= low)
          scanRow[atomicAdd(&scanCount, 1)] = r;
      __syncthreads();
      const int scans = scanCount;
      for (int i = 0; i < scans; ++i) {
        const int r = scanRow[i], k = mine0 + r;
        const size_t base = condensedIndex(k, k + 1, n) - (size_t)(k + 1);
        unsigned long long lowest = kEmptyKey, second = kEmptyKey;
        for (int j0 = k + 1; j0 < n; j0 += kThreads * kScanPer) {
          float v[kScanPer];
#pragma unroll
          for (int u = 0; u < kScanPer; ++u) {
            const int j = j0 + tid + u * kThreads;
            v[u] = j < n ? s.D[base + j] : 0.0f;
          }
#pragma unroll
          for (int u = 0; u < kScanPer; ++u) {
            const int j = j0 + tid + u * kThreads;
            if (j < n && isActive(activeBits, j))
              offer(lowest, second, denseKey(v[u], (unsigned)j));
          }
        }
        waveLowest2(lowest, second);
        if (lane == 0) {
          outFn[wave] = lowest;
          outNext[wave] = second;
        }
        __syncthreads();
        if (r % kThreads == tid) {
          lowest = second = kEmptyKey;
          for (int w = 0; w < kWaves; ++w) {
            offer(lowest, second, outFn[w]);
            second = minKey(second, outNext[w]);
          }
          ownFn[r] = lowest;
          ownNext[r] = second;
        }
        __syncthreads(); // outFn is written again
      }
      if (tid == 0)
        scanCount = 0;
      key = bound = kEmptyKey;
      for (int r = tid; r < rows; r += kThreads)
        note(r);
      prevA = -1;
      publish(kEmptyKey, kEmptyKey, buffer ^ 1);
      lap(3);
      if (!gridBarrier(s.bar, generation, &barrierOk))
        return;
      lap(2);
      continue;
    }
    if (low == kEmptyKey) {
      // No pair (non-finite distances): the remaining rows report -1, as in the
      // batch loop.
      if (g == 0)
        for (int r = done + tid; r < n - 1; r += kThreads)
          for (int c = 0; c < 4; ++c)
            s.tree[(size_t)r * 4 + c] = -1.0;
      done = n - 1;
      break;
    }
    const int a = keyIndex(low), b = (int)col;
    const float dab = fromOrderedBits((unsigned)(low >> 32));
    // The previous merge's size is on its way to memory.
    const int na = a == prevA ? prevSize : s.size[a];
    const int nb = b == prevA ? prevSize : s.size[b];
    lap(0);

    unsigned long long part = kEmptyKey, partNext = kEmptyKey;
    key = bound = kEmptyKey;
    for (int r = tid; r < rows; r += kThreads) {
      const int k = mine0 + r;
      if (!isActive(activeBits, k))
        continue;
      if (k == a || k == b) { // b retires; a's nearest is known in the next phase
        ownFn[r] = kEmptyKey;
        ownNext[r] = kEmptyKey;
        continue;
      }
      const float dak = s.D[entry(a, k)], dbk = s.D[entry(b, k)];
      const float nd = lanceWilliams<LINKAGE>(dak, dbk, dab, na, nb, ownSize[r]);
      s.D[entry(a, k)] = nd;
      const unsigned long long c = k < a ? denseKey(nd, (unsigned)a) : kEmptyKey;
      if (k > a)
        offer(part, partNext, denseKey(nd, (unsigned)k));
      unsigned long long f = ownFn[r], other = ownNext[r];
      const int at = f == kEmptyKey ? -1 : keyIndex(f);
      if (f == kEmptyKey || at == a || at == b) // pending, or its nearest is gone
        f = c < other ? c : kEmptyKey;
      else
        offer(f, other, c);
      ownFn[r] = f;
      ownNext[r] = other;
      note(r);
    }
    publish(part, partNext, buffer ^ 1);
    if (tid == 0) {
      activeBits[b >> 5] &= ~(1u << (b & 31));
      if (g == 0) {
        double *row = s.tree + (size_t)done * 4;
        const int ia = s.id[a], ib = s.id[b];
        row[0] = (double)min(ia, ib);
        row[1] = (double)max(ia, ib);
        row[2] = (double)dab;
        row[3] = (double)(na + nb);
        s.id[a] = s.firstNewId + done;
      }
    }
    prevA = a;
    prevSize = na + nb;
    ++done;
    lap(3);
    if (!gridBarrier(s.bar, generation, &barrierOk))
      return;
    lap(2);
  }
  for (int r = tid; r < rows; r += kThreads) {
    s.scanned[mine0 + r] = ownFn[r];
    s.scanned[n + mine0 + r] = ownNext[r];
  }
  if (g == 0)
    for (int w = tid; w < words; w += kThreads)
      s.active[w] = activeBits[w];
  if (g == 0 && tid == 0)
    *s.done = done;
  if (clocked)
    for (int i = 0; i < 4; ++i)
      s.clocks[i] += ticks[i];
}

__global__ void denseSetupKernel(DenseState s, const int *initialSize, const int *initialId) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < s.n; i += gridDim.x * blockDim.x) {
    s.size[i] = initialSize ? initialSize[i] : 1;
    s.id[i] = initialId ? initialId[i] : i;
    s.scanned[i] = kEmptyKey;
    s.scanned[s.n + i] = kEmptyKey;
  }
  const int words = (s.n + 31) >> 5; // every slot is active
  for (int w = blockIdx.x * blockDim.x + threadIdx.x; w < words; w += gridDim.x * blockDim.x) {
    const int rest = s.n - 32 * w;
    s.active[w] = rest >= 32 ? 0xffffffffu : (1u << rest) - 1u;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0)
    *s.done = 0;
}

__global__ void denseInitItemsKernel(int2 *items, int n) {
  // Row r's chunks start at sum over rows < r of ceil((n - 1 - r') / kChunk);
  // rows are enumerated by a single thread per row with a closed form below.
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n - 1)
    return;
  // Each row gets ceil((n-1-r)/kChunk) items; prefix over rows computed on
  // the host is avoided by giving every row a fixed stride of maxChunks.
  const int maxChunks = (n - 1 + kChunk - 1) / kChunk;
  const int len = n - 1 - r;
  const int chunks = (len + kChunk - 1) / kChunk;
  for (int c = 0; c < maxChunks; ++c)
    items[(size_t)r * maxChunks + c] = c < chunks ? make_int2(r, r + 1 + c * kChunk)
                                                  : make_int2(r, n); // empty segment
}

} // namespace

int denseLinkageOnCondensed(float *D, int n, int linkage, const int *initialSize,
                            const int *initialId, int firstNewId, double *hostTree) {
  if (n < 2)
    return 0;
  const int G = std::min(numCUs(), std::max(kMinGroups, (n + 63) / 64));
  if ((n + G - 1) / G > kMaxOwned || G > kThreads)
    return kErrInvalidShape; // beyond any condensed matrix that fits in HBM
  DenseState st{};
  DevArray<int> size, id;
  DevArray<unsigned long long> scanned, records, steps, partFn, partNext;
  DevArray<unsigned int> partMin, active;
  DevArray<int> pendingRows;
  DevArray<int2> initItems;
  DevArray<double> tree;
  DevArray<unsigned long long> clocks;
  DevArray<unsigned int> barrierWords;
  Status s;
  const int maxChunks = (n - 1 + kChunk - 1) / kChunk;
  const long long initCount = (long long)(n - 1) * maxChunks;
  const int groups = (G + kGroup - 1) / kGroup;
  // The barrier's words, then the merges made.
  const size_t numBarrierWords = (size_t)kLineWords * (3 + groups), doneWord = numBarrierWords;
  // The merge kernel keeps one bit per slot and the batch's new distances of
  // its rows in LDS beside its static arrays.
  const size_t activeBytes = (size_t)(n + 31) / 32 * sizeof(unsigned int);
  const int per = (n + G - 1) / G;
  int device = 0, maxLds = 0;
  s((int)hipGetDevice(&device));
  s((int)hipDeviceGetAttribute(&maxLds, hipDeviceAttributeMaxSharedMemoryPerBlock, device));
  if (!s.ok())
    return s.code;
  const void *chain = linkage == kSingle     ? (const void *)denseChainKernel<kSingle>
                      : linkage == kComplete ? (const void *)denseChainKernel<kComplete>
                      : linkage == kAverage  ? (const void *)denseChainKernel<kAverage>
                                             : (const void *)denseChainKernel<kWard>;
  const void *kernel = linkage == kSingle     ? (const void *)denseMergeKernel<kSingle>
                       : linkage == kComplete ? (const void *)denseMergeKernel<kComplete>
                       : linkage == kAverage  ? (const void *)denseMergeKernel<kAverage>
                                              : (const void *)denseMergeKernel<kWard>;
  hipFuncAttributes attr{};
  s((int)hipFuncGetAttributes(&attr, kernel));
  if (!s.ok())
    return s.code;
  if (activeBytes + per * sizeof(float) + attr.sharedSizeBytes > (size_t)maxLds)
    return kErrInvalidShape; // beyond any condensed matrix that fits in HBM
  const int batch = (int)std::min<size_t>(
      kMaxBatch, (maxLds - attr.sharedSizeBytes - activeBytes) / (per * sizeof(float)));
  const size_t dynamicBytes = activeBytes + (size_t)batch * per * sizeof(float);
  s(size.alloc(n));
  s(id.alloc(n));
  s(scanned.alloc((size_t)2 * n));
  s(records.alloc((size_t)G * kRecordWords));
  s(steps.alloc((size_t)2 * G * kStepWords));
  s(active.alloc((n + 31) / 32));
  s(partFn.alloc((size_t)kMaxBatch * G));
  s(partNext.alloc((size_t)kMaxBatch * G));
  s(partMin.alloc((size_t)kMaxBatch * G));
  s(pendingRows.alloc((size_t)G * per));
  s(initItems.alloc(initCount));
  s(tree.alloc((size_t)(n - 1) * 4));
  s(barrierWords.alloc(numBarrierWords + 1));
  if (!s.ok())
    return s.code;
  st.D = D;
  st.n = n;
  st.firstNewId = firstNewId;
  st.per = per;
  st.batch = batch;
  st.partFn = partFn;
  st.partNext = partNext;
  st.partMin = partMin;
  st.size = size;
  st.id = id;
  st.scanned = scanned;
  st.records = records;
  st.steps = steps;
  st.active = active;
  st.done = reinterpret_cast<int *>(barrierWords.get() + doneWord);
  st.pendingRows = pendingRows;
  st.items = initItems;
  st.tree = tree;
  st.clocks = nullptr;
  st.bar.words = barrierWords;
  st.bar.groups = groups;
  if (timingEnabled()) {
    s(clocks.alloc(4));
    s(fill(clocks, 0, 4 * sizeof(unsigned long long)));
    st.clocks = clocks;
  }
  s(fill(barrierWords, 0, numBarrierWords * sizeof(unsigned int)));
  PhaseTimer timer(kPhaseDense);
  hipLaunchKernelGGL(denseSetupKernel, dim3(std::min(1024, (n + 255) / 256)), dim3(256), 0,
                     stream(), st, initialSize, initialId);
  hipLaunchKernelGGL(denseInitItemsKernel, dim3((n + 255) / 256), dim3(256), 0, stream(),
                     initItems.get(), n);
  hipLaunchKernelGGL(denseInitKernel,
                     dim3((unsigned)std::max<long long>(1, std::min<long long>(initCount, 8LL * G))),
                     dim3(kThreads), 0, stream(), st, (int)initCount);
  s((int)hipGetLastError());
  // Batches until the tree is whole or few merges of a batch stand; then a run of
  // single merges, and batches again.
  std::vector<unsigned int> words(numBarrierWords + 1);
  int from = 0, run = kFirstRun; // merges made when the batches begin
  st.average = kFirstAverage;
  while (s.ok()) {
    void *args[] = {&st};
    s((int)hipLaunchCooperativeKernel(kernel, dim3(G), dim3(kThreads),
                                      args, (unsigned int)dynamicBytes, stream()));
    s(sync());
    if (s.ok())
      s(download(words.data(), barrierWords, words.size() * sizeof(unsigned int)));
    if (s.ok() && words[kLineWords])
      return (int)hipErrorLaunchTimeOut; // a barrier wait exceeded its limit
    const int done = (int)words[doneWord];
    if (!s.ok() || done >= n - 1)
      break;
    if (done - from >= kFirstRun)
      run = kFirstRun;
    void *runArgs[] = {&st, &run};
    s((int)hipLaunchCooperativeKernel(chain, dim3(G), dim3(kThreads), runArgs,
                                      (unsigned int)activeBytes, stream()));
    from = std::min(n - 1, done + run);
    run = std::min(2 * run, kLongestRun);
    st.average = kNextAverage;
  }
  if (s.ok() && st.clocks) {
    unsigned long long ticks[4];
    s(download(ticks, clocks, sizeof(ticks)));
    const double khz = wallClockKHz();
    addMs(kPhaseDenseSelect, (double)ticks[0] / khz, 1);
    addMs(kPhaseDenseUpdate, (double)ticks[1] / khz, 1);
    addMs(kPhaseDenseBarrier, (double)ticks[2] / khz, 1);
    addMs(kPhaseDenseRescan, (double)ticks[3] / khz, 1);
  }
  if (s.ok())
    s(download(hostTree, tree, (size_t)(n - 1) * 4 * sizeof(double)));
  if (s.ok())
    for (int step = 0; step < n - 1; ++step)
      if (hostTree[(size_t)step * 4] < 0)
        return kErrNonFinite;
  return s.code;
}

int denseLinkage(const float *X, int n, int d, MetricSpec m, int linkage, double *hostTree) {
  if (n < 2)
    return 0;
  const size_t count = (size_t)n * (n - 1) / 2;
  DevArray<float> D;
  Status s;
  s(D.alloc(count));
  if (!s.ok())
    return s.code;
  s(condensedMatrix(X, n, d, m, D));
  if (s.ok())
    s(denseLinkageOnCondensed(D, n, linkage, nullptr, nullptr, n, hostTree));
  return s.code;
}

} // namespace cuhc

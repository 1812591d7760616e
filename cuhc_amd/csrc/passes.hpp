// Host entry points of the all-pairs kernels (distance matrices, nearest
// other component passes, spatial pruning). All pointers are device pointers
// unless noted; everything runs on cuhc::stream().
#pragma once

#include "common.hpp"
#include "runtime.hpp"

#include <vector>

namespace cuhc {

struct MetricSpec {
  int id;
  float p; // Minkowski order
};

enum WeightKind : int { kWeightPlain = 0, kWeightMReach = 1, kWeightWard = 2 };

struct WeightSpec {
  int kind = kWeightPlain;
  const float *core = nullptr; // device, for kWeightMReach
  float alpha = 1.0f;
  const int *size = nullptr; // device, for kWeightWard
};

bool validMetric(int id);
bool metricHasBoxBound(int id);
int tilePoints(int metricId); // tile side of the metric's all-pairs kernels (128 or 64)

// out[i * nB + j] = metric(A[i], B[j]).
int pairwiseMatrix(const float *A, int nA, const float *B, int nB, int d, MetricSpec m,
                   float *out);

// Condensed upper triangle: out[i*n - i*(i+1)/2 + (j - i - 1)] = metric(X[i], X[j]), i < j.
int condensedMatrix(const float *X, int n, int d, MetricSpec m, float *out);

// nearest[i] = min over j with comp[j] != comp[i] of packKey(weight(i, j), id(j)),
// combined by atomicMin, so nearest[] must start at kEmptyKey. Each unordered
// pair is computed once (tiles I <= J). id(j) = orig[j] (device) for points in
// spatial order, else j (orig == nullptr). numComp (device, nullable): nothing
// is computed when it holds 1 (passes queued ahead of the host).
int nearestOtherSymmetric(const float *X, int n, int d, MetricSpec m, WeightSpec w,
                          const int *comp, const int *orig, unsigned long long *nearest,
                          const int *numComp = nullptr);

// ---------------------------------------------------------------------------
// Spatial pruning (reference src/spatial.cuh)

constexpr int kPruneMinPoints = 16384;
constexpr int kPruneMaxFeatures = 64;
constexpr int kPruneHardMaxFeatures = 256;
constexpr double kPruneGiveUpShare = 0.5;
// Ward. A pruned pass finds every cluster's nearest again, where a search takes
// up the few that lost theirs, and the share grows by the round (0.03 of single
// points, 0.3 three rounds on), so that pruning pays for few features only, by
// the sampled share: 60,000 points, 0.03 (3 features) 12.7 ms pruned and 15.4
// searched, 0.05 13.1 and 15.0, 0.07 16.2 and 15.8, 0.18 19.3 and 16.3, 0.33 (8
// features in blobs) 24.3 and 18.2; 150,000, 0.03 44 and 52, 0.08 62 and 53. Given
// up at 0.25 and 0.5, 60,000 points of 2 features took 10.3 and 11.1, of 3 13.3
// and 12.7.
constexpr double kWardPruneShare = 0.06, kWardGiveUpShare = 0.35;
enum PruneMode : int { kPruneAuto = 0, kPruneAlways = 1, kPruneNever = 2 };

bool shouldPrune(int mode, int metricId, int n, int d);

// k-d order of the listed points (indices into X; null: all of the first
// count), all arrays on the device: order[i] = index of the point at position i.
int spatialOrder(const float *X, int d, const int *list, int count, int *order);
// The order of mutual-reachability passes over X (n points in k-d order, orig:
// position -> original index): the points above the 90th percentile of core
// distances (noise, in sparse regions) get their own k-d order after the
// others'. A pruned pass skips a column tile when its bound exceeds the
// largest current best of the row tile, and one sparse point's large
// mutual-reachability weight would otherwise hold that bound up for the dense
// points it shares a tile with. newToOld: new position -> position in X;
// newOrig: new position -> original index. Left alone (*stratified false)
// when one class would have less than a tile.
int coreStratifiedOrder(const float *X, int n, int d, const float *core, const int *orig,
                        int *newToOld, int *newOrig, bool *stratified);
// dst[to[i]] = src[i].
int scatterFloats(const float *src, const int *to, int n, float *dst);

// dst[i] = src[order[i]] (rows of d floats).
int gatherRows(const float *src, const int *order, int n, int d, float *dst);

struct PassStats {
  unsigned long long tilesComputed = 0, tilesTotal = 0;
};

// Pruned pass for points in spatial order: same contract as
// nearestOtherSymmetric, except that keys carry orig[j] (device array; null:
// positions, as for rnn cluster slots), so ties break by original index
// exactly as in an unpruned run. compBest (nullable,
// one u32 per component, seedComponentBest) holds the weight bits of the best
// edge known for each component; rows stop searching above it, so a row's
// result is exact only when it holds its component's smallest edge, which is
// all the contraction uses. Returns the share of tile pairs computed in
// *share. rowTileStride > 1 runs every stride-th row tile only (sampling).
// skipComp (nullable, device): rows of that component (-1: none) search
// nothing and keep their nearest[] entries; so do rows p with closedRows[p]
// set (nullable, device), whose exact answers are already in nearest[].
// kept (nullable, device, n x 4 keys by position; not with Ward weights, closed
// rows or sampling): every row also keeps its 4 smallest keys over
// the other components (ascending, empty keys ~0 padded), searched without
// the component bounds, for settling rows in later rounds.
// keptShare (with closed rows): the share of the tile pairs that the keeping
// walk computed. Where the open rows' walk would compute more pairs than
// nearestOtherSymmetric at that share, it computes none: *share = -1.
int nearestOtherWalk(const float *X, int n, int d, MetricSpec m, WeightSpec w, const int *comp,
                     const int *orig, unsigned int *compBest, unsigned long long *nearest,
                     double *share, PassStats *stats, int rowTileStride = 1,
                     const int *skipComp = nullptr, const unsigned char *closedRows = nullptr,
                     unsigned long long *kept = nullptr, double keptShare = 0.0);

// Rows settled from the 4 keys each row kept in an earlier round (kept, by
// position; keys carry original indices, posOf maps them to positions, null:
// identity): a row whose list holds a point outside its component now takes
// the first such key as its exact nearest (the list holds the row's smallest
// keys over all other points, so every point outside the component that it
// misses weighs more), lowers its component's best known weight and is
// closed; so is a row whose last key weighs more than that best, without an
// answer. The others, and rows of skipComp, stay open.
int settleFromKept(const unsigned long long *kept, int n, const int *comp, const int *posOf,
                   const int *skipComp, unsigned long long *nearest, unsigned int *compBest,
                   unsigned char *closed);

// *majority (device) = the component holding more than half of the n points,
// or -1. sizes: numComp ints of scratch.
int majorityComponent(const int *comp, int n, int numComp, int *sizes, int *majority);

// compBest[c] for c < numComp: "none", then (fromNearest) the weight bits of
// the previous pass's candidates whose partner is still in another component.
// posOf maps an original index to its position (null: identity).
int seedComponentBest(const unsigned long long *nearest, const int *comp, const int *posOf,
                      int n, int numComp, bool fromNearest, unsigned int *compBest);

// posOf[orig[p]] = p.
int inverseOrder(const int *orig, int n, int *posOf);

// Share of tiles a pruned pass would compute, from a sample of row tiles
// (Boruvka's first pass: plain weights, every point its own component).
int estimatePrunedShare(const float *X, int n, int d, MetricSpec m, double *share);

} // namespace cuhc

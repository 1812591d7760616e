// Boruvka's MST over the complete graph, matrix-free (reference
// src/mst.cuh:83-186), plus the single-linkage and HDBSCAN drivers
// (src/hdbscan.cuh:353-391, src/capi.cu:68-119).
//
// Each round: the GPU finds, for every point, its nearest point in another
// component (one all-pairs pass), then contracts (contract.hip): each
// component's smallest edge under the total order (weight, u, v) in original
// indices joins it to its neighbour and the components are relabelled, all in
// device memory. Every chosen edge is the minimum edge leaving its component under
// a strict total order, so the result is the unique MST under that order:
// independent of the pass's tile order, pruning, or point permutation.
#include "mst.hpp"

#include <algorithm>
#include <cmath>

namespace cuhc {

int DevicePoints::arrange(const float *X, int n, int d) {
  Status s;
  s(orig.alloc(n));
  if (s.ok())
    s(spatialOrder(X, d, nullptr, n, orig));
  if (s.ok())
    s(gatherRows(X, orig, n, d, points));
  inOrder = s.ok();
  return s.code;
}

// Both entry paths check the coordinates first (kErrNonFinite for NaN or
// infinity): the FP16 candidate kernels are compiled without NaN semantics and
// the k-d order needs ordered comparisons.
int DevicePoints::upload(const float *hostPoints, int n, int d, bool spatial, bool keep) {
  const size_t count = (size_t)n * d;
  Status s;
  s(points.alloc(count));
  if (!s.ok())
    return s.code;
  if (!spatial) {
    s(cuhc::upload(points, hostPoints, count * sizeof(float)));
    s(checkFinite(points, count));
    return s.code;
  }
  s(raw.alloc(count));
  s(cuhc::upload(raw, hostPoints, count * sizeof(float)));
  s(checkFinite(raw, count));
  if (s.ok())
    s(arrange(raw, n, d));
  if (keep)
    given = raw;
  else
    raw.release();
  return s.code;
}

void DevicePoints::leaveOrder() {
  if (!inOrder || !given)
    return;
  external = given;
  points.release();
  orig.release();
  inOrder = false;
}

// The caller may have written devicePoints on another stream of this HIP
// runtime: the device is synchronised before the library stream reads them.
int DevicePoints::adopt(const float *devicePoints, int n, int d, bool spatial) {
  const size_t count = (size_t)n * d;
  Status s;
  s((int)hipDeviceSynchronize());
  s(checkFinite(devicePoints, count));
  if (!s.ok())
    return s.code;
  if (!spatial) {
    external = devicePoints;
    return 0;
  }
  s(points.alloc(count));
  if (s.ok())
    s(arrange(devicePoints, n, d));
  given = devicePoints;
  return s.code;
}

int boruvkaMst(const float *X, int n, int d, MetricSpec m, WeightSpec w, const MstOptions &opt,
               Contraction &ct) {
  Status s;
  s(ct.alloc(n));
  if (!s.ok() || n < 2)
    return s.code;
  DevArray<int> dComp, dPosOf, dSizes, dSkip;
  DevArray<unsigned int> dCompBest;
  DevArray<unsigned long long> dNearest;
  s(dComp.alloc(n));
  s(dNearest.alloc(n));
  if (opt.devOrig) {
    s(dPosOf.alloc(n));
    if (s.ok())
      s(inverseOrder(opt.devOrig, n, dPosOf));
  }
  // Pruned passes bound each component's search by its best known edge, and
  // skip the rows of a component holding more than half of the points: it
  // proposes no edge in that round and joins through the others' smallest
  // edges (Boruvka only needs every proposed edge to be its component's
  // smallest; every other component still proposes).
  if (opt.prune) {
    s(dCompBest.alloc(n));
    s(dSizes.alloc(n));
    s(dSkip.alloc(1));
  }
  // Rows settled from the learned candidate lists (mutual reachability,
  // alpha = 1) are closed to the walk.
  const bool useLists = opt.lists && opt.prune && w.kind == kWeightMReach && w.alpha == 1.0f;
  // Without lists, the first round's walk keeps each row's 4 smallest keys over
  // all other points, and the later rounds' rows settle from them: whatever
  // share of the tiles that walk computes, it replaces most of the later
  // rounds' passes. Without the memory for them (33 bytes a point) the rounds
  // walk every row or, past the give-up share, compute every pair once.
  bool keepKeys = !useLists && opt.prune;
  DevArray<unsigned char> dClosed;
  DevArray<unsigned long long> dListCounters, dKept;
  if (useLists)
    s(dClosed.alloc(n));
  if (keepKeys && (dKept.alloc((size_t)n * 4) || dClosed.alloc(n))) {
    (void)hipGetLastError();
    dKept.release();
    keepKeys = false;
  }
  if (useLists) {
    s(dListCounters.alloc(64 * 16));
    if (s.ok())
      s(fill(dListCounters, 0, dListCounters.bytes()));
  }
  bool keptValid = false; // dKept holds the first round's lists
  // Of the tile pairs, computed by the walk that kept them. Plain weights only:
  // under mutual reachability the later walks leave out more than that one did
  // (HDBSCAN of 100,000 x 14 normal points 46.8 ms, by this share 49.1).
  double keptShare = 0.0;
  if (s.ok())
    s(resetComponents(dComp, n));
  MixedPass *mixed = nullptr;
  if (s.ok() && opt.mixed) {
    int st = 0;
    mixed = mixedPassCreate(X, n, d, &st);
    s(st);
  }
  const int *posOf = opt.devOrig ? dPosOf.get() : nullptr;
  int numComponents = n;
  bool pruneThisPass = opt.prune;
  bool haveResult = false; // dNearest holds the last round's exact result
  if (s.ok() && ct.small && !mixed && !opt.prune) {
    // Few points: rounds cost launches and host reads, so as many as such
    // inputs take (components fall to a quarter or less per round) are queued
    // before the first read; rounds past the last find one component and end.
    s(fill(dNearest, 0xff, n * sizeof(unsigned long long)));
    int rounds = std::max(1, (int)std::ceil(std::log2((double)n) / 2));
    while (s.ok() && numComponents > 1) {
      for (int q = 0; q < rounds && s.ok(); ++q) {
        s(nearestOtherSymmetric(X, n, d, m, w, dComp, opt.devOrig, dNearest, ct.state + 1));
        PhaseTimer timer(kPhaseContract);
        s(contractSmallQueue(ct, dNearest, dComp, opt.devOrig, posOf, true));
      }
      int added = 0;
      if (s.ok())
        s(contractState(ct, &numComponents, &added));
      rounds = 1;
    }
  }
  while (s.ok() && numComponents > 1) {
    if (mixed) {
      s(mixedPassRun(mixed, dComp, numComponents, m.id == kSqEuclidean, !haveResult, dNearest));
    } else {
      if (pruneThisPass)
        s(seedComponentBest(dNearest, dComp, posOf, n, numComponents, haveResult, dCompBest));
      s(fill(dNearest, 0xff, n * sizeof(unsigned long long)));
      if (!s.ok())
        break;
      if (pruneThisPass) {
        double share = 1.0;
        s(majorityComponent(dComp, n, numComponents, dSizes, dSkip));
        if (useLists)
          s(settleFromLists(*opt.lists, n, dComp, opt.devOrig, w.core, dSkip, dNearest,
                            dCompBest, dClosed, dListCounters));
        if (keepKeys && !keptValid) {
          s(nearestOtherWalk(X, n, d, m, w, dComp, opt.devOrig, nullptr, dNearest, &share,
                             opt.stats, 1, dSkip, nullptr, dKept));
          keptValid = true;
          keptShare = w.kind == kWeightPlain ? share : 0.0;
          share = 0.0; // the next rounds walk the rows that the keys leave open
        } else {
          if (keepKeys)
            s(settleFromKept(dKept, n, dComp, posOf, dSkip, dNearest, dCompBest, dClosed));
          s(nearestOtherWalk(X, n, d, m, w, dComp, opt.devOrig, dCompBest, dNearest, &share,
                             opt.stats, 1, dSkip,
                             useLists || keepKeys ? dClosed.get() : nullptr, nullptr,
                             keptShare));
          if (s.ok() && share < 0.0) { // too many open rows: every pair, once
            s(nearestOtherSymmetric(X, n, d, m, w, dComp, opt.devOrig, dNearest));
            share = 0.0; // the next round's open rows decide again
          }
        }
        pruneThisPass = share <= kPruneGiveUpShare;
      } else {
        s(nearestOtherSymmetric(X, n, d, m, w, dComp, opt.devOrig, dNearest));
      }
    }
    if (!s.ok())
      break;
    haveResult = true;
    PhaseTimer timer(kPhaseContract);
    int next = numComponents, added = 0;
    s(contractRound(ct, dNearest, dComp, opt.devOrig, posOf, numComponents, &next, &added));
    if (s.ok() && added == 0)
      s(kErrDisconnected);
    numComponents = next;
  }
  if (mixed)
    mixedPassDestroy(mixed);
  if (useLists && s.ok()) {
    std::vector<unsigned long long> ctr(64 * 16);
    s(download(ctr.data(), dListCounters, dListCounters.bytes()));
    LearnedStats st;
    for (int k = 0; k < 64; ++k) {
      st.settled += ctr[k * 16];
      st.considered += ctr[k * 16 + 1];
    }
    if (s.ok())
      learnedStatsAdd(st);
  }
  return s.code;
}

int singleLinkageMst(const DevicePoints &pts, int n, int d, MetricSpec m, bool prune, bool mixed,
                     PassStats *stats, double *tree) {
  MstOptions opt;
  opt.prune = prune && pts.ordered();
  opt.devOrig = pts.ordered() ? pts.orig.get() : nullptr;
  opt.stats = stats;
  opt.mixed = mixed && !pts.ordered() && (m.id == kEuclidean || m.id == kSqEuclidean) &&
              mixedPassSupports(d);
  Contraction ct;
  int status = boruvkaMst(pts.data(), n, d, m, WeightSpec{}, opt, ct);
  if (status == 0)
    status = treeFromDeviceEdges(ct.edges, n, tree);
  return status;
}

int hdbscanTree(const DevicePoints &pts, int n, int d, MetricSpec m, int minSamples, float alpha,
                int coreMethod, bool prune, PassStats *stats, double *tree, float *hostCore) {
  DevArray<float> core;
  Status s;
  s(core.alloc(n));
  // The learned method's candidate lists also settle Boruvka rows (pruned
  // passes, mutual reachability with alpha = 1, a box metric).
  RadiusLists lists;
  const bool keepLists = coreMethod == kCoreLearned && prune && pts.ordered() && alpha == 1.0f &&
                         metricHasBoxBound(m.id);
  if (s.ok()) {
    if (keepLists)
      s(coreLearned(pts.data(), n, d, m, minSamples, core, true, &lists));
    else
      s(coreDistances(pts.data(), n, d, m, minSamples, core, coreMethod,
                      prune && pts.ordered()));
  }
  // Pruned passes: reorder by core-distance class (the tree does not depend
  // on the order).
  const float *X = pts.data();
  const int *devOrig = pts.ordered() ? pts.orig.get() : nullptr;
  bool stratified = false;
  DevArray<float> sPoints, sCore;
  DevArray<int> sOrig, sMap;
  if (s.ok() && prune && pts.ordered() && n >= 1024) {
    s(sOrig.alloc(n));
    s(sMap.alloc(n));
    if (s.ok())
      s(coreStratifiedOrder(X, n, d, core, devOrig, sMap, sOrig, &stratified));
    if (s.ok() && stratified) {
      s(sPoints.alloc((size_t)n * d));
      s(sCore.alloc(n));
      if (s.ok()) {
        s(gatherRows(X, sMap, n, d, sPoints));
        s(gatherRows(core, sMap, n, 1, sCore));
      }
      if (s.ok()) {
        X = sPoints;
        devOrig = sOrig;
      }
      if (s.ok() && keepLists) {
        // List rows stay in the old order (rowMap = new -> old); partners
        // are renumbered to the new positions.
        DevArray<int> oldToNew;
        s(oldToNew.alloc(n));
        if (s.ok())
          s(inverseOrder(sMap, n, oldToNew));
        if (s.ok())
          s(remapRadiusLists(lists, n, oldToNew));
        lists.rowMap = sMap;
        s(sync());
      }
    }
  }
  MstOptions opt;
  opt.prune = prune && pts.ordered();
  opt.devOrig = devOrig;
  opt.stats = stats;
  opt.lists = keepLists && lists.pos.get() ? &lists : nullptr;
  WeightSpec w;
  w.kind = kWeightMReach;
  w.core = stratified ? sCore.get() : core.get();
  w.alpha = alpha;
  Contraction ct;
  if (s.ok())
    s(boruvkaMst(X, n, d, m, w, opt, ct));
  if (s.ok() && hostCore) {
    DevArray<float> byIndex; // in original order
    if (devOrig) {
      s(byIndex.alloc(n));
      if (s.ok())
        s(scatterFloats(w.core, devOrig, n, byIndex));
    }
    if (s.ok())
      s(download(hostCore, devOrig ? byIndex.get() : w.core, n * sizeof(float)));
  }
  if (s.ok())
    s(treeFromDeviceEdges(ct.edges, n, tree));
  return s.code;
}

} // namespace cuhc

// Boruvka's contraction between rounds, on the GPU (the reference does this
// step on the host, src/mst.cuh:130-181, with the same result).
//
// From nearest[p] (the key of p's nearest point in another component: weight
// bits << 32 | original index) every component takes its smallest outgoing
// edge under the global order (weight, smaller endpoint, larger endpoint) in
// two minimum passes: (weight, smaller endpoint) as one u64, then the larger
// endpoint among the points that reached that minimum. Each component hooks
// onto the component at the edge's other end. With a strict total order the
// only cycles are pairs that chose the same edge; the lower component of such
// a pair stays a root. Every component that is not a root emits its edge: at
// its index less the number of roots before it, which the scan that numbers
// the roots gives. Pointer jumping turns the hooks into roots and every point
// is relabelled. The edges, the component count and an error flag stay in
// device memory (Contraction::state); the host reads the state once per round.
//
// Bound by launches and that read for small inputs, by one read and write of
// the points' state for large ones. Two forms:
//   one workgroup, up to kSmallPoints points: everything in LDS, one launch
//     per round, so that several rounds can be queued without a host read;
//   several kernels above: about ten launches and one host read per round.
// A round took sixteen launches, with atomics for the edges' places, and three
// or four reads: whole single-linkage trees of 500 points took 0.98 ms and take
// 0.31 ms; of 20,000 (with the edges sorted on the device) 3.9 and 2.4 ms.
#include "mst.hpp"

#include "primitives.hpp"

namespace cuhc {

namespace {

__global__ void iotaIntKernel(int *out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    out[i] = i;
}

DEV unsigned long long lowKey(unsigned long long key, int a) {
  const int b = (int)keyIndex(key);
  return (key & 0xffffffff00000000ull) | (unsigned int)min(a, b);
}

// The first round: every component is one point, so its minima are the
// point's own key.
__global__ void firstMinKernel(const unsigned long long *__restrict__ nearest,
                               const int *__restrict__ comp, const int *__restrict__ orig, int n,
                               unsigned long long *__restrict__ best1,
                               unsigned int *__restrict__ best2) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n)
    return;
  const unsigned long long key = nearest[p];
  const int c = comp[p], a = orig ? orig[p] : p;
  best1[c] = key == kEmptyKey ? kEmptyKey : lowKey(key, a);
  best2[c] = key == kEmptyKey ? 0xffffffffu : (unsigned int)max(a, (int)keyIndex(key));
}

__global__ void componentMinKernel(const unsigned long long *__restrict__ nearest,
                                   const int *__restrict__ comp, const int *__restrict__ orig,
                                   int n, unsigned long long *best1) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n)
    return;
  const unsigned long long key = nearest[p];
  if (key == kEmptyKey)
    return;
  atomicMin(&best1[comp[p]], lowKey(key, orig ? orig[p] : p));
}

// The same with few components: same-address atomics from many waves
// serialise (one component holding every point would take one atomic per
// point), so each workgroup first reduces into LDS and then flushes one atomic
// per component it saw.
constexpr int kLdsComponents = 4096;

__global__ void __launch_bounds__(256)
    componentMinLdsKernel(const unsigned long long *__restrict__ nearest,
                          const int *__restrict__ comp, const int *__restrict__ orig, int n,
                          int numComp, unsigned long long *best1) {
  __shared__ unsigned long long local[kLdsComponents];
  for (int c = threadIdx.x; c < numComp; c += blockDim.x)
    local[c] = kEmptyKey;
  __syncthreads();
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    const unsigned long long key = nearest[p];
    if (key != kEmptyKey)
      atomicMin(&local[comp[p]], lowKey(key, orig ? orig[p] : p));
  }
  __syncthreads();
  for (int c = threadIdx.x; c < numComp; c += blockDim.x)
    if (local[c] != kEmptyKey)
      atomicMin(&best1[c], local[c]);
}

__global__ void componentMin2Kernel(const unsigned long long *__restrict__ nearest,
                                    const int *__restrict__ comp, const int *__restrict__ orig,
                                    int n, const unsigned long long *__restrict__ best1,
                                    unsigned int *best2) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n)
    return;
  const unsigned long long key = nearest[p];
  if (key == kEmptyKey)
    return;
  const int a = orig ? orig[p] : p;
  const int c = comp[p];
  if (lowKey(key, a) == best1[c])
    atomicMin(&best2[c], (unsigned int)max(a, (int)keyIndex(key)));
}

// The component that c's smallest edge leads to (c itself: no edge leaves it).
DEV int hookOf(int c, unsigned long long k1, unsigned int hi32, const int *comp,
               const int *posOf, int n) {
  const unsigned int lo32 = (unsigned int)(k1 & 0xffffffffu);
  if (k1 == kEmptyKey || lo32 >= (unsigned)n || hi32 >= (unsigned)n)
    return c;
  const int lo = (int)lo32, hi = (int)hi32;
  const int cl = comp[posOf ? posOf[lo] : lo], ch = comp[posOf ? posOf[hi] : hi];
  return cl == c ? ch : cl;
}

// The root link of c with hook pc, whose own hook is ppc: of two components
// that chose the same edge the lower stays a root.
DEV int rootLink(int c, int pc, int ppc) { return ppc == c && c < pc ? c : pc; }

__global__ void hookKernel(const unsigned long long *__restrict__ best1,
                           const unsigned int *__restrict__ best2, const int *__restrict__ comp,
                           const int *__restrict__ posOf, int n, int numComp, int *parent) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < numComp)
    parent[c] = hookOf(c, best1[c], best2[c], comp, posOf, n);
}

__global__ void rootLinksKernel(const int *__restrict__ parent, int numComp, int *root,
                                int *flags) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < numComp) {
    const int pc = parent[c];
    const int r = rootLink(c, pc, parent[pc]);
    root[c] = r;
    flags[c] = r == c;
  } else if (c == numComp) {
    flags[c] = 0;
  }
}

// Up to kHops steps towards the root. Reads may see links that other threads
// already moved; every value read is an ancestor, at least as far along as the
// link it replaces, so after k passes a link spans at least kHops^k of the
// first ones (or ends at its root).
constexpr int kHops = 16;
constexpr int kJumpPasses = 3;

DEV int climb(const int *root, int r, int steps) {
  for (int i = 0; i < steps; ++i) {
    const int up = __hip_atomic_load(&root[r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (up == r)
      break;
    r = up;
  }
  return r;
}

__global__ void jumpKernel(int *root, int numComp) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < numComp)
    root[c] = climb(root, c, kHops);
}

// Points relabelled (each climbs the rest of its way: a link spans kHops^3
// hooks by now), edges of the components that are no roots emitted behind the
// forest's edgeBase edges, and the minima reset for the next round. A climb
// that does not end (hooks with a cycle: inconsistent keys) sets state[2].
__global__ void relabelKernel(int *comp, int n, const int *__restrict__ root,
                              const int *__restrict__ newId, int numComp, int edgeBase,
                              unsigned long long *best1, unsigned int *best2, EdgeArrays edges,
                              int *state) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) {
    const int r = climb(root, comp[p], numComp / (kHops * kHops * kHops) + 64);
    if (root[r] != r)
      state[2] = 1;
    comp[p] = newId[r];
  }
  if (p < numComp) {
    if (root[p] != p) {
      const unsigned long long k1 = best1[p];
      const int at = edgeBase + p - newId[p];
      if (at < edges.capacity) {
        edges.u[at] = (int)(k1 & 0xffffffffu);
        edges.v[at] = (int)best2[p];
        edges.w[at] = floatOf((unsigned int)(k1 >> 32));
      }
    }
    best1[p] = kEmptyKey;
    best2[p] = 0xffffffffu;
  }
  if (p == 0) {
    state[0] = edgeBase + numComp - newId[numComp];
    state[1] = newId[numComp];
  }
}

// The whole contraction of up to kSmallPoints points by one workgroup, every
// per-component array in LDS; nearest[] is emptied for the next pass on
// request. state[1] holds the component count on entry: with one component it
// returns at once.
constexpr int kSmallPoints = 7168; // 20 bytes of LDS per point: 140 KB
constexpr int kSmallThreads = 1024;
constexpr int kSmallPer = kSmallPoints / kSmallThreads;

__global__ void __launch_bounds__(kSmallThreads)
    contractSmallKernel(unsigned long long *nearest, int *comp, const int *__restrict__ orig,
                        const int *__restrict__ posOf, int n, bool empty, EdgeArrays edges, int *state) {
  extern __shared__ unsigned long long best1[]; // [n], then best2 [n], root [n], points [n]
  __shared__ int waveTotal[kSmallThreads / 64];
  unsigned int *best2 = reinterpret_cast<unsigned int *>(best1 + n);
  int *root = reinterpret_cast<int *>(best2 + n), *sComp = root + n;
  const int numComp = state[1], edgeBase = state[0];
  if (numComp <= 1)
    return;
  const int t = threadIdx.x;
  for (int i = t; i < n; i += kSmallThreads) {
    sComp[i] = comp[i];
    best1[i] = kEmptyKey;
    best2[i] = 0xffffffffu;
  }
  unsigned long long key[kSmallPer];
  int a[kSmallPer];
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j) {
    const int p = t + j * kSmallThreads;
    key[j] = p < n ? nearest[p] : kEmptyKey;
    a[j] = p < n ? (orig ? orig[p] : p) : 0;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j)
    if (key[j] != kEmptyKey)
      atomicMin(&best1[sComp[t + j * kSmallThreads]], lowKey(key[j], a[j]));
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j)
    if (key[j] != kEmptyKey) {
      const int c = sComp[t + j * kSmallThreads];
      if (lowKey(key[j], a[j]) == best1[c])
        atomicMin(&best2[c], (unsigned int)max(a[j], (int)keyIndex(key[j])));
    }
  __syncthreads();
  for (int c = t; c < numComp; c += kSmallThreads)
    root[c] = hookOf(c, best1[c], best2[c], sComp, posOf, n);
  __syncthreads();
  // A thread's components are consecutive from here on (the scan's order).
  const int per = (numComp + kSmallThreads - 1) / kSmallThreads;
  const int c0 = min(numComp, t * per), c1 = min(numComp, c0 + per);
  int link[kSmallPer];
  int roots = 0;
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j) {
    const int c = c0 + j;
    if (c < c1) {
      const int pc = root[c];
      link[j] = rootLink(c, pc, root[pc]);
      roots += link[j] == c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j)
    if (c0 + j < c1)
      root[c0 + j] = link[j];
  const int lane = t & 63, wave = t >> 6;
  int before = roots;
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    const int up = __shfl_up(before, m, 64);
    if (lane >= m)
      before += up;
  }
  if (lane == 63)
    waveTotal[wave] = before;
  __syncthreads();
  before -= roots;
  int newNum = 0;
  for (int w = 0; w < kSmallThreads / 64; ++w) {
    before += w < wave ? waveTotal[w] : 0;
    newNum += waveTotal[w];
  }
  // Emit the others' edges and number the roots (best2 becomes newId).
#pragma unroll
  for (int j = 0; j < kSmallPer; ++j) {
    const int c = c0 + j;
    if (c >= c1)
      continue;
    if (link[j] == c) {
      best2[c] = (unsigned int)before++;
    } else {
      const int at = edgeBase + c - before;
      if (at < edges.capacity) {
        edges.u[at] = (int)(best1[c] & 0xffffffffu);
        edges.v[at] = (int)best2[c];
        edges.w[at] = floatOf((unsigned int)(best1[c] >> 32));
      }
    }
  }
  // Doubling until no link moves (at most 13 steps; 16 without an end: hooks
  // with a cycle).
  int moved = 1;
  for (int step = 0; step < 16 && moved; ++step) {
    moved = 0;
    for (int c = t; c < numComp; c += kSmallThreads) {
      const int r = root[c], rr = root[r];
      if (rr != r) {
        root[c] = rr;
        moved = 1;
      }
    }
    moved = __syncthreads_or(moved);
  }
  for (int p = t; p < n; p += kSmallThreads) {
    comp[p] = (int)best2[root[sComp[p]]];
    if (empty)
      nearest[p] = kEmptyKey;
  }
  if (t == 0) {
    state[0] = edgeBase + numComp - newNum;
    state[1] = newNum;
    if (moved)
      state[2] = 1;
    if (newNum == numComp)
      state[3] = 1; // no edge leaves any component
  }
}

__global__ void stateKernel(int *state, int n) {
  if (threadIdx.x < 4)
    state[threadIdx.x] = threadIdx.x == 1 ? n : 0;
}

inline dim3 gridFor(long long count) { return dim3((unsigned)((count + 255) / 256)); }

} // namespace

int Contraction::alloc(int points) {
  n = points;
  const int most = std::max(1, n - 1);
  Status s;
  s(state.alloc(4));
  s(storage.alloc((size_t)3 * most));
  small = n <= kSmallPoints;
  if (!small) {
    s(best1.alloc(n));
    s(best2.alloc(n));
    s(parent.alloc(n));
    s(root.alloc(n));
    s(flags.alloc(n + 1));
    s(newId.alloc(n + 1));
    s(scanTemp.alloc(scanTempBytes(n + 1)));
  }
  if (!s.ok())
    return s.code;
  edges = EdgeArrays{storage.get(), storage.get() + most,
                     reinterpret_cast<float *>(storage.get() + 2 * (size_t)most), most, 0};
  hipLaunchKernelGGL(stateKernel, dim3(1), dim3(64), 0, stream(), state.get(), n);
  return (int)hipGetLastError();
}

int resetComponents(int *comp, int n) {
  hipLaunchKernelGGL(iotaIntKernel, gridFor(n), dim3(256), 0, stream(), comp, n);
  return (int)hipGetLastError();
}

int contractSmallQueue(Contraction &ct, unsigned long long *nearest, int *comp, const int *orig,
                       const int *posOf, bool empty) {
  const size_t lds = (size_t)ct.n * (sizeof(unsigned long long) + 3 * sizeof(int));
  hipLaunchKernelGGL(contractSmallKernel, dim3(1), dim3(kSmallThreads), lds, stream(), nearest,
                     comp, orig, posOf, ct.n, empty, ct.edges, ct.state.get());
  return (int)hipGetLastError();
}

int contractState(Contraction &ct, int *numComp, int *added) {
  int host[4] = {0, 0, 0, 0};
  Status s;
  s(download(host, ct.state, sizeof(host)));
  if (!s.ok())
    return s.code;
  if (host[2] || host[0] > ct.n - 1)
    return kErrNonFinite; // hooks with a cycle, or more edges than a forest holds
  if (host[3])
    return kErrDisconnected;
  *added = host[0] - ct.edges.count;
  ct.edges.count = host[0];
  *numComp = host[1];
  return 0;
}

int contractRound(Contraction &ct, unsigned long long *nearest, int *comp, const int *orig,
                  const int *posOf, int numComp, int *newNumComp, int *added) {
  const int n = ct.n;
  Status s;
  if (ct.small) {
    s(contractSmallQueue(ct, nearest, comp, orig, posOf, false));
    if (s.ok())
      s(contractState(ct, newNumComp, added));
    return s.code;
  }
  if (numComp == n) {
    hipLaunchKernelGGL(firstMinKernel, gridFor(n), dim3(256), 0, stream(), nearest, comp, orig, n,
                       ct.best1.get(), ct.best2.get());
  } else {
    if (numComp <= kLdsComponents)
      hipLaunchKernelGGL(componentMinLdsKernel,
                         dim3(std::max(1, std::min(1024, (n + 255) / 256))), dim3(256), 0,
                         stream(), nearest, comp, orig, n, numComp, ct.best1.get());
    else
      hipLaunchKernelGGL(componentMinKernel, gridFor(n), dim3(256), 0, stream(), nearest, comp,
                         orig, n, ct.best1.get());
    hipLaunchKernelGGL(componentMin2Kernel, gridFor(n), dim3(256), 0, stream(), nearest, comp,
                       orig, n, ct.best1.get(), ct.best2.get());
  }
  hipLaunchKernelGGL(hookKernel, gridFor(numComp), dim3(256), 0, stream(), ct.best1.get(),
                     ct.best2.get(), comp, posOf, n, numComp, ct.parent.get());
  hipLaunchKernelGGL(rootLinksKernel, gridFor(numComp + 1), dim3(256), 0, stream(),
                     ct.parent.get(), numComp, ct.root.get(), ct.flags.get());
  s((int)hipGetLastError());
  s(exclusiveScan(ct.flags.get(), ct.newId.get(), numComp + 1, ct.scanTemp.get()));
  for (int pass = 0; pass < kJumpPasses; ++pass)
    hipLaunchKernelGGL(jumpKernel, gridFor(numComp), dim3(256), 0, stream(), ct.root.get(),
                       numComp);
  hipLaunchKernelGGL(relabelKernel, gridFor(n), dim3(256), 0, stream(), comp, n, ct.root.get(),
                     ct.newId.get(), numComp, ct.edges.count, ct.best1.get(), ct.best2.get(),
                     ct.edges, ct.state.get());
  s((int)hipGetLastError());
  if (s.ok())
    s(contractState(ct, newNumComp, added));
  return s.code;
}

} // namespace cuhc

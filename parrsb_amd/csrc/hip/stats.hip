// Neighbouring segments (statistics.c:17-113, recorded as RSB_NEIGHBORS at
// rsb.c:342-343): for every current segment, the number of other segments
// that share a vertex with it.  Vertex sharing is the dual graph's relation,
// so the pairs come from the graph rows: the distinct (segment, foreign
// segment) pairs among the elements' neighbours, counted per segment.
#include <algorithm>
#include <vector>

#include "state.hpp"

// A workgroup takes 256 consecutive positions of the element order (one
// segment or a few, with few neighbours), collects its distinct pairs in LDS
// and puts those into a hash set in memory; whoever adds a pair counts it for
// its segment.  (Every element's pairs appended one by one at a common
// counter, sorted and counted took 250 us and fifteen launches for 1M
// elements.)
#define NB_LDS 1024   // slots of a workgroup's set (power of two)
#define NB_PROBE 64   // slots looked at before a set counts as full
#define NB_SLOTS (1 << 24)  // most slots to begin with, if elements are fewer
__device__ inline unsigned nb_hash(uint64_t k) {
  return (unsigned)((k * 0x9e3779b97f4a7c15ull) >> 32);
}
__device__ inline void nb_add(uint64_t k, uint64_t *table, unsigned mask, int *nb, int *full) {
  unsigned h = nb_hash(k);
  for (int i = 0; i < NB_PROBE; i++, h++) {
    const unsigned long long old =
        atomicCAS((unsigned long long *)&table[h & mask], ~0ull, (unsigned long long)k);
    if (old == ~0ull) {
      atomicAdd(&nb[k >> 32], 1);
      return;
    }
    if (old == k) return;
  }
  *full = 1;
}

__global__ void __launch_bounds__(256) k_nb_pairs(int nel, const int *__restrict__ order,
                                                  const int64_t *__restrict__ growptr,
                                                  const uint32_t *__restrict__ gadj,
                                                  const int *__restrict__ segof, uint64_t *table,
                                                  unsigned mask, int *nb, int *full) {
  __shared__ unsigned long long set[NB_LDS];
  for (int i = threadIdx.x; i < NB_LDS; i += 256) set[i] = ~0ull;
  __syncthreads();
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < nel) {
    const int e = order[i], s = segof[e];
    const int64_t r1 = growptr[e + 1];
    int last = s;
    // eight entries and their segments in flight, then examined in order
    for (int64_t k0 = growptr[e]; k0 < r1; k0 += 8) {
      int tt[8];
#pragma unroll
      for (int u = 0; u < 8; u++) tt[u] = k0 + u < r1 ? (int)(gadj[k0 + u] & 0x0fffffffu) : e;
#pragma unroll
      for (int u = 0; u < 8; u++) tt[u] = segof[tt[u]];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int t = tt[u];
        if (t == s || t == last) continue;  // padding entries are e itself: t == s
        last = t;
        const unsigned long long key = ((unsigned long long)(uint32_t)s << 32) | (uint32_t)t;
        unsigned h = nb_hash(key);
        int p = 0;
        for (; p < NB_PROBE; p++, h++) {
          const unsigned long long old = atomicCAS(&set[h & (NB_LDS - 1)], ~0ull, key);
          if (old == ~0ull || old == key) break;
        }
        if (p == NB_PROBE) nb_add(key, table, mask, nb, full);
      }
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < NB_LDS; k += 256)
    if (set[k] != ~0ull) nb_add(set[k], table, mask, nb, full);
}

__global__ void k_nb_clear(uint64_t *__restrict__ table, int64_t slots, int *__restrict__ nb, int n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (int64_t k = i; k < slots; k += (int64_t)gridDim.x * blockDim.x) table[k] = ~0ull;
  for (int64_t k = i; k < n; k += (int64_t)gridDim.x * blockDim.x) nb[k] = 0;
}

extern "C" int rsbgpu_neighbors(rsbgpu *g, int *nbrs) {
  RSB_TRY(hipSetDevice(g->device));
  const int nel = g->nel, nseg = g->nseg;
  for (int s = 0; s < nseg; s++) nbrs[s] = 0;
  if (nel == 0 || nseg <= 1) return 0;
  hipStream_t st = g->stream;
  // room for 64 neighbours a segment (hexes have up to 26 parts around one),
  // but 128 MiB or a slot an element where that is more: millions of segments
  // may have few neighbours, and 512 bytes for each of 8M would be 4 GiB.  A
  // set that fills up is doubled and filled again (262,144 segments of one hex
  // in a set half as large to begin with: 95 ms a call instead of 92).
  int64_t slots = 1024;
  while (slots < 64 * (int64_t)nseg && (slots < NB_SLOTS || slots < nel)) slots *= 2;
  std::vector<int> h((size_t)nseg + 1);
  for (;; slots *= 2) {
    uint64_t *table = nullptr;
    int *nb = nullptr;  // counts, then the flag of a full set
    RSB_TRY(RSB_SCRATCH(table, sizeof(uint64_t) * (size_t)slots));
    RSB_TRY(RSB_SCRATCH(nb, sizeof(int) * h.size()));
    k_nb_clear<<<(unsigned)std::min<int64_t>(nblocks(slots, 256), 2048), 256, 0, st>>>(
        table, slots, nb, nseg + 1);
    k_nb_pairs<<<nblocks(nel, 256), 256, 0, st>>>(nel, g->d_order, g->d_growptr, g->d_gadj,
                                                  g->d_segof, table, (unsigned)(slots - 1), nb,
                                                  nb + nseg);
    RSB_LAUNCH_CHECK();
    RSB_READ(g, {h.data(), nb, sizeof(int) * h.size()});
    if (!h[nseg]) break;
    if (slots >= ((int64_t)1 << 31)) RSB_FAIL(2, "too many neighbour pairs");
  }
  std::copy(h.begin(), h.begin() + nseg, nbrs);
  return 0;
}

// Device-wide radix sorts and scans (rocPRIM building blocks), in place on
// the caller's arrays.  LSD radix sorting is stable, which every sort of the
// partitioner relies on: equal keys keep the current order.
#include <cstring>
#include <rocprim/rocprim.hpp>

#include "state.hpp"

static int ensure_tmp(rsbgpu *g, size_t bytes) {
  if (bytes <= g->sort_tmp_bytes && g->d_sort_tmp) return 0;
  const size_t old = g->d_sort_tmp ? g->sort_tmp_bytes : 0;
  g->sort_tmp_bytes = 0;
  RSB_TRY(rsb_retire(g, g->d_sort_tmp, old));
  size_t got = 0;
  RSB_TRY(rsb_dev_malloc_grown(g, &g->d_sort_tmp, bytes + 256, old, &got));
  g->sort_tmp_bytes = got;
  return 0;
}

static int ensure_kv(rsbgpu *g, size_t n) {
  if (n <= g->sort_cap && g->d_k1) return 0;
  const size_t old = g->sort_cap;
  g->sort_cap = 0;
  RSB_TRY(rsb_retire(g, g->d_k1, old * sizeof(uint64_t)));
  RSB_TRY(rsb_retire(g, g->d_v1, old * sizeof(int)));
  RSB_TRY(rsb_dev_malloc((void **)&g->d_k1, n * sizeof(uint64_t)));
  RSB_TRY(rsb_dev_malloc((void **)&g->d_v1, n * sizeof(int)));
  g->sort_cap = n;
  return 0;
}

// The radix sort's single-pass (onesweep) form costs about 22 us per 8 key
// bits whatever the size, the merge sort about one launch per doubling.  Pairs,
// merge / onesweep in us: 200,000 keys of 64 bits 75 / 207, of 32 bits 60 / 120,
// of 12 bits 59 / 63; 300,000 keys of 64 bits 130 / 215, of 32 bits 120 / 121,
// of 20 bits 118 / 92; 1M keys of 64 bits 199 / 242, of 44 bits 194 / 183, of
// 32 bits 164 / 135; 1.5M keys of 64 bits 234 / 262, of 44 bits 227 / 199.
static bool sort_by_merging(int64_t n, int bits) {
  return n <= (bits > 32 ? 1 << 20 : 1 << 18);
}
template <unsigned MERGE_MAX>
using sort_cfg = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config,
                                            rocprim::default_config, MERGE_MAX>;
#define SORT_MERGE (1u << 20)  // every size that the rule merges
#define SORT_ONESWEEP 1u

template <unsigned M, typename K>
static hipError_t pairs(rsbgpu *g, void *tmp, size_t &bytes, const K *keys, K *kout,
                        const int *vals, int *vout, int64_t n, int bb, int eb) {
  return rocprim::radix_sort_pairs<sort_cfg<M>>(tmp, bytes, keys, kout, vals, vout, (size_t)n, bb,
                                                eb, g->stream);
}
template <typename K>
static int sort_into(rsbgpu *g, const K *keys, K *kout, const int *vals, int *vout, int64_t n,
                     int bb, int eb) {
  auto *sort = sort_by_merging(n, eb - bb) ? pairs<SORT_MERGE, K> : pairs<SORT_ONESWEEP, K>;
  size_t bytes = 0;
  RSB_TRY(sort(g, nullptr, bytes, keys, kout, vals, vout, n, bb, eb));
  int rc = ensure_tmp(g, bytes);
  if (rc) return rc;
  bytes = g->sort_tmp_bytes;
  RSB_TRY(sort(g, g->d_sort_tmp, bytes, keys, kout, vals, vout, n, bb, eb));
  return 0;
}

int rsb_sort_pairs_u64(rsbgpu *g, uint64_t *keys, int *vals, int64_t n, int bb, int eb) {
  if (n <= 1) return 0;
  int rc = ensure_kv(g, (size_t)n);
  if (rc) return rc;
  if ((rc = sort_into(g, keys, g->d_k1, vals, g->d_v1, n, bb, eb))) return rc;
  RSB_TRY(hipMemcpyAsync(keys, g->d_k1, n * sizeof(uint64_t), hipMemcpyDeviceToDevice,
                         g->stream));
  RSB_TRY(hipMemcpyAsync(vals, g->d_v1, n * sizeof(int), hipMemcpyDeviceToDevice, g->stream));
  return 0;
}

int rsb_sort_pairs_u32(rsbgpu *g, uint32_t *keys, int *vals, int64_t n, int bb, int eb) {
  if (n <= 1) return 0;
  int rc = ensure_kv(g, (size_t)n);
  if (rc) return rc;
  uint32_t *k1 = (uint32_t *)g->d_k1;
  if ((rc = sort_into(g, keys, k1, vals, g->d_v1, n, bb, eb))) return rc;
  RSB_TRY(hipMemcpyAsync(keys, k1, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, g->stream));
  RSB_TRY(hipMemcpyAsync(vals, g->d_v1, n * sizeof(int), hipMemcpyDeviceToDevice, g->stream));
  return 0;
}

// Stable sorts of n values by their keys into another array (the keys' array
// is scratch afterwards): no copies back.
int rsb_sort_vals_u64(rsbgpu *g, const uint64_t *keys, const int *vals, int *out, int64_t n,
                      int bb, int eb) {
  int rc = ensure_kv(g, (size_t)n);
  if (rc) return rc;
  return sort_into(g, keys, g->d_k1, vals, out, n, bb, eb);
}

int rsb_sort_vals_u32(rsbgpu *g, const uint32_t *keys, const int *vals, int *out, int64_t n,
                      int bb, int eb) {
  int rc = ensure_kv(g, (size_t)n);
  if (rc) return rc;
  return sort_into(g, keys, (uint32_t *)g->d_k1, vals, out, n, bb, eb);
}

// Keys alone, into the handle's own array: *out, valid until its next sort.
template <unsigned M, typename K>
static hipError_t only_keys(rsbgpu *g, void *tmp, size_t &bytes, const K *keys, K *out, int64_t n,
                            int eb) {
  return rocprim::radix_sort_keys<sort_cfg<M>>(tmp, bytes, keys, out, (size_t)n, 0, eb, g->stream);
}
template <typename K>
static int sort_keys(rsbgpu *g, const K *keys, const K **out, int64_t n, int eb) {
  auto *sort = sort_by_merging(n, eb) ? only_keys<SORT_MERGE, K> : only_keys<SORT_ONESWEEP, K>;
  int rc = ensure_kv(g, (size_t)n);
  if (rc) return rc;
  K *sorted = (K *)g->d_k1;
  size_t bytes = 0;
  RSB_TRY(sort(g, nullptr, bytes, keys, sorted, n, eb));
  if ((rc = ensure_tmp(g, bytes))) return rc;
  bytes = g->sort_tmp_bytes;
  RSB_TRY(sort(g, g->d_sort_tmp, bytes, keys, sorted, n, eb));
  *out = sorted;
  return 0;
}
int rsb_sort_keys_u32(rsbgpu *g, const uint32_t *keys, const uint32_t **out, int64_t n, int eb) {
  return sort_keys(g, keys, out, n, eb);
}
int rsb_sort_keys_u64(rsbgpu *g, const uint64_t *keys, const uint64_t **out, int64_t n, int eb) {
  return sort_keys(g, keys, out, n, eb);
}

int rsb_exclusive_scan_i64(rsbgpu *g, const int64_t *in, int64_t *out, int64_t n) {
  if (n <= 0) return 0;
  size_t bytes = 0;
  RSB_TRY(rocprim::exclusive_scan(nullptr, bytes, in, out, (int64_t)0, (size_t)n,
                                  rocprim::plus<int64_t>(), g->stream));
  int rc = ensure_tmp(g, bytes);
  if (rc) return rc;
  bytes = g->sort_tmp_bytes;
  RSB_TRY(rocprim::exclusive_scan(g->d_sort_tmp, bytes, in, out, (int64_t)0, (size_t)n,
                                  rocprim::plus<int64_t>(), g->stream));
  return 0;
}

int rsb_exclusive_scan_i32(rsbgpu *g, const int *in, int *out, int64_t n) {
  if (n <= 0) return 0;
  size_t bytes = 0;
  RSB_TRY(rocprim::exclusive_scan(nullptr, bytes, in, out, 0, (size_t)n, rocprim::plus<int>(),
                                  g->stream));
  int rc = ensure_tmp(g, bytes);
  if (rc) return rc;
  bytes = g->sort_tmp_bytes;
  RSB_TRY(rocprim::exclusive_scan(g->d_sort_tmp, bytes, in, out, 0, (size_t)n,
                                  rocprim::plus<int>(), g->stream));
  return 0;
}

// attention_deal.h - how the attention backward deals the (key tile, query tile) pairs of a head to
// workgroups (Deal, attention_bwd.hip). Plain integer arithmetic, compiled for the device, for its
// launcher and, without HIP, for the tests.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define HK_ATTN_FN __host__ __device__ inline
#else
#define HK_ATTN_FN inline
#endif

namespace hk {
namespace attn {

constexpr int kBKV = 128;  // keys per key tile
constexpr int kBQ = 64;    // queries per query tile

// Query tiles of key tile kt: all of them, or under causal masking from the one that holds the
// tile's first key.
HK_ATTN_FN int query_tiles(int64_t T, bool causal, int kt) {
  const int64_t first = causal ? static_cast<int64_t>(kt) * kBKV / kBQ * kBQ : 0;
  return static_cast<int>((T - first + kBQ - 1) / kBQ);
}
HK_ATTN_FN int key_items(int64_t T, bool causal, int kt, int chunk) {
  return (query_tiles(T, causal, kt) + chunk - 1) / chunk;
}
// Items of a head before key tile kt (kt == nkt: all of them), without a walk over the key tiles. Under
// causal masking key tile kt has two query tiles fewer than the one before it, so the last m key tiles
// have sum over j < m of ceil((last + 2 j) / chunk) items, last = 1 or 2: for even chunks the summand
// grows by one every chunk / 2 tiles, for odd ones by two every chunk tiles, the first `ones` of which
// have one item (and the first `ones` after each step one fewer than the others).
HK_ATTN_FN int first_item(int64_t T, bool causal, int nkt, int kt, int chunk) {
  if (!causal) return kt * key_items(T, false, 0, chunk);
  const int last = query_tiles(T, true, nkt - 1);
  auto tail = [&](int m) {
    if (chunk % 2 == 0) {
      const int d = chunk / 2, q = m / d;
      return m + d * (q * (q - 1) / 2) + q * (m - q * d);
    }
    const int q = m / chunk, r = m - q * chunk, ones = (chunk - last + 2) / 2;
    return chunk * q * (q - 1) + q * (2 * chunk - ones) + 2 * r * q + 2 * r - (r < ones ? r : ones);
  };
  return tail(nkt) - tail(nkt - kt);
}
// The key tile of item `item`: the last one whose first item is not behind it.
HK_ATTN_FN int item_key_tile(int64_t T, bool causal, int nkt, int item, int chunk) {
  if (!causal) return item / key_items(T, false, 0, chunk);
  int lo = 0, hi = nkt - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (first_item(T, true, nkt, mid, chunk) <= item) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Query tiles per workgroup: the number with the least modelled time. A workgroup takes about 11 us
// plus 3 us per query tile; the launch lasts as long as its longest workgroup and, with more
// workgroups than CUs (one runs per CU), as the work per CU; a split adds the sum's 5 us. Large
// grids stay unsplit. The pick is made on every call, so its loop has no walk over the key tiles (host
// time of one causal head of 65,536: 561 us with one, 16 without; 12 of 8,192: 20 and 12). Whole backward on MI355X, us unsplit and as picked: 12 causal heads at
// T = 1024 66.5 and 35.2 (4 tiles), 24 heads at T = 333 34.1 and 26.9 (2 tiles).
inline int pick_chunk(int64_t T, bool causal, int nkt, int64_t nbh, int cus) {
  const int most = query_tiles(T, causal, 0);
  double best = 0.0;
  int best_chunk = most;
  if (nkt * nbh >= int64_t{4} * cus) return most;
  const int64_t tiles = first_item(T, causal, nkt, nkt, 1);  // query tiles of all key tiles
  for (int chunk = most; chunk >= 1; --chunk) {
    const int64_t wgs = first_item(T, causal, nkt, nkt, chunk);
    if (wgs * nbh > int64_t{8} * cus) break;
    const double longest = 11.0 + 3.0 * chunk;
    const double share = (11.0 * static_cast<double>(wgs) + 3.0 * static_cast<double>(tiles)) *
                         static_cast<double>(nbh) / cus;
    double cost = wgs * nbh <= cus ? longest : (share > longest ? share : longest) + 0.3 * longest;
    if (wgs > nkt) cost += 5.0;
    if (chunk == most || cost < 0.95 * best) {
      best = cost;
      best_chunk = chunk;
    }
  }
  return best_chunk;
}

}  // namespace attn
}  // namespace hk

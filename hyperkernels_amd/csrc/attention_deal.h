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
inline int query_tiles(int T, bool causal, int kt) {
  return (T - (causal ? kt * kBKV : 0) + kBQ - 1) / kBQ;
}

// A head's items, numbered key tile by key tile: each is a key tile and at most `chunk` of its query
// tiles. Under causal masking key tile kt has two query tiles fewer than the one before it.
struct Deal {
  int nkt, chunk;
  float inv;  // 1 / chunk
  int items;  // of all key tiles
  int last;   // causal: query tiles (1 or 2) of the last key tile; else the items of each key tile
  bool causal;

  // a / chunk or a / (chunk / 2): every count here is under 2^21, where (a + 1/2) / n in fp32 has the
  // whole part of a / n. (An integer division is a chain of some 40 instructions on the device; with
  // those, a workgroup took 0.8 us to find its item.)
  HK_ATTN_FN static int over(int a, float inv) {
    return static_cast<int>((static_cast<float>(a) + 0.5f) * inv);
  }
  // Items of the last m key tiles under causal masking: sum over j < m of ceil((last + 2 j) / chunk). For
  // even chunks the summand grows by one every chunk / 2 tiles, for odd ones by two every chunk tiles,
  // the first `ones` of which have one item (and the first `ones` after each step one fewer than the
  // others).
  HK_ATTN_FN int tail(int m) const {
    if (chunk % 2 == 0) {
      const int d = chunk / 2, q = over(m, 2.0f * inv);
      return m + d * (q * (q - 1) / 2) + q * (m - q * d);
    }
    const int q = over(m, inv), r = m - q * chunk, ones = (chunk - last + 2) / 2;
    return chunk * q * (q - 1) + q * (2 * chunk - ones) + 2 * r * q + 2 * r - (r < ones ? r : ones);
  }
  // Items of key tile kt, and those before it (kt == nkt: all), without a walk over the key tiles.
  HK_ATTN_FN int key_items(int kt) const {
    return causal ? over(last + 2 * (nkt - 1 - kt) + chunk - 1, inv) : last;
  }
  HK_ATTN_FN int first_item(int kt) const { return causal ? items - tail(nkt - kt) : kt * last; }
  // The key tile of an item: the last one whose first item is not behind it.
  HK_ATTN_FN int key_tile(int item) const {
    if (!causal) return over(item, 1.0f / static_cast<float>(last));
    int lo = 0, hi = nkt - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) / 2;
      if (first_item(mid) <= item) lo = mid;
      else hi = mid - 1;
    }
    return lo;
  }
};

inline Deal make_deal(int T, bool causal, int chunk) {
  Deal d{(T + kBKV - 1) / kBKV, chunk, 1.0f / static_cast<float>(chunk), 0, 0, causal};
  if (causal) {
    d.last = query_tiles(T, true, d.nkt - 1);
    d.items = d.tail(d.nkt);
  } else {
    d.last = Deal::over(query_tiles(T, false, 0) + chunk - 1, d.inv);
    d.items = d.nkt * d.last;
  }
  return d;
}

// Query tiles per workgroup: the number with the least modelled time. A workgroup takes about 11 us
// plus 3 us per query tile; the launch lasts as long as its longest workgroup and, with more
// workgroups than CUs (one runs per CU), as the work per CU; a split adds the sum's 5 us. Large
// grids stay unsplit. The pick is made on every call, so its loop has no walk over the key tiles (host
// time of one causal head of 65,536: 561 us with one, 16 without; 12 of 8,192: 20 and 12). Whole backward on MI355X, us unsplit and as picked: 12 causal heads at
// T = 1024 66.5 and 35.2 (4 tiles), 24 heads at T = 333 34.1 and 26.9 (2 tiles).
inline int pick_chunk(int T, bool causal, int64_t nbh, int cus) {
  const int most = query_tiles(T, causal, 0), nkt = (T + kBKV - 1) / kBKV;
  double best = 0.0;
  int best_chunk = most;
  if (nkt * nbh >= int64_t{4} * cus) return most;
  const int64_t tiles = make_deal(T, causal, 1).items;  // query tiles of all key tiles
  for (int chunk = most; chunk >= 1; --chunk) {
    const int64_t wgs = make_deal(T, causal, chunk).items;
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

"""The attention backward's dealing of key and query tiles to workgroups (csrc/attention_deal.h), compiled
for the CPU: the closed forms against a walk over the key tiles, and the pick against one that walks them."""
from __future__ import annotations

import subprocess

from conftest import ROOT

DRIVER = r"""
#include <initializer_list>
#include <stdio.h>
#include "attention_deal.h"
using namespace hk::attn;

static int pick_by_walk(int T, bool causal, int nkt, int64_t nbh, int cus) {
  const int most = query_tiles(T, causal, 0);
  if (nkt * nbh >= int64_t{4} * cus) return most;
  double best = 0.0;
  int best_chunk = most;
  for (int chunk = most; chunk >= 1; --chunk) {
    int64_t wgs = 0, tiles = 0;
    for (int kt = 0; kt < nkt; ++kt) {
      wgs += (query_tiles(T, causal, kt) + chunk - 1) / chunk;
      tiles += query_tiles(T, causal, kt);
    }
    if (wgs * nbh > int64_t{8} * cus) break;
    const double longest = 11.0 + 3.0 * chunk;
    const double share = (11.0 * double(wgs) + 3.0 * double(tiles)) * double(nbh) / cus;
    double cost = wgs * nbh <= cus ? longest : (share > longest ? share : longest) + 0.3 * longest;
    if (wgs > nkt) cost += 5.0;
    if (chunk == most || cost < 0.95 * best) best = cost, best_chunk = chunk;
  }
  return best_chunk;
}

int main() {
  for (int T : {1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 333, 520, 1000, 1024, 1025, 2031, 4097, 8192,
                16383, 65536, 130000})
    for (int causal = 0; causal < 2; ++causal) {
      const int nkt = (T + kBKV - 1) / kBKV, most = query_tiles(T, causal, 0);
      for (int chunk = 1; chunk <= most; chunk += most > 600 && chunk > 40 ? 37 : 1) {
        const Deal d = make_deal(T, causal, chunk);
        int sum = 0;
        for (int kt = 0; kt < nkt; ++kt) {
          const int n = (query_tiles(T, causal, kt) + chunk - 1) / chunk;
          if (d.key_items(kt) != n || d.first_item(kt) != sum) return printf("items\n"), 1;
          for (int i : {sum, sum + n / 2, sum + n - 1})
            if (d.key_tile(i) != kt) return printf("key tile\n"), 1;
          sum += n;
        }
        if (d.items != sum || d.nkt != nkt) return printf("all items\n"), 1;
      }
      for (int nbh : {1, 2, 4, 12, 24, 96, 400})
        for (int cus : {64, 256})
          if (pick_chunk(T, causal, nbh, cus) != pick_by_walk(T, causal, nkt, nbh, cus))
            return printf("pick T %d causal %d heads %d\n", T, causal, nbh), 1;
    }
  printf("ok\n");
  return 0;
}
"""


def test_closed_forms_equal_the_walk(tmp_path):
    src, exe = tmp_path / "deal.cpp", tmp_path / "deal"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", f"-I{ROOT / 'hyperkernels_amd' / 'csrc'}",
                    str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout

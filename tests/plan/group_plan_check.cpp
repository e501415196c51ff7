// Property check of grouped decode plans (build_decode_groups,
// orionserve-rs_amd/csrc/decode_plan.cpp), host only.  For random batches a
// grouped plan must hold group_waves records per planned (row, KV head), in
// order, whose pieces cover [0, position] exactly once from 16-token-aligned
// starts, with the row's piece count, at most 32 tokens, the
// right table offset and first block, and empty records after them; and the
// plan must stay ungrouped where a row is longer than 32 tokens per wave, the
// pairs outnumber the CUs, rows share blocks, or nothing is split.  Prints one
// line per failure and a summary; exit status 1 on any failure.
#include "kernels.hpp"

#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

int main(int argc, char** argv) {
  const int trials = argc > 1 ? atoi(argv[1]) : 2000;
  std::mt19937 rng(20261205);
  int fails = 0, grouped = 0;
  auto fail = [&](int trial, const char* what) {
    if (fails++ < 20) printf("trial %d: %s\n", trial, what);
  };
  for (int trial = 0; trial < trials; ++trial) {
    const int rows = 1 + rng() % 70, bs = 1 << (rng() % 8), hkv = 1 + rng() % 8;
    const int waves = orion::kGroupWaves[rng() % 2];
    const int maxctx = trial % 3 == 0 ? 40 : trial % 3 == 1 ? 32 * waves : 32 * waves + 100;
    std::vector<uint32_t> pos(rows), ids;
    std::vector<int32_t> row_seq(rows);
    std::vector<int64_t> off(rows + 1, 0);
    std::vector<uint8_t> skip(rows, 0);
    int planned = 0, longest = 0;
    for (int r = 0; r < rows; ++r) {
      pos[r] = rng() % maxctx;
      row_seq[r] = r;
      skip[r] = trial % 5 == 0 && rng() % 3 == 0;
      for (int j = 0; j <= (int)pos[r] / bs; ++j) ids.push_back(trial % 7 ? (uint32_t)ids.size() : rng() % 100000);
      off[r + 1] = (int64_t)ids.size();
      if (!skip[r]) ++planned, longest = std::max(longest, (int)pos[r] + 1);
    }
    orion::DecodePlanHost plan;
    orion::build_decode_plan(pos.data(), row_seq.data(), off.data(), ids.data(), rows, hkv, bs,
                             2048, skip.data(), &plan, 0);
    orion::build_decode_groups(pos.data(), row_seq.data(), off.data(), ids.data(), rows, hkv, bs,
                               256, waves, skip.data(), &plan);
    const bool want = plan.max_splits > 1 && plan.stream_kv && planned * hkv <= 256 && longest <= 32 * waves &&
                      bs <= 32;
    if ((plan.group_waves != 0) != want) fail(trial, "grouped or not");
    if (!plan.group_waves) continue;
    ++grouped;
    if (plan.groups.size() != (size_t)planned * hkv * waves) {
      fail(trial, "record count");
      continue;
    }
    size_t at = 0;
    for (int r = 0; r < rows; ++r) {
      if (skip[r]) continue;
      for (int h = 0; h < hkv; ++h) {
        int next = 0, n = 0;
        for (int s = 0; s < waves; ++s, ++at) {
          const orion::DecodeWork& w = plan.groups[at];
          if (w.item != r * hkv + h || w.split != s) fail(trial, "order");
          if (w.end == 0) continue;
          if (n != s || w.start != next || w.start % 16 || w.end <= w.start) fail(trial, "piece");
          if (w.end - w.start > 32 || (w.end - 1) / bs - w.start / bs + 1 > 32)
            fail(trial, "piece length");
          if (w.tbl_off != off[r] + w.start / bs || w.blk0 != (int32_t)ids[w.tbl_off])
            fail(trial, "table");
          next = w.end;
          ++n;
        }
        if (next != (int)pos[r] + 1) fail(trial, "cover");
        for (int s = 0; s < waves; ++s)
          if (plan.groups[at - waves + s].nsplit != n) fail(trial, "piece count");
      }
    }
  }
  printf("%d trials %d grouped %d failures\n", trials, grouped, fails);
  return fails != 0;
}

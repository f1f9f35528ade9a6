"""The rule that picks the decode splits' length, on the host: every split of a
batch fits the work list, whatever the shape and the lengths, and the general
kernel splits nothing where it has no merge launch."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

# Replays the device's choice for batches of a shape: random lengths from one
# to the table's reach, evenly or unevenly spread, some of them not decodes.
PROGRAM = r"""
#include "worklists.h"
#include <algorithm>
#include <cstdio>
#include <random>

using namespace mvllm;

int main() {
  std::mt19937_64 rng(7);
  auto log_int = [&](double lo, double hi) {
    return static_cast<int64_t>(std::exp(std::uniform_real_distribution<double>(std::log(lo), std::log(hi + 1))(rng)));
  };
  const int32_t head_counts[] = {1, 2, 3, 4, 5, 8, 9, 16, 32, 64}, dims[] = {64, 96, 128};
  int64_t batches = 0, whole = 0;
  for (int shape = 0; shape < 20000; ++shape) {
    AttnArgs a = {};
    a.num_requests = log_int(1, 2000);
    a.num_kv_heads = head_counts[rng() % 10];
    a.group = 1 + static_cast<int32_t>(rng() % 16);
    a.head_dim = dims[rng() % 3];
    a.num_cus = rng() % 4 ? 256 : 64;
    a.merge_apart = static_cast<int32_t>(rng() % 2);
    const int64_t reach = log_int(1, 140000);
    // The workspace's slots, whose split length is 64 to 2,048 (16 or more asked for).
    const int64_t layout = 64 << (rng() % 6);
    const int64_t capacity = a.num_requests * ((reach + 15 + layout) / layout);
    const bool decodes = rng() % 2, general = rng() % 4 == 0;
    if (general) a.merge_apart = general_merges(reach, 0);
    a.item_capacity = item_slots(a.num_requests, reach, capacity, a.num_cus, a.head_dim, a.num_kv_heads, decodes, general);
    a.rule = split_rule(a, general);
    for (int trial = 0; trial < 4; ++trial, ++batches) {
      const int64_t least = trial == 0 ? reach : trial == 1 ? 1 : log_int(1, reach);
      const bool others = trial == 3;
      std::vector<int64_t> tokens;
      int64_t pages = 0, longest = 0, seen = 0;
      for (int64_t r = 0; r < a.num_requests; ++r) {
        // Visible tokens from a 16-aligned position on.
        const int64_t v = others && rng() % 3 == 0 ? 0 : least + static_cast<int64_t>(rng() % (reach - least + 1));
        tokens.push_back(v);
        pages += (v + 15) / 16;
        longest = std::max(longest, v);
        seen += v > 0;
      }
      const int32_t split = choose_split(16 * pages, static_cast<int32_t>(longest), static_cast<int32_t>(seen), others, a.rule);
      int64_t items = 0;
      for (int64_t v : tokens) items += (v + split - 1) / split;
      whole += split >= longest;
      if (split < 16 || split % 16 || split > kMaxSplit || items > a.item_capacity ||
          (general && !a.merge_apart && split < longest)) {
        std::printf("requests %lld reach %lld heads %d group %d dim %d slots %lld split %d items %lld\n",
                    (long long)a.num_requests, (long long)reach, a.num_kv_heads, a.group, a.head_dim,
                    (long long)a.item_capacity, split, (long long)items);
        return 1;
      }
    }
  }
  std::printf("%lld batches, %lld whole\n", (long long)batches, (long long)whole);
  return 0;
}
"""


def test_every_split_fits_the_work_list(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("hipcc not found")
    source, program = tmp_path / "rule.hip", tmp_path / "rule"
    source.write_text(PROGRAM)
    subprocess.run(
        [hipcc, "--offload-host-only", "-O1", "-std=c++17", "-Wno-unused-function", f"-I{ROOT / 'include'}",
         f"-I{ROOT / 'micro-vllm_amd' / 'csrc'}", str(source), "-o", str(program)],
        check=True, capture_output=True, text=True, timeout=300,
    )
    done = subprocess.run([str(program)], capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stdout

// How a gated batch is split into runs that share their launches. Host code
// only: no HIP types, so that the split can be checked without a GPU.
#pragma once

#include <algorithm>
#include <cstddef>
#include <utility>
#include <vector>

namespace sc {

constexpr int kMaxFusedSet = 8;  // channels of one shape sharing a launch

// The runs [a, e) of a gated batch of n instances: consecutive instances that
// can share a launch (shared(a): how many from a on, at least one), the first
// run of at most four. Nothing hides the first run's front, so it is shorter:
// 16 x (16 x 2^18) at 60 % flagged take 1.68 ms in runs of 8 and 8, 1.64 in 4,
// 8 and 4, 1.67 in 2, 4, 8 and 2 (whose second front outlasts the first tree).
template <typename Shared>
std::vector<std::pair<size_t, size_t>> gated_runs(size_t n, Shared&& shared) {
  std::vector<std::pair<size_t, size_t>> runs;
  for (size_t a = 0; a < n; a = runs.back().second) {
    const size_t most = runs.empty() ? 4 : kMaxFusedSet;
    runs.push_back({a, a + std::min<size_t>(shared(a), most)});
  }
  return runs;
}

}  // namespace sc

// Splits batches of given sizes into gated runs and prints them, one batch per
// line: "n width: length length ...". Arguments: pairs of the number of
// instances and of how many neighbours can share a launch. A split that does
// not advance ends the program with status 1 (no memory is filled).
#include <cstdio>
#include <cstdlib>

#include "../../seticore_amd/csrc/batch_runs.h"

int main(int argc, char** argv) {
  for (int i = 1; i + 1 < argc; i += 2) {
    const size_t n = (size_t)std::atol(argv[i]), width = (size_t)std::atol(argv[i + 1]);
    size_t calls = 0;
    const auto runs = sc::gated_runs(n, [&](size_t a) {
      if (a >= n || ++calls > n) {
        std::fprintf(stderr, "%zu instances, %zu together: the split does not end\n", n, width);
        std::exit(1);
      }
      return std::min(width, n - a);
    });
    std::printf("%zu %zu:", n, width);
    size_t at = 0;
    for (const auto& r : runs) {
      if (r.first != at || r.second <= r.first) {
        std::fprintf(stderr, "run [%zu, %zu) after %zu\n", r.first, r.second, at);
        return 1;
      }
      std::printf(" %zu", r.second - r.first);
      at = r.second;
    }
    if (at != n) return 1;
    std::printf("\n");
  }
  return 0;
}

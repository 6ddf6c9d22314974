// The kernel shape under which a captured search is looked up: an untuned
// handle's follows the sample type, a tuned handle's is the caller's, whatever
// its default was. Returns 0 when all holds (host only, no device call).
#include <cstdio>

#include "../../seticore_amd/csrc/dd_internal.h"

int main() {
  int bad = 0;
  for (int T = 2; T <= 256; T *= 2)
    for (int N : {1000, 1 << 14, 1 << 16, 1 << 17, 1 << 18, 3 << 18, 1 << 20}) {
      sc::KernelShape set;  // as sc_dd_create leaves the handle
      sc::default_tuning(T, N, false, &set.lanes, &set.group, &set.prefetch);
      for (int dtype : {SC_F32, SC_F16, SC_BF16}) {
        sc::KernelShape want;
        sc::default_tuning(T, N, dtype != SC_F32, &want.lanes, &want.group, &want.prefetch);
        const sc::KernelShape untuned = sc::search_shape(T, N, dtype, false, set);
        // The caller names the shape the handle holds already.
        const sc::KernelShape tuned = sc::search_shape(T, N, dtype, true, set);
        if (!(untuned == want) || !(tuned == set) || (untuned == tuned) != (want == set)) {
          std::printf("%d x %d, type %d\n", T, N, dtype);
          bad = 1;
        }
      }
    }
  // 256 x 2^18 in 16 bits: 16 drift blocks per workgroup by default, 256 asked for.
  const sc::KernelShape asked = {4, 256, 1};
  if (sc::search_shape(256, 1 << 18, SC_F16, false, asked) ==
      sc::search_shape(256, 1 << 18, SC_F16, true, asked)) {
    std::printf("a search with the default and one with the asked shape are told apart by nothing\n");
    bad = 1;
  }
  return bad;
}

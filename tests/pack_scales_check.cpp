// Host check of unified_scale (srg_amd/csrc/tdbp_pack.h): the pulses of a call
// take their final scales in any order, each from a largest value over scales of
// which any part may be final already, and end with the same scales.  Exits 1
// at the first call that does not.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "../srg_amd/csrc/tdbp_pack.h"

int main() {
  std::mt19937 rng(1);
  for (int trial = 0; trial < 20000; ++trial) {
    const int dtype = trial % 3 == 0 ? TDBP_CF16 : trial % 3 == 1 ? TDBP_CI16 : TDBP_CBF16;
    const int L = 1 + rng() % 9, spread = 1 + rng() % 40;
    std::vector<float> own(L);
    for (float& s : own) {
      const int kind = rng() % 8;
      s = kind < 2 || trial % 50 == 0 ? 0.f
          : kind == 2                 ? 1.f   // infinite samples
                                      : std::ldexp(1.f, -100 + (int)(rng() % spread));
    }
    float m = 0.f;
    for (float s : own) m = std::max(m, s);
    std::vector<float> want(L), scale = own;
    for (int p = 0; p < L; ++p) want[p] = tdbp::unified_scale(own[p], m, dtype);
    std::vector<int> order(L);
    for (int p = 0; p < L; ++p) order[p] = p;
    std::shuffle(order.begin(), order.end(), rng);
    for (int p : order) {
      float seen = 0.f;   // each of the others' as it was or as it will be
      for (int i = 0; i < L; ++i)
        seen = std::max(seen, i == p ? own[p] : rng() % 2 ? scale[i] : own[i]);
      scale[p] = tdbp::unified_scale(own[p], seen, dtype);
    }
    if (scale != want) {
      std::printf("trial %d: %d pulses, largest scale %g\n", trial, L, m);
      return 1;
    }
  }
  return 0;
}

// Host check of the aperture fit's arithmetic (srg_amd/csrc/tdbp_geom.h):
// div_by equals the division bit for bit, and the four hermite_term added in
// order equal hermite4 bit for bit.  Exits 1 on the first difference.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

#include "../srg_amd/csrc/tdbp_geom.h"

static bool same(double a, double b) { return std::memcmp(&a, &b, sizeof a) == 0; }

int main() {
  std::mt19937_64 rng(7);
  std::uniform_real_distribution<double> um(1.0, 2.0), us(-1.0, 1.0);
  std::uniform_int_distribution<int> ue(-40, 40);
  auto draw = [&] { return std::ldexp(us(rng) < 0 ? -um(rng) : um(rng), ue(rng)); };
  for (long i = 0; i < 20000000; ++i) {
    const double b = draw(), a = i % 4 ? draw() : b * (1.0 + std::ldexp((double)(i % 64), -52));
    if (!same(tdbp::div_by(a, b, 1.0 / b), a / b)) {
      std::printf("div_by(%a, %a) differs\n", a, b);
      return 1;
    }
  }
  for (int i = 0; i < 200000; ++i) {
    // State vectors 10 s apart (or at uneven times), times in and around them.
    double t[4], x[12], v[12];
    const double t0 = 43200.0 + 1e4 * us(rng), step = i % 2 ? 10.0 : um(rng) * 7.0;
    for (int k = 0; k < 4; ++k) {
      t[k] = t0 + k * step + (i % 3 == 2 ? 0.3 * us(rng) : 0.0);
      for (int c = 0; c < 3; ++c) {
        x[3 * k + c] = 7.0e6 * us(rng);
        v[3 * k + c] = 7.6e3 * us(rng);
      }
    }
    const double time = i % 5 == 4 ? t[i & 3] : t0 + step * (1.5 + 3.0 * us(rng));
    double p[3], w[3], ps[3] = {0., 0., 0.}, ws[3] = {0., 0., 0.};
    tdbp::hermite4(x, v, t, time, p, w);
    for (int k = 0; k < 4; ++k) {
      tdbp::HermiteNode n;
      double a[3], b[3];
      if (!tdbp::hermite_node(t, x, v, k, &n)) return 1;
      tdbp::hermite_term(n, time, a, b);
      for (int c = 0; c < 3; ++c) {
        ps[c] = ps[c] + a[c];
        ws[c] = ws[c] + b[c];
      }
    }
    for (int c = 0; c < 3; ++c)
      if (!(ps[c] == p[c]) || !(ws[c] == w[c])) {
        std::printf("case %d: %a %a, %a %a\n", i, ps[c], p[c], ws[c], w[c]);
        return 1;
      }
  }
  // Two equal times: no reciprocal, the split is refused.
  double t[4] = {0., 10., 10., 30.}, z[12] = {0.};
  tdbp::HermiteNode n;
  return tdbp::hermite_node(t, z, z, 1, &n) ? 1 : 0;
}

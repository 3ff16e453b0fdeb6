// Host check of the 1024- and 2048-point FFT pairs of srg_amd/csrc/tdbp_osfft.h
// (the interferograms' upsampling of narrower images), run through the header's
// own stages, layout and per-thread registers on random complex data:
//   DIF: position p = (N/16) d0 + R d1 + d2 holds bin d0 + 16 d1 + 256 d2 of the
//        direct DFT (long double; relative RMS over all bins);
//   round trip: conj(DIT(conj(DIF(x)))) = N x.
// Prints the figures; exits 1 when a bound fails.
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "../srg_amd/csrc/tdbp_osfft.h"

template <int N>
bool check(const std::vector<float2>& tw) {
  std::vector<float2> x(N);
  std::mt19937_64 rng(N);
  std::normal_distribution<float> g(0.f, 1.f);
  for (float2& v : x) v = make_float2(g(rng), g(rng));
  std::vector<float2> y = x;
  tdbp::up_dif_host<N>(y.data(), tw.data());
  const long double pi = 3.141592653589793238462643383279502884L;
  long double num = 0, den = 0, n2 = 0, d2 = 0;
  const int r = N / 256;
  for (int p = 0; p < N; ++p) {
    const int k = p / (N / 16) + 16 * ((p / r) % 16) + 256 * (p % r);
    long double re = 0, im = 0;
    for (int n = 0; n < N; ++n) {
      const long double a = -2 * pi * ((long long)n * k % N) / N;
      const long double c = cosl(a), s = sinl(a);
      re += x[n].x * c - x[n].y * s;
      im += x[n].x * s + x[n].y * c;
    }
    num += (y[p].x - re) * (y[p].x - re) + (y[p].y - im) * (y[p].y - im);
    den += re * re + im * im;
  }
  for (float2& v : y) v.y = -v.y;
  tdbp::up_dit_host<N>(y.data(), tw.data());
  for (int i = 0; i < N; ++i) {
    const long double re = y[i].x / (long double)N, im = -y[i].y / (long double)N;
    n2 += (re - x[i].x) * (re - x[i].x) + (im - x[i].y) * (im - x[i].y);
    d2 += (long double)x[i].x * x[i].x + (long double)x[i].y * x[i].y;
  }
  const double dif = std::sqrt((double)(num / den)), rt = std::sqrt((double)(n2 / d2));
  std::printf("fft%d relative RMS error: DIF %.3e, round trip %.3e\n", N, dif, rt);
  return dif < 1e-6 && rt < 2e-6;
}

int main() {
  std::vector<float2> tw(tdbp::kOsN);
  for (int m = 0; m < tdbp::kOsN; ++m) {
    const double a = -2.0 * 3.141592653589793238462643383279502884 * m / tdbp::kOsN;
    tw[m] = make_float2((float)std::cos(a), (float)std::sin(a));
  }
  const bool a = check<1024>(tw), b = check<2048>(tw);
  return a && b ? 0 : 1;
}

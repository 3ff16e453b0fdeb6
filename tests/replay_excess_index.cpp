// Host replay of the gather addressing of two forms in
// srg_amd/csrc/tdbp_kernels.hip that replay_mixed_index.cpp does not hold, over
// every tile, wave, lane and pulse of the bursts in a scene file:
//   split: the mixed kernel's split tiles (four waves on one 4 x 16 tile, a
//     quarter of a stage's pulses each, the pixel's fraction fa added to the
//     index rather than to the quadratic).  Local index in [0, 2048), sample
//     index in [0, S - 2], scalar offset in 32 bits, and the index within its
//     FP32 rounding (two steps of 2^-14 below 1024) of the pair's range.
//   fp64: the FP64 kernel's tiles (shape TILE_ROWS, STACK), blocks of pulses about
//     their centres.  Every pulse in a lane's window gathered once; index in [0,
//     r_hi], rows' offsets in 31 bits, and the index's range within 5e-10 m of
//     the pair's (fit 1e-10, look vector 1e-10, block 2e-11, FP64 roundings of R
//     and R0 1.2e-10 each).
// Stages that fail the safety test, and waves without a fit, take checked pairs
// in the kernels and are not replayed.  Scene file as for replay_mixed_index.cpp.
// Usage: replay_excess_index FILE split | fp64 TILE_ROWS STACK
#define main replay_mixed_main
#include "replay_mixed_index.cpp"
#undef main

namespace {

struct Pixel {
  int azs = 0, aze = 0, key = INT_MAX;
  double x[3] = {0., 0., 0.};
  bool live() const { return aze > azs; }
};

// The pixels of a tile by thread (STACK 0: waves side by side, 1: stacked, 2: all
// on one tile); returns the reference thread or -1, and the tile's window.
int tile_pixels(const Burst& b, int TR, int STACK, int tile, int tiles_r, Pixel* px, int* wlo,
                int* whi) {
  const int TC = kWave / TR, WR = STACK == 1 ? 4 * TR : TR, WC = STACK == 0 ? 4 * TC : TC;
  const int band = tile / tiles_r, rt = tile - band * tiles_r;
  int ref = INT_MAX;
  *wlo = INT_MAX;
  *whi = -1;
  for (int tid = 0; tid < kBlock; ++tid) {
    const int wr = (STACK == 1 ? (tid >> 6) * TR : 0) + (tid & 63) / TC;
    const int wc = (STACK == 0 ? (tid >> 6) * TC : 0) + (tid & 63) % TC;
    const int row = rt * WR + wr, col = band * WC + wc;
    Pixel& p = px[tid] = Pixel();
    if (row >= b.nlines || col >= b.W || row >= b.nfit || col < b.firstpix || col > b.lastpix)
      continue;
    const double az = tdbp::pixel_azoff(&b.coef[3 * row], col, b.firstpix, b.lastpix, b.A, b.L);
    if (!(az > 0.)) continue;
    tdbp::pulse_window(az, b.A, b.L, &p.azs, &p.aze);
    if (!p.live()) continue;
    tdbp::dem_to_ecef(row, b.firstline, col, b.firstlat, b.deltalat, b.firstlon, b.deltalon,
                      (double)b.dem[(size_t)row * b.W + col], p.x);
    ref = std::min(ref, (std::abs(2 * wr - WR) + std::abs(2 * wc - WC)) * 256 + tid);
    *wlo = std::min(*wlo, p.azs);
    *whi = std::max(*whi, p.aze);
  }
  return ref == INT_MAX ? -1 : ref & 255;
}

// A wave's pulses: any lane's (qlo, qhi), every live lane's (qc0, qc1).
struct WaveWindow {
  int qlo = INT_MAX, qhi = -1, qc0 = -1, qc1 = INT_MAX;
  explicit WaveWindow(const Pixel* px) {
    for (int k = 0; k < kWave; ++k) {
      if (!px[k].live()) continue;
      qlo = std::min(qlo, px[k].azs);
      qhi = std::max(qhi, px[k].aze);
      qc0 = std::max(qc0, px[k].azs);
      qc1 = std::min(qc1, px[k].aze);
    }
  }
};

void split_stage(int wave, int p0, int p1, int* qa, int* qb) {
  const int seg = (p1 - p0 + 3) >> 2;
  *qa = std::max(*qa, p0 + wave * seg);
  *qb = std::min(*qb, p0 + (wave + 1) * seg);
}

double range_of(const Burst& b, const double* x, int q) {
  long double r2 = 0;
  for (int i = 0; i < 3; ++i) {
    const long double d = (long double)x[i] - b.sat[3 * q + i];
    r2 += d * d;
  }
  return (double)(sqrtl(r2) - b.rngstart);
}

struct Found {
  long pairs = 0, bad_index = 0, bad_offset = 0, bad_range = 0, lost = 0, waves = 0, fits = 0;
  double worst = 0;
  void add(const Found& o) {
    pairs += o.pairs; bad_index += o.bad_index; bad_offset += o.bad_offset;
    bad_range += o.bad_range; lost += o.lost; waves += o.waves; fits += o.fits;
    worst = std::max(worst, o.worst);
  }
};

// ------------------------------------------------------------ split tiles

void replay_split(const Burst& b, int tile, int tiles_r, Found& st) {
  Pixel px[kBlock];
  int wlo, whi;
  const int ref = tile_pixels(b, 4, 2, tile, tiles_r, px, &wlo, &whi);
  if (ref < 0) return;
  ++st.waves;
  const double inv_dmrg = 1.0 / b.dmrg, *x0 = px[ref].x;
  const int pc = (wlo + whi - 1) >> 1;
  double uref[3], R0ref = 0;
  for (int i = 0; i < 3; ++i) uref[i] = x0[i] - b.sat[3 * pc + i];
  R0ref = std::sqrt(uref[0] * uref[0] + uref[1] * uref[1] + uref[2] * uref[2]);
  for (int i = 0; i < 3; ++i) uref[i] *= 1.0 / R0ref;
  const WaveWindow w(px);   // the four waves hold the same pixels
  const int qc1 = std::max(w.qc1, w.qc0);
  if (w.qhi - w.qlo < 16) return;
  const double mid = 0.5 * (w.qlo + w.qhi - 1), hh = 0.5 * (w.qhi - 1 - w.qlo);
  const int qn[5] = {(int)std::rint(mid - 0.8660254037844386 * hh), (int)std::rint(mid),
                     (int)std::rint(mid + 0.8660254037844386 * hh), w.qlo, w.qhi - 1};
  double gu[5][4];
  for (int j = 0; j < 5; ++j) {
    const double* s = &b.sat[3 * qn[j]];
    const double v[3] = {x0[0] - s[0], x0[1] - s[1], x0[2] - s[2]};
    const double inv = rsqrt64(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    for (int i = 0; i < 3; ++i) gu[j][i] = v[i] * inv;
    gu[j][3] = 0.5 * inv;
  }
  float c0[kWave], c1[kWave], c2[kWave], fa[kWave], dmaxf = 0.f, pmaxf = 0.f;
  int ia[kWave], ia_min = INT_MAX;
  for (int k = 0; k < kWave; ++k) {
    const Pixel& p = px[k];
    double d[3], y[5];
    for (int i = 0; i < 3; ++i) d[i] = p.live() ? p.x[i] - x0[i] : 0.;
    const double bb = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    const double aref = uref[0] * d[0] + uref[1] * d[1] + uref[2] * d[2];
    for (int j = 0; j < 5; ++j) y[j] = node_excess(gu[j][0], gu[j][1], gu[j][2], gu[j][3], d, bb, aref);
    const double k0 = qn[0] - pc, k1 = qn[1] - pc, k2 = qn[2] - pc;
    const double a1 = (y[1] - y[0]) / (k1 - k0), a2 = ((y[2] - y[1]) / (k2 - k1) - a1) / (k2 - k0);
    const double q1 = a1 - a2 * (k0 + k1), q0 = y[0] - k0 * (a1 - a2 * k1);
    const double kl = w.qlo - pc, kh = w.qhi - 1 - pc;
    const auto at = [&](double t) { return (a2 * t + q1) * t + q0; };
    double pm = std::max(std::fabs(at(kl)), std::fabs(at(kh)));
    const double kv = a2 != 0.0 ? -q1 / (2.0 * a2) : kl;
    if (kv > kl && kv < kh) pm = std::max(pm, std::fabs(at(kv)));
    if (!(std::fabs(at(kl) - y[3]) <= 1e-7 && std::fabs(at(kh) - y[4]) <= 1e-7 &&
          pm <= 2.0 * std::sqrt(bb) + 1e-3 && (size_t)b.L * b.S * 8 + kSbufBias < 0x7fffffffu))
      return;   // the FP32 chain
    if (p.live()) {
      dmaxf = std::max(dmaxf, (float)std::sqrt(bb));
      pmaxf = std::max(pmaxf, (float)(pm * (1.0 + 1e-6)));
    }
    ia[k] = (int)std::rint(aref * inv_dmrg);
    ia_min = std::min(ia_min, ia[k]);
    fa[k] = (float)(aref * inv_dmrg - ia[k]);
    c0[k] = (float)q0;
    c1[k] = (float)q1;
    c2[k] = (float)a2;
  }
  ++st.fits;
  const double dmax = dmaxf, pmx = (double)pmaxf + 1e-6, mq = (dmax + pmx + 1e-3) * inv_dmrg;
  const int i0s = (int)std::floor((R0ref - b.rngstart) * inv_dmrg) - 64 -
                  (int)std::fmin(pmx * inv_dmrg, 4096.0);
  const double ext_lo = dmax * inv_dmrg + 1.0;
  const double ext_hi = (dmax + dmax * dmax / R0ref) * inv_dmrg + 1.0;
  for (int p0 = wlo; p0 < whi; p0 += kStage) {
    const int p1 = std::min(p0 + kStage, whi);
    float f0s[kStage];
    bool safe = true;
    for (int q = p0; q < p1; ++q) {
      const double* s = &b.sat[3 * q];
      const double u[3] = {x0[0] - s[0], x0[1] - s[1], x0[2] - s[2]};
      const double r2 = u[0] * u[0] + u[1] * u[1] + u[2] * u[2], R0 = r2 * rsqrt64(r2);
      const double rb = (R0 - b.rngstart) * inv_dmrg, f = rb - i0s;
      safe = safe && R0 >= 0.5 * R0ref + dmax && rb - ext_lo >= 1.0 &&
             rb + ext_hi <= b.r_hi - 1.0 && f - pmx * inv_dmrg - 1.5 >= 0.0 && f <= 1024.0 &&
             rb - mq - 3.0 >= 0.0 && rb + mq + 3.0 <= b.S - 1;
      f0s[q - p0] = (float)f;
    }
    if (!safe) continue;
    for (int wave = 0; wave < 4; ++wave) {
      int qa = std::max(p0, w.qlo), qb = std::min(p0 + kStage, w.qhi);
      split_stage(wave, p0, p1, &qa, &qb);
      const int ca = std::max(qa, w.qc0), cb = std::min(qb, qc1);
      for (int q = ca; q < cb; ++q)
        for (int k = 0; k < kWave; ++k) {
          const float kk = (float)(q - pc);
          const float P = std::fmaf(std::fmaf(c2[k], kk, c1[k]), kk, c0[k]);
          const float rho = std::fmaf(P, (float)inv_dmrg, f0s[q - p0]) + fa[k];
          const long il = floor_i(rho), idx = (long)i0s + ia[k] + il;
          const long long so = ((long long)q * b.S + i0s + ia_min) * 8 + kSbufBias;
          ++st.pairs;
          st.bad_index += il < 0 || il >= kIndexLimit || idx < 0 || idx > b.S - 2;
          st.bad_offset += so < 0 || so >= (1ll << 32);
          if (!px[k].live()) continue;
          const double off =
              std::fabs(rho + (double)(i0s + ia[k]) - range_of(b, px[k].x, q) * inv_dmrg);
          st.worst = std::max(st.worst, off);
          st.bad_range += !(off <= 2.0 / 16384);
        }
    }
  }
}

// ------------------------------------------------------------------ FP64

constexpr int kNodes = 5, kHalf = 16, kPlainStage = 768;
constexpr double kTol = 1e-10;

void newton4(const double* t, const double* y, double* c) {
  double a[5];
  for (int i = 0; i < 5; ++i) a[i] = y[i];
  for (int l = 1; l < 5; ++l)
    for (int i = 4; i >= l; --i) a[i] = (a[i] - a[i - 1]) * (1.0 / (t[i] - t[i - l]));
  for (int i = 0; i < 5; ++i) c[i] = 0.0;
  c[0] = a[4];
  for (int l = 3; l >= 0; --l) {
    for (int i = 4; i >= 1; --i) c[i] = std::fma(-t[l], c[i], c[i - 1]);
    c[0] = std::fma(-t[l], c[0], a[l]);
  }
}
double quartic(const double* c, double t) {
  return std::fma(std::fma(std::fma(std::fma(c[4], t, c[3]), t, c[2]), t, c[1]), t, c[0]);
}

void replay_fp64(const Burst& b, int TR, int STACK, int tile, int tiles_r, Found& st) {
  Pixel px[kBlock];
  int wlo, whi;
  const int ref = tile_pixels(b, TR, STACK, tile, tiles_r, px, &wlo, &whi);
  if (ref < 0) return;
  const double* x0 = px[ref].x;
  const double inv_dmrg = 1.0 / b.dmrg, two_over_wvl = 2.0 / b.wvl;
  const int span = whi - 1 - wlo;
  st.waves += STACK == 2 ? 1 : 4;
  if (whi - wlo < 32 || (size_t)b.L * b.S * 8u >= (size_t)0x7fffffff) return;
  const double dt = 2.0 / span;
  const double g[kNodes + 2] = {0.024471741852423214, 0.20610737385376343, 0.5,
                                0.79389262614623657, 0.97552825814757679, 0.0, 1.0};
  double u[kNodes + 2][3], r2[kNodes + 2], R0[kNodes + 2], t[kNodes + 2], look[3][kNodes];
  for (int j = 0; j < kNodes + 2; ++j) {
    const int q = wlo + (int)std::rint(g[j] * span);
    for (int i = 0; i < 3; ++i) u[j][i] = x0[i] - b.sat[3 * q + i];
    r2[j] = u[j][0] * u[j][0] + u[j][1] * u[j][1] + u[j][2] * u[j][2];
    R0[j] = std::sqrt(r2[j]);
    t[j] = std::fma((double)(q - wlo), dt, -1.0);
  }
  for (int i = 0; i < 3; ++i) {
    double y[kNodes];
    for (int j = 0; j < kNodes; ++j) y[j] = u[j][i] / R0[j];
    newton4(t, y, look[i]);
  }
  static thread_local double c[kBlock][kNodes];
  bool fit[kBlock];
  int half[kBlock];
  float emax = 0.f, dmaxf = 0.f;
  for (int tid = 0; tid < kBlock; ++tid) {
    const Pixel& p = px[tid];
    for (double& v : c[tid]) v = 0.;
    fit[tid] = true;
    half[tid] = kHalf;
    if (!p.live()) continue;
    const double d[3] = {p.x[0] - x0[0], p.x[1] - x0[1], p.x[2] - x0[2]};
    const double bb = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    double y[kNodes + 2], *cc = c[tid];
    for (int j = 0; j < kNodes + 2; ++j) {
      const double num =
          std::fma(2.0, std::fma(u[j][0], d[0], std::fma(u[j][1], d[1], u[j][2] * d[2])), bb);
      y[j] = num / (std::sqrt(r2[j] + num) + R0[j]);
    }
    newton4(t, y, cc);
    bool ok = std::fabs(quartic(cc, t[kNodes]) - y[kNodes]) <= kTol &&
              std::fabs(quartic(cc, t[kNodes + 1]) - y[kNodes + 1]) <= kTol;
    const double b2 = (std::fabs(cc[2]) + 3.0 * std::fabs(cc[3]) + 6.0 * std::fabs(cc[4])) * dt *
                      dt * two_over_wvl * 6.2832;
    const double b3 = (std::fabs(cc[3]) + 4.0 * std::fabs(cc[4])) * dt * dt * dt * 0.385;
    int h = kHalf;
    while (h > 1 && !(b2 * h * h <= 1e-3 && b3 * h * h * h <= 2e-11)) h >>= 1;
    ok = ok && h >= 4;
    double em = 0;
    for (int i = 0; i < kNodes; ++i) em += std::fabs(cc[i]);
    if (ok) emax = std::max(emax, (float)(em * (1.0 + 1e-6)));
    dmaxf = std::max(dmaxf, (float)(std::sqrt(bb) * (1.0 + 1e-6)));
    fit[tid] = ok;
    half[tid] = h;
  }
  const double ext = 2.0 * emax * inv_dmrg + 2.0;
  std::vector<double> rb(kPlainStage + 1);
  for (int p0 = wlo; p0 < whi; p0 += kPlainStage) {
    const int p1 = std::min(p0 + kPlainStage, whi);
    bool safe = true;
    for (int q = p0; q < p1; ++q) {
      double v[3], n2 = 0, dev = 0;
      for (int i = 0; i < 3; ++i) v[i] = x0[i] - b.sat[3 * q + i];
      n2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
      const double R = std::sqrt(n2), tq = std::fma((double)(q - wlo), dt, -1.0);
      for (int i = 0; i < 3; ++i) dev = std::max(dev, std::fabs(quartic(look[i], tq) - v[i] / R));
      rb[q - p0] = (R - b.rngstart) * inv_dmrg;
      safe = safe && rb[q - p0] - ext >= 0.0 && rb[q - p0] + ext <= b.r_hi && dev * dmaxf <= kTol;
    }
    rb[p1 - p0] = -1e9;
    for (int wave = 0; wave < 4; ++wave) {
      const Pixel* wp = STACK == 2 ? px : px + kWave * wave;
      const int lane0 = STACK == 2 ? 0 : kWave * wave;
      const WaveWindow w(wp);
      bool wave_fit = w.qhi > w.qlo;
      int blk = 2 * kHalf;
      for (int k = 0; k < kWave; ++k) {
        wave_fit = wave_fit && fit[lane0 + k];
        blk = std::min(blk, 2 * half[lane0 + k]);
      }
      if (!wave_fit || !safe) continue;
      ++st.fits;
      int qa = std::max(p0, w.qlo), qb = std::min(p1, w.qhi);
      if (STACK == 2) split_stage(wave, p0, p1, &qa, &qb);
      long summed[kWave] = {};
      for (int q = qa; q < qb;) {
        const int ce = std::min(qb, w.qc1);
        const bool core = q >= w.qc0 && q + 1 < ce;
        const int n = core ? std::min(blk, ce - q) & ~1
                           : std::min(blk, (q < w.qc0 ? std::min(qb, w.qc0) : qb) - q);
        const int m = (n + 1) >> 1;
        for (int k = 0; k < kWave; ++k) {
          const Pixel& p = wp[k];
          const double* cc = c[lane0 + k];
          const double h = m, hi = 1.0 / m, tc = std::fma((double)(q - wlo) + (m - 0.5), dt, -1.0);
          const double e0 = quartic(cc, tc), em = quartic(cc, std::fma(-h, dt, tc)),
                       ep = quartic(cc, std::fma(h, dt, tc));
          const double a1 = (ep - em) * (0.5 * hi), a2 = ((ep - e0) - (e0 - em)) * (0.5 * hi * hi);
          double pp = std::fma(0.5, a1, std::fma(0.25, a2, e0)) * inv_dmrg;
          double pm = std::fma(-0.5, a1, std::fma(0.25, a2, e0)) * inv_dmrg;
          double dp = std::fma(2.0, a2, a1) * inv_dmrg, dm = std::fma(2.0, a2, -a1) * inv_dmrg;
          const double d2 = 2.0 * a2 * inv_dmrg;
          const int last = core ? q + n : std::min(q + n, p.aze);
          for (int j = 0; j < m; ++j) {
            for (int side = 0; side < 2; ++side) {
              const int s = side ? q + m - 1 - j : q + m + j;
              const double at = rb[s - p0] + (side ? pm : pp);
              const long long so = (long long)s * b.S * 8;
              st.bad_offset += so < 0 || so >= (1ll << 31);
              if (!(p.live() && s >= p.azs && s < last)) continue;
              ++st.pairs;
              ++summed[k];
              st.bad_index += !(at >= 0.0 && at <= b.r_hi && (int)at <= b.S - 2);
              const double off = std::fabs(at * b.dmrg - range_of(b, p.x, s));
              st.worst = std::max(st.worst, off);
              st.bad_range += !(off <= 5e-10);
            }
            pp += dp;
            pm += dm;
            dp += d2;
            dm += d2;
          }
        }
        q += n;
      }
      for (int k = 0; k < kWave; ++k) {
        const int lo = std::max(qa, wp[k].azs), hi = std::min(qb, wp[k].aze);
        st.lost += wp[k].live() && summed[k] != std::max(0, hi - lo);
      }
    }
  }
}

}  // namespace

int main(int argc, char** argv) {
  const bool split = argc == 3 && !std::strcmp(argv[2], "split");
  if (!split && !(argc == 5 && !std::strcmp(argv[2], "fp64"))) return 2;
  const int TR = split ? 4 : std::atoi(argv[3]), STACK = split ? 2 : std::atoi(argv[4]);
  if ((TR != 1 && TR != 2 && TR != 4 && TR != 8) || STACK < 0 || STACK > 2) return 2;
  FILE* f = std::fopen(argv[1], "rb");
  if (!f) return 2;
  Found total;
  for (;;) {
    int32_t h[9];
    double d[9];
    Burst b;
    if (!rd(f, h, 9)) break;
    if (!rd(f, d, 9)) return 2;
    b.L = h[0]; b.S = h[1]; b.W = h[2]; b.nlines = h[3]; b.nfit = h[4]; b.firstline = h[5];
    b.firstpix = h[6]; b.lastpix = h[7]; b.A = h[8];
    b.rngstart = d[0]; b.rng_hi = d[1]; b.dmrg = d[2]; b.wvl = d[3]; b.r_hi = d[4];
    b.firstlat = d[5]; b.firstlon = d[6]; b.deltalat = d[7]; b.deltalon = d[8];
    b.coef.resize(3 * (size_t)b.nlines);
    b.sat.resize(3 * (size_t)b.L);
    b.dem.resize((size_t)b.nlines * b.W);
    if (!rd(f, b.coef.data(), b.coef.size()) || !rd(f, b.sat.data(), b.sat.size()) ||
        !rd(f, b.dem.data(), b.dem.size()))
      return 2;
    const int TC = kWave / TR, WR = STACK == 1 ? 4 * TR : TR, WC = STACK == 0 ? 4 * TC : TC;
    const int tiles_r = (b.nlines + WR - 1) / WR, tiles_c = (b.W + WC - 1) / WC;
    std::vector<Found> per(omp_get_max_threads());
#pragma omp parallel for schedule(dynamic, 16)
    for (int t = 0; t < tiles_r * tiles_c; ++t)
      if (split) replay_split(b, t, tiles_r, per[omp_get_thread_num()]);
      else replay_fp64(b, TR, STACK, t, tiles_r, per[omp_get_thread_num()]);
    for (auto& s : per) total.add(s);
  }
  std::fclose(f);
  const bool ok = !total.bad_index && !total.bad_offset && !total.bad_range && !total.lost &&
                  total.pairs;
  std::printf("pairs %ld waves %ld fits %ld worst %.3g; bad index %ld offset %ld range %ld, "
              "windows not summed once %ld -> %s\n",
              total.pairs, total.waves, total.fits, total.worst, total.bad_index,
              total.bad_offset, total.bad_range, total.lost, ok ? "OK" : "FAIL");
  return ok ? 0 : 1;
}
